// Prefill GEMM launch policy: tile shape per problem size and split-K.
// Included by the translation units that instantiate the products (gemm.hip,
// gemm_qkv.hip, gemm_ffn.hip, gemm_train.hip: one per group of epilogues, so
// that they compile in parallel); the kernel is in gemm_kernel.hpp.
#pragma once
#include "gemm_kernel.hpp"

namespace hb {

// The tiles gemm_nt_kernel runs; the others run on gemm_nt_kernel_reg.
template <int FT, int TT>
constexpr bool kDmaTile = (TT == 256 && FT >= 128) || (TT == 128 && FT >= 192);

// kw: W's row length; K (the X row length and the reduction length) is kw,
// or 2 * kw for split X rows (gemm_kernel.hpp). 0 means K.
template <int FT, int TT, class Epi>
static hipError_t launch_tile(const f16* W, const f16* X, int N, int T, int K, const Epi& epi,
                              hipStream_t st, int splits = 1, int kw = 0) {
  const int tiles = ((N + FT - 1) / FT) * ((T + TT - 1) / TT);
  const int nk = K / 64, kq = (nk + splits - 1) / splits;
  if (kw == 0) kw = K;
  if (nk < 1 || K % 64 || splits < 1 || (splits - 1) * kq >= nk) return hipErrorInvalidValue;
  if ((kw != K && 2 * kw != K) || kw % 64) return hipErrorInvalidValue;
  if constexpr (kDmaTile<FT, TT>)
    hipLaunchKernelGGL((gemm_nt_kernel<FT, TT, Epi>), dim3(tiles, splits), dim3(512), 0, st, W, X, N, T, K, kw, kq,
                       epi);
  else
    hipLaunchKernelGGL((gemm_nt_kernel_reg<FT, TT, 2, 2, Epi>), dim3(tiles, splits), dim3(256), 0, st, W, X, N, T,
                       K, kw, kq, epi);
  return hipGetLastError();
}

// Split-K reduction: v = P[0] + P[1] + ... + P[S-1] (in that order, so the
// result does not depend on scheduling), handed to the epilogue four features
// at a time. HBM/MALL-bound; every split's loads are in flight together.
template <class Epi>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ P, int S,
                                                            int T, int N, size_t stride, Epi epi) {
  constexpr int MAXS = GEMM_MAX_SPLITS;
  const size_t n4 = (size_t)T * N / 4;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
    const size_t e = i * 4;
    f32x4 part[MAXS];
#pragma unroll
    for (int s = 0; s < MAXS; ++s)
      if (s < S) part[s] = *(const f32x4*)(P + s * stride + e);
    f32x4 v = part[0];
#pragma unroll
    for (int s = 1; s < MAXS; ++s)
      if (s < S) v += part[s];
    epi((int)(e / N), (int)(e % N), v);
  }
}

// A tile (index into GEMM_TILES, gemm.hip) and a number of K splits.
struct GemmChoice {
  int tile, splits;
};
struct GemmTile {
  int ft, tt;
  float slice_us, tile_us;
};
constexpr int GEMM_NTILES = 7, GEMM_192x256 = 1, GEMM_128x256 = 2, GEMM_256x128 = 6;  // 6: launch_gemm's only
extern const GemmTile GEMM_TILES[GEMM_NTILES];
// The fastest of the first `tiles` tiles of a product in `splits` K splits, and its
// predicted time.
GemmChoice gemm_tile(int N, int T, int K, int splits, float* us = nullptr, int tiles = GEMM_256x128);

template <class Epi>
static hipError_t launch_choice(GemmChoice c, const f16* W, const f16* X, int N, int T, int K, const Epi& epi,
                                hipStream_t st, int kw) {
  switch (c.tile) {
    case 0: return launch_tile<256, 256>(W, X, N, T, K, epi, st, c.splits, kw);
    case 1: return launch_tile<192, 256>(W, X, N, T, K, epi, st, c.splits, kw);
    case 2: return launch_tile<128, 256>(W, X, N, T, K, epi, st, c.splits, kw);
    case 3: return launch_tile<192, 128>(W, X, N, T, K, epi, st, c.splits, kw);
    case 4: return launch_tile<128, 128>(W, X, N, T, K, epi, st, c.splits, kw);
    default: return launch_tile<64, 128>(W, X, N, T, K, epi, st, c.splits, kw);
  }
}
inline long ntiles(int N, int T, int ft, int tt) { return (long)((N + ft - 1) / ft) * ((T + tt - 1) / tt); }

inline bool gemm_fits(int N, int T, int K) { return (long)N * K < (1L << 31) && (long)T * K < (1L << 31); }

// Unsplit product; tiles (nullable) receives the number of output tiles.
template <class Epi>
static hipError_t launch_gemm(const f16* W, const f16* X, int N, int T, int K, const Epi& epi,
                              hipStream_t st, int kw = 0, int* tiles = nullptr) {
  if (!gemm_fits(N, T, K)) return hipErrorInvalidValue;
  // 256x128 fills one round of the CUs where no other tile does; not where the
  // tile sets the order of a sum of squares
  constexpr bool tall = !EpiSumSq<Epi>::value;
  const GemmChoice c = gemm_tile(N, T, K, 1, nullptr, tall ? GEMM_NTILES : GEMM_256x128);
  if (tiles) *tiles = (int)ntiles(N, T, GEMM_TILES[c.tile].ft, GEMM_TILES[c.tile].tt);
  if constexpr (tall)
    if (c.tile == GEMM_256x128) return launch_tile<256, 128>(W, X, N, T, K, epi, st, 1, kw);
  return launch_choice(c, W, X, N, T, K, epi, st, kw);
}

// Product in S splits of K through the caller's scratch.
template <class Epi>
static hipError_t launch_split_gemm(const f16* W, const f16* X, int N, int T, int K, const Epi& epi,
                                    int S, const GemmScratch* scr, hipStream_t st, int kw = 0) {
  if (!gemm_fits(N, T, K)) return hipErrorInvalidValue;
  const GemmChoice c = gemm_tile(N, T, K, S);
  if (c.splits == 1) return launch_choice(c, W, X, N, T, K, epi, st, kw);
  const size_t stride = (size_t)T * N;
  if (!scr->p || c.splits * stride > scr->floats) return hipErrorInvalidValue;
  const hipError_t e = launch_choice(c, W, X, N, T, K, EpiSplit{scr->p, N, stride}, st, kw);
  if (e != hipSuccess) return e;
  const size_t n4 = stride / 4;
  const int grid = (int)std::min<size_t>((n4 + 255) / 256, 4096);
  hipLaunchKernelGGL((splitk_reduce_kernel<Epi>), dim3(grid), dim3(256), 0, st, scr->p, c.splits, T, N,
                     stride, epi);
  return hipGetLastError();
}

}  // namespace hb
