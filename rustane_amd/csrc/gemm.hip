// Prefill GEMMs with residual epilogues (split-K, fused reduce + RMSNorm),
// the plain store, and the split counts.
#include "gemm_launch.hpp"

namespace hb {

// Split-K reduction fused with the RMSNorm that follows a residual projection
// (cpu/rmsnorm.rs:149-183): one workgroup of 256 threads per token row adds the
// splits in order, applies the residual epilogue (out = res + alpha * v), and
// normalises the row into xn. The element-to-thread mapping and the block sum
// are those of rmsnorm_kernel, so xn is bit-identical to reduce + rmsnorm.
template <int NPT, bool RAG = false>  // as rmsnorm_kernel: N = NPT * 1024 (RAG: N <= NPT * 1024) in registers, or 0 = any N
__global__ __launch_bounds__(256) void splitk_reduce_norm_kernel(const float* __restrict__ P, int S,
                                                                 int N, size_t stride,
                                                                 EpiResidual e, NormOut no) {
  constexpr int MAXS = GEMM_MAX_SPLITS;
  __shared__ float red[4];
  const int t = blockIdx.x;
  const size_t row = (size_t)t * N;
  f16* orow = no.xn + (no.split ? 2 * row : row);
  const size_t lo = no.split ? (size_t)N : 0;  // split xn rows: [hi | lo]
  float ss = 0.f;
  if constexpr (NPT > 0) {
    auto in = [&](int i) { return !RAG || (int)threadIdx.x * 4 + i * 1024 < N; };
    f32x4 y[NPT], g[NPT];
    {
      f32x4 part[NPT][MAXS], r[NPT];
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        if (!in(i)) continue;
        const size_t c = row + threadIdx.x * 4 + i * 1024;
#pragma unroll
        for (int s = 0; s < MAXS; ++s)
          if (s < S) part[i][s] = *(const f32x4*)(P + s * stride + c);
        r[i] = *(const f32x4*)(e.res + c);
      }
#pragma unroll
      for (int i = 0; i < NPT; ++i) g[i] = in(i) ? *(const f32x4*)(no.gamma + threadIdx.x * 4 + i * 1024) : f32x4{};
#pragma unroll
      for (int i = 0; i < NPT; ++i) {
        if (!in(i)) {  // past N: adds 0 to the sum of squares
          y[i] = f32x4{};
          continue;
        }
        f32x4 v = part[i][0];
#pragma unroll
        for (int s = 1; s < MAXS; ++s)
          if (s < S) v += part[i][s];
        y[i].x = __builtin_fmaf(v.x, e.alpha, r[i].x);  // as EpiResidual
        y[i].y = __builtin_fmaf(v.y, e.alpha, r[i].y);
        y[i].z = __builtin_fmaf(v.z, e.alpha, r[i].z);
        y[i].w = __builtin_fmaf(v.w, e.alpha, r[i].w);
        *(f32x4*)(e.out + row + threadIdx.x * 4 + i * 1024) = y[i];
        ss += y[i].x * y[i].x + y[i].y * y[i].y + y[i].z * y[i].z + y[i].w * y[i].w;
      }
    }
    ss = block_sum<4>(ss, red);
    const float rinv = 1.0f / sqrtf(ss * (1.0f / (float)N) + no.eps);
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
      if (!in(i)) continue;
      f32x4 o;
      o.x = y[i].x * rinv * g[i].x;
      o.y = y[i].y * rinv * g[i].y;
      o.z = y[i].z * rinv * g[i].z;
      o.w = y[i].w * rinv * g[i].w;
      store_f16x4(orow + threadIdx.x * 4 + i * 1024, o, lo);
    }
  } else {
    for (int c = threadIdx.x * 4; c < N; c += 1024) {
      f32x4 part[MAXS];
#pragma unroll
      for (int s = 0; s < MAXS; ++s)
        if (s < S) part[s] = *(const f32x4*)(P + s * stride + row + c);
      f32x4 v = part[0];
#pragma unroll
      for (int s = 1; s < MAXS; ++s)
        if (s < S) v += part[s];
      const f32x4 r = *(const f32x4*)(e.res + row + c);
      f32x4 y;
      y.x = __builtin_fmaf(v.x, e.alpha, r.x);
      y.y = __builtin_fmaf(v.y, e.alpha, r.y);
      y.z = __builtin_fmaf(v.z, e.alpha, r.z);
      y.w = __builtin_fmaf(v.w, e.alpha, r.w);
      *(f32x4*)(e.out + row + c) = y;
      ss += y.x * y.x + y.y * y.y + y.z * y.z + y.w * y.w;
    }
    ss = block_sum<4>(ss, red);
    const float rinv = 1.0f / sqrtf(ss * (1.0f / (float)N) + no.eps);
    for (int c = threadIdx.x * 4; c < N; c += 1024) {
      const f32x4 y = *(const f32x4*)(e.out + row + c);  // this thread's own stores
      const f32x4 g = *(const f32x4*)(no.gamma + c);
      f32x4 o;
      o.x = y.x * rinv * g.x;
      o.y = y.y * rinv * g.y;
      o.z = y.z * rinv * g.z;
      o.w = y.w * rinv * g.w;
      store_f16x4(orow + c, o, lo);
    }
  }
}

// Tile and split choice by predicted time. A launch of n workgroups (tiles x
// splits) takes n / 256 rounds of the 256 CUs, a partly filled last round
// counting 0.65 + 0.35 x its fill (its tiles run faster with fewer
// neighbours), of slice_us per 64-wide K slice plus tile_us per tile
// (prologue and epilogue). The constants are fitted to launches at 45 to 4096
// tokens of the 7B, 5B and 600M shapes with K = 512 to 11008: the choice is
// the fastest measured tile in 15 of 16 of them and 2% off in the other. For
// instance, us per tile 256x256 / 192x256 / 128x256 / 192x128 / 128x128 /
// 64x128: 12288 x 4096 x 4096 320 / 328 / 350 / 372 / 445 / 575; 22016 x 512 x
// 4096 87 / 78 / 104 / 90 / 106 / 133; 22016 x 45 x 4096 69 / 55 / 46 / 43 / 31 /
// 42. 192x128 and 128x128 workgroups run two to a CU, one's epilogue under the
// other's main loop (tile_us): QKV of 600M at 4096 tokens 88 us on 192x128
// with its attention, 94 on 192x256.
// Unsplit products have a seventh tile, 256x128 (launch_gemm): 513 to 640 tokens
// are five columns of it, where 256-token tiles run 17-33% padding and smaller
// ones a second round. Blocks of the other tiles -> 256x128, us, one stream: 7B
// attention block at 513 / 640 tokens 86.4 / 94.9 -> 79.2 / 84.8, GQA FFN 63.5 /
// 70.7 -> 61.2 / 66.1, 7B FFN 225.9 / 242.7 -> 225.6 / 238.4. Forced on the QKV and
// W1|W3 products at 45 to 2048 other tokens it is level or up to 70% slower: its
// constants are fitted at K = 2048 and 4096, and its tile_us keeps it from shorter K.
const GemmTile GEMM_TILES[GEMM_NTILES] = {{256, 256, 1.43f, 12.f}, {192, 256, 1.11f, 10.f}, {128, 256, 0.83f, 8.f},
                                          {192, 128, 0.64f, 5.5f}, {128, 128, 0.49f, 5.f},  {64, 128, 0.42f, 4.5f},
                                          {256, 128, 0.81f, 15.f}};
static constexpr int GEMM_CUS = 256;  // MI355X compute units

GemmChoice gemm_tile(int N, int T, int K, int S, float* us, int tiles) {
  const int kq = (K / 64 + S - 1) / S;
  GemmChoice best{0, S};
  float best_us = INFINITY;
  for (int i = 0; i < tiles; ++i) {
    const GemmTile& g = GEMM_TILES[i];
    const long n = ntiles(N, T, g.ft, g.tt) * S;
    const float fill = (float)(n % GEMM_CUS) / GEMM_CUS;
    const float rounds = (float)(n / GEMM_CUS) + (fill > 0.f ? 0.65f + 0.35f * fill : 0.f);
    const float t = rounds * ((float)kq * g.slice_us + g.tile_us);
    if (t < best_us) {
      best_us = t;
      best.tile = i;
    }
  }
  if (us) *us = best_us;
  return best;
}

// Long-K residual projections with few output tiles (Wo and W2 at 512 tokens:
// 128 tiles of 128x128) split K over up to GEMM_MAX_SPLITS ranges of >= 8
// slices so that ~256 workgroups run; the partials go through the caller's
// scratch and splitk_reduce applies the epilogue. The number of splits fixes
// the order of the sums, the tile (gemm_tile) does not. K from 1024 splits too
// (600M shape, Wo with K = 1536 at 512 tokens: 96 workgroups of 64x128 unsplit,
// 144 of 128x128 in 3 splits; the batch-1 forward 2.28 -> 2.16 ms).
int gemm_splits(int N, int T, int K) {
  const long t = ntiles(N, T, 128, 128);
  const int nk = K / 64;
  if (t >= GEMM_CUS || nk < 16) return 1;
  int S = (int)std::min<long>(GEMM_MAX_SPLITS, GEMM_CUS / t);
  S = std::min(S, nk / 8);
  return S >= 2 ? S : 1;
}

// The residual + RMSNorm projections (gemm_residual_norm): a long reduction
// (K >= 2N) takes the split count in which blocks of 256 features x 128 tokens
// fill the CUs exactly (7B W2 at 512 tokens: 64 blocks, 4 splits instead of 2;
// GEMM alone 54 -> 45.5 us, run on 64 tiles of 128x256 as gemm_tile picks them:
// the wider tile's main loop outweighs the reduce reading 4 partials instead of
// 2; Wo, K = N, gains less). The block shape is that of the tile these launches
// first ran on and is kept because the count fixes the order of the forward's
// sums; where it does not divide the CUs, gemm_splits' count stands.
int gemm_norm_splits(int N, int T, int K) {
  const int S = gemm_splits(N, T, K);
  if (S <= 1 || K < 2 * N) return S;
  const long t = ntiles(N, T, 256, 128);
  if (t <= 0 || GEMM_CUS % t) return S;
  const int Sw = (int)(GEMM_CUS / t);
  return Sw < 2 || Sw > GEMM_MAX_SPLITS || Sw * 8 > K / 64 ? S : Sw;
}

// The input-gradient products (gemm_store_split): any number of splits of >= 8
// slices, by predicted time: REDUCE_US for the reduction's launch and
// (splits + 2) x T x N floats through memory at ~4.5 TB/s. N = 2560 at 2048
// tokens has 80 tiles of 256x256; K = 13824 and 32000 take them in 3 splits
// (all five products of a layer and head 186 us on average unsplit on 192x128
// tiles, 158 with the reduction).
int gemm_store_splits(int N, int T, int K) {
  constexpr float REDUCE_US = 3.f, US_PER_BYTE = 1.f / 4.5e6f;
  const int nk = K / 64;
  const size_t TN = (size_t)T * N;
  int best = 1;
  float best_us = INFINITY;
  for (int S = 1; S <= GEMM_MAX_SPLITS && (S == 1 || nk >= 8 * S); ++S) {
    if ((S - 1) * ((nk + S - 1) / S) >= nk) continue;
    float us;
    (void)gemm_tile(N, T, K, S, &us);
    if (S > 1) us += REDUCE_US + (float)(S + 2) * 4.f * (float)TN * US_PER_BYTE;
    if (us < best_us) {
      best_us = us;
      best = S;
    }
  }
  return best;
}

hipError_t gemm_store(const f16* W, const f16* X, int N, int T, int K, float* C, hipStream_t st) {
  return launch_gemm(W, X, N, T, K, EpiStore{C, N}, st);
}
hipError_t gemm_residual(const f16* W, const f16* X, int N, int T, int K, const EpiResidual& e,
                         const GemmScratch* scr, hipStream_t st, int kw) {
  return launch_split_gemm(W, X, N, T, K, e, scr ? gemm_splits(N, T, K) : 1, scr, st, kw);
}
hipError_t gemm_residual_norm(const f16* W, const f16* X, int N, int T, int K, const EpiResidual& e,
                              const NormOut& no, const GemmScratch* scr, hipStream_t st, int kw,
                              hipEvent_t mid) {
  if (e.ld != N) return hipErrorInvalidValue;
  if (!gemm_fits(N, T, K)) return hipErrorInvalidValue;
  const GemmChoice c = gemm_tile(N, T, K, scr ? gemm_norm_splits(N, T, K) : 1);
  const int S = c.splits;
  hipError_t err2 = hipSuccess;
  if (S > 1) {
    const size_t stride = (size_t)T * N;
    if (!scr->p || (size_t)S * stride > scr->floats) return hipErrorInvalidValue;
    const hipError_t err = launch_choice(c, W, X, N, T, K, EpiSplit{scr->p, N, stride}, st, kw);
    if (err != hipSuccess) return err;
    if (mid && (err2 = hipEventRecord(mid, st)) != hipSuccess) return err2;
    // 1..8: whole multiples of 1024; 9..16: ragged, ceil(N / 1024) = 1..8
    switch (N % 1024 == 0 ? N / 1024 : N % 4 == 0 && N < 8192 ? 8 + N / 1024 + 1 : 0) {
#define HB_RN(n, c, rag)                                                                        \
  case c:                                                                                       \
    hipLaunchKernelGGL((splitk_reduce_norm_kernel<n, rag>), dim3(T), dim3(256), 0, st, scr->p, S, \
                       N, stride, e, no);                                                       \
    break;
      HB_RN(1, 1, false) HB_RN(2, 2, false) HB_RN(3, 3, false) HB_RN(4, 4, false)
      HB_RN(5, 5, false) HB_RN(6, 6, false) HB_RN(7, 7, false) HB_RN(8, 8, false)
      HB_RN(1, 9, true) HB_RN(2, 10, true) HB_RN(3, 11, true) HB_RN(4, 12, true)
      HB_RN(5, 13, true) HB_RN(6, 14, true) HB_RN(7, 15, true) HB_RN(8, 16, true)
#undef HB_RN
      default:
        hipLaunchKernelGGL(splitk_reduce_norm_kernel<0>, dim3(T), dim3(256), 0, st, scr->p, S, N,
                           stride, e, no);
    }
    return hipGetLastError();
  }
  const hipError_t err = launch_choice(c, W, X, N, T, K, e, st, kw);
  if (err != hipSuccess) return err;
  if (mid && (err2 = hipEventRecord(mid, st)) != hipSuccess) return err2;
  return rmsnorm(e.out, N, no.gamma, T, N, no.eps, no.xn, nullptr, st, no.split);
}
// ---- training ----
hipError_t gemm_store_split(const f16* W, const f16* X, int N, int T, int K, float* C,
                            const GemmScratch* scr, hipStream_t st, float scale) {
  return launch_split_gemm(W, X, N, T, K, EpiStore{C, N, scale}, scr ? gemm_store_splits(N, T, K) : 1, scr, st);
}

}  // namespace hb
