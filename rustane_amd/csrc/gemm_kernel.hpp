// Prefill GEMM kernels (launch policy in gemm_launch.hpp): gemm_nt_kernel for
// tiles of at least 192x128 or 128x256, gemm_nt_kernel_reg for smaller ones.
//
// C^T tile = W_tile · X_tile^T on v_mfma_f32_{16x16x32,32x32x16}_f16:
//   W [N, K] fp16, K contiguous (weights repacked output-major at upload)
//   X [T, K] fp16, K contiguous (token-major activations)
//   result(t, f) = sum_k X[t,k] * W[f,k], fp32 accumulate, handed to an epilogue.
// MFMA rows are output features and MFMA columns are tokens, so each lane ends
// up holding 4 consecutive features of one token — the shape every epilogue
// (RoPE pairs, SwiGLU pairs, residual float4) wants. The two instruction
// shapes give the same bits.
//
// Split-K: blockIdx.y selects one of gridDim.y contiguous ranges of 64-wide K
// slices (kq slices each, the last one shorter); with gridDim.y = 1 the range
// is all of K. Each split hands its partial sums to the epilogue (EpiSplit).
//
// Split X rows (common.hpp): X rows hold K = 2*kw halves [hi | lo] while W
// rows hold kw; k-slice k0 reads W columns k0 mod kw, so the hi and the lo
// halves of each row meet the same weights. kw = K otherwise.
//
// LDS rows are 128 B (64 halfs) of eight 16-byte chunks; chunk c of row r is
// stored at c ^ swz(r), which keeps the ds_write_b128 of gemm_nt_kernel_reg and
// its 32-row operands' ds_read_b128 free of bank conflicts; the 16-row operand
// reads of gemm_nt_kernel take 4 conflict cycles each (SQ_LDS_BANK_CONFLICT is
// 4.00 x SQ_INSTS_LDS in every tile).
#pragma once
#include <type_traits>

#include "internal.hpp"

namespace hb {

HB_DEV int lds_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// f(integral_constant<int, I>) for I = B .. E-1, unrolled by the template
// expansion itself.
template <int B, int E, class F>
HB_DEV void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// Epilogues that read memory declare `Aux`, `Aux load(t, f0, fb)` and
// `operator()(t, f0, v, aux, fb)`, where fb is the wave-uniform start of the
// 32-feature block that holds f0; the others only `operator()(t, f0, v)`.
template <class E, class = void>
struct EpiAux {
  struct type {};
  static HB_DEV type load(const E&, int, int, int) { return {}; }
  static HB_DEV auto apply(const E& e, int t, int f0, f32x4 v, const type&, int) { return e(t, f0, v); }
};
template <class E>
struct EpiAux<E, std::void_t<typename E::Aux>> {
  using type = typename E::Aux;
  static HB_DEV type load(const E& e, int t, int f0, int fb) { return e.load(t, f0, fb); }
  static HB_DEV auto apply(const E& e, int t, int f0, f32x4 v, const type& a, int fb) {
    return e(t, f0, v, a, fb);
  }
};

// Epilogues with kStage copy a table the epilogue reads into the operand
// LDS once the main loop is done -- `stage<TT, NT>(lo, hi, t_base, f_base,
// tid)` by all threads, then `load_staged(lo, hi, t - t_base, TT, f0, fb)` in
// place of load() -- so that the epilogue's operand reads wait on LDS
// instead of behind its own global stores (one counter covers both).
template <class E, class = void>
struct EpiStage : std::false_type {};
template <class E>
struct EpiStage<E, std::void_t<decltype(E::kStage)>> : std::bool_constant<E::kStage> {};

// Epilogues with `Tok tok(t)`, `row(tok, fb)` and `store_row(row, f0, v, aux,
// fb)` can split their output addressing: tok() once per token of a lane, row()
// once per (32-feature block, token), store_row() per quad.
// Selected by `kRows`.
template <class E, class = void>
struct EpiRows : std::false_type {
  struct Tok {};
};
template <class E>
struct EpiRows<E, std::enable_if_t<E::kRows>> : std::true_type {
  using Tok = typename E::Tok;
};

// Epilogues with kSumSq return the sum of squares of the four values they
// stored; the kernel adds them up per workgroup and writes the total to
// epi.sq_out[tile] (one slot per output tile, fixed order for the reader).
template <class E, class = void>
struct EpiSumSq : std::false_type {};
template <class E>
struct EpiSumSq<E, std::void_t<decltype(E::kSumSq)>> : std::bool_constant<E::kSumSq> {};

// Tile order: groups of GM weight-row panels, token tiles iterated inside a
// group (tile = group*GM*ntt + tt*rows + row), and each XCD takes a
// contiguous range of that order. With 8+ token tiles the 32 tiles an XCD
// runs at a time then share 8 weight panels and 4 token panels in its L2
// instead of 2 and 16 (7B at 4096 tokens: W1|W3 749 -> 663 us, QKV 372 ->
// 338 us); with fewer token tiles GM = 1 (plain row-major order) measures
// ~1% better.
HB_DEV void tile_of(int nft, int ntt, int& tile, int& ft, int& tt) {
  const int GM = ntt >= 8 ? 8 : 1;
  tile = xcd_remap(blockIdx.x, nft * ntt);
  const int grp = tile / (GM * ntt), rem = tile - grp * (GM * ntt);
  const int rows = min(GM, nft - grp * GM);
  tt = rem / rows;
  ft = grp * GM + (rem - tt * rows);
}

// Issue schedule of gemm_nt_kernel's LDS copies, as seen by one wave: per K
// slice of 64 each wave issues one 1 KB copy per 32-row weight block of the
// wave grid (W_i, i < FM) and two per 128-token block (X_j, j < TM), in the
// order below; cum(p) counts those issued by the end of phase p, wait(p) is
// the largest number of copies that may still be in flight at the end of
// phase p's memory half so that everything phase p + 1 reads has landed.
//   phase 0: W_{FM-1} of slice k+1, X_0 of slice k+2
//   phase 1: X_1 of slice k+2        (FM == 2: also W_0 of k+2)
//   phase 2: W_0, W_1 of slice k+2
//   phase 3: W_2 of slice k+2
// W_i is read from LDS in phase i, X_j in phase FM - TM + j of the slice
// before, each at least one phase before its buffer is copied into again.
template <int FT, int TT>
struct GemmPlan {
  static constexpr int FM = FT / 64, TM = TT / 128, N = FM + 2 * TM;
  static_assert(FT % 64 == 0 && TT % 128 == 0 && FM >= 2 && FM <= 4 && TM >= 1 && TM <= 2, "tile");
  static constexpr int cum(int p) {
    int c = 3;
    if (FM == 2) return p >= 1 ? N : c;
    if (p >= 1) c += 2 * (TM - 1);
    if (p >= 2) c += 2;
    if (p >= 3) c += 1;
    return c;
  }
  static constexpr int wait(int p) {
    const int k = 4, issued = k * N + cum(p);  // any slice k: the differences do not depend on it
    const int kr = p + 1 == FM ? k + 1 : k, ph = p + 1 == FM ? 0 : p + 1;  // slice and phase that read
    // index of W_ph(kr)'s copy in issue order
    int first = ph == FM - 1 ? (kr - 1) * N : (kr - 2) * N + 1 + 2 * TM + ph;
    int w = issued - 1 - first;
    for (int j = 0; j < TM; ++j)
      if (ph == FM - TM + j) {  // X_j(kr + 1), second copy
        const int v = issued - 1 - ((kr - 1) * N + 2 + 2 * j);
        if (v < w) w = v;
      }
    return w;
  }
};

// The GEMM kernel: 8 waves (2 feature rows x 4 token columns), two per SIMD,
// on v_mfma_f32_16x16x32_f16.
//
// Operand tiles go from global memory straight into LDS (buffer_load ... lds,
// no registers), two 64-wide K slices deep; wave (wf, wt) owns the features
// i*64 + wf*32 .. +32 (i < FM) and the tokens j*128 + wt*32 .. +32 (j < TM). A
// slice is FM phases; phase i reads the 32-feature fragments of block i
// (and, in the last TM phases, the next slice's token fragments), issues the
// copies of GemmPlan and then runs the 8 * TM MFMAs of its accumulator row.
// Each phase has two halves separated by barriers -- LDS reads and copies,
// then MFMAs -- and the waves of the second feature row run half a phase
// behind those of the first, so on every SIMD one wave feeds the matrix core
// while the other reads and issues (s_setprio favours the one in its MFMA
// half). Each LDS region (one W_i or X_j) is refilled as soon as both halves
// have read it, about 1.5 slices before its next use, and the waits count
// copies (dma_wait) instead of draining them.
//
// What bounds it: the matrix cores under the chip's power limit. MFMA busy is
// 64-70% of the active cycles at 4096 tokens and 53% at 512 (60-70% and 50% in
// the 4-wave register-staged kernel on these shapes), in 6% fewer cycles; the
// rest of the gain is the clock, which settles with the energy per flop,
// so the instruction shape matters: 16x16x32 touches half the accumulator
// registers per flop of 32x32x16 and took the same schedule from 393 to 328 us
// on 12288 x 4096 x 4096 (results bit-identical), and consecutive MFMAs that
// keep the token operand another 2-4%. The clock follows the operand values
// too: all-zero operands run 16-30% faster. Register-staged kernel -> this one,
// fp32 output, back to back on one box, weights and activations N(0, 1) (N x T x
// K): 12288 x 4096 x 4096 357 -> 323 us (1278 TFLOP/s), 22016 x 4096 x 4096 683
// -> 617, 4096 x 4096 x 11008 299 -> 264, 8192^3 885 -> 793 (1387 TFLOP/s),
// 22016 x 512 x 4096 90 -> 79; 12288 x 512 x 4096, one round of 192x128 tiles,
// 57 -> 58. Weights N(0, 0.02): 353 -> 313, 683 -> 623, 302 -> 264, 893 -> 800,
// 89 -> 79 and 55 -> 55.
//
// LDS is written by copies the compiler does not see: its address enters
// their asm, and every copy is waited for before the barrier that precedes its
// reads. Past the last slice the copies re-read the last slice, so every
// phase has the same shape; they are drained before LDS is used again.
template <int FT, int TT, class Epi>
__global__ __launch_bounds__(512, 1) void gemm_nt_kernel(const f16* __restrict__ W, const f16* __restrict__ X,
                                                         int N, int T, int K, int kw, int kq, Epi epi) {
  using P = GemmPlan<FT, TT>;
  constexpr int NT = 512, FM = P::FM, TM = P::TM;
  constexpr uint32_t STAGE = (FT + TT) * 128, XOFF = FT * 128;  // bytes
  __shared__ f16x8 smem[2 * (FT + TT) * 8];  // [stage][W rows, X rows][8 swizzled chunks]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int wf = wave >> 2, wt = wave & 3;
  int tile, ft, tt;
  tile_of((N + FT - 1) / FT, (T + TT - 1) / TT, tile, ft, tt);
  const int f_base = ft * FT, t_base = tt * TT;

  // Copies: one instruction fills 8 rows of 128 bytes; lane l writes chunk l%8
  // of row l/8, so it reads source chunk (l%8) ^ swz(row). Instruction n of
  // wave w takes rows n*64 + w*8 .. +8 of its operand. Byte offsets are
  // 32-bit: the launchers keep N*K and T*K below 2^31 elements.
  const int lr = lane >> 3, lc = (lane & 7) ^ lr ^ (wave & 1);
  uint32_t wvo[FM], xvo[2 * TM];
#pragma unroll
  for (int i = 0; i < FM; ++i) wvo[i] = (uint32_t)(min(f_base + i * 64 + wave * 8 + lr, N - 1) * kw + lc * 8) * 2u;
#pragma unroll
  for (int j = 0; j < 2 * TM; ++j) xvo[j] = (uint32_t)(min(t_base + j * 64 + wave * 8 + lr, T - 1) * K + lc * 8) * 2u;
  const i32x4 wrs = dma_rsrc(W), xrs = dma_rsrc(X);
  const uint32_t lds0 = lds_addr(smem) + wave * 1024;
  const int kt0 = blockIdx.y * kq;
  const int nk = min(kq, K / 64 - kt0);
  auto dma_w = [&](int i, int stage, int k) {
    const int k0 = (kt0 + min(k, nk - 1)) * 64;
    dma_1k(lds0 + stage * STAGE + i * 8192, wvo[i], wrs, (uint32_t)(k0 < kw ? k0 : k0 - kw) * 2u);
  };
  auto dma_x = [&](int j, int stage, int k) {
    const uint32_t so = (uint32_t)(kt0 + min(k, nk - 1)) * 128u;
    dma_1k(lds0 + stage * STAGE + XOFF + (2 * j) * 8192, xvo[2 * j], xrs, so);
    dma_1k(lds0 + stage * STAGE + XOFF + (2 * j + 1) * 8192, xvo[2 * j + 1], xrs, so);
  };

  // acc[i][j][g]: 16x16 block (feature half g>>1, token half g&1) of block (i, j)
  f32x4 acc[FM][TM][4];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) acc[i][j][g] = f32x4{};

  // fragment s of a 32-row block: its rows (s>>1)*16 + lane%16, k (s&1)*32 + 8*(lane/16)
  const int l16 = lane & 15, quad = lane >> 4;
  int ao[4], bo[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int row = (s >> 1) * 16 + l16, c = ((s & 1) * 4 + quad) ^ lds_swz(row);
    ao[s] = (wf * 32 + row) * 8 + c;
    bo[s] = FT * 8 + (wt * 32 + row) * 8 + c;
  }
  f16x8 a[4], b[2][TM][4];

  // Prologue: the copies of issue slices -2 and -1, then slice 0's token fragments.
#pragma unroll
  for (int j = 0; j < TM; ++j) dma_x(j, 0, 0);
#pragma unroll
  for (int i = 0; i < FM; ++i) dma_w(i, 0, 0);
#pragma unroll
  for (int j = 0; j < TM; ++j) dma_x(j, 1, 1);
#pragma unroll
  for (int i = 0; i < FM - 1; ++i) dma_w(i, 1, 1);
  dma_wait<P::wait(FM - 1)>();
  raw_barrier();
#pragma unroll
  for (int j = 0; j < TM; ++j)
#pragma unroll
    for (int s = 0; s < 4; ++s) b[0][j][s] = smem[bo[s] + j * 1024];
  dma_wait<63>();
  raw_barrier();
  if (wf == 1) raw_barrier();  // the second feature row runs half a phase behind

  auto slice = [&](auto sc, int k) {
    constexpr int S = decltype(sc)::value;
    static_for<0, FM>([&](auto pc) {
      constexpr int p = decltype(pc)::value;
#pragma unroll
      for (int s = 0; s < 4; ++s) a[s] = smem[S * (STAGE / 16) + ao[s] + p * 512];
      if constexpr (p >= FM - TM) {
        constexpr int j = p - (FM - TM);
#pragma unroll
        for (int s = 0; s < 4; ++s) b[S ^ 1][j][s] = smem[(S ^ 1) * (STAGE / 16) + bo[s] + j * 1024];
      }
      if constexpr (p == 0) {
        dma_w(FM - 1, S ^ 1, k + 1);
        dma_x(0, S, k + 2);
      }
      if constexpr (p == 1 && TM == 2) dma_x(1, S, k + 2);
      if constexpr (p == 1 && FM == 2) dma_w(0, S, k + 2);
      if constexpr (p == 2) {
        dma_w(0, S, k + 2);
        dma_w(1, S, k + 2);
      }
      if constexpr (p == 3) dma_w(2, S, k + 2);
      dma_wait<P::wait(p)>();
      raw_barrier();
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
          for (int jh = 0; jh < 2; ++jh)
#pragma unroll
            for (int ih = 0; ih < 2; ++ih)
              acc[p][j][ih * 2 + jh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  a[ih * 2 + s], b[S][j][jh * 2 + s], acc[p][j][ih * 2 + jh], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
      raw_barrier();
    });
  };
  // nk >= 1 for every split (the launcher checks (splits - 1) * kq < K / 64)
  int k = 0;
  for (; k + 2 <= nk; k += 2) {
    slice(std::integral_constant<int, 0>{}, k);
    slice(std::integral_constant<int, 1>{}, k + 1);
  }
  if (k < nk) slice(std::integral_constant<int, 0>{}, k);
  if (wf == 0) raw_barrier();
  dma_wait<0>();

  using AX = EpiAux<Epi>;
  using AuxT = typename AX::type;
  // a staged table of up to 32 float4 per token (hd <= 128) fits in the
  // operand LDS, its first half in 16*FT float4 and its second in the 16*TT
  // after them, when TT <= FT; staged on the 256-feature tiles, whose long
  // epilogues gain (7B QKV at 4096 tokens 424 -> 392 us, 5B at 2048 tokens
  // 105 -> 100 us), not on 128x128 (600M QKV 25.6 -> 26.6 us)
  constexpr bool STAGED = EpiStage<Epi>::value && TT <= FT && FT == 256;
  float4* const stab_lo = reinterpret_cast<float4*>(smem);
  float4* const stab_hi = stab_lo + 16 * FT;
  if constexpr (STAGED) {
    raw_barrier();  // every wave's copies are in, every wave's reads done
    epi.template stage<TT, NT>(stab_lo, stab_hi, t_base, f_base, tid);
    __syncthreads();
  }

  // Epilogue over the FM x 2*TM x 2 accumulator quads as straight-line code: a
  // loop would be left rolled once the epilogue body is large, and indexing
  // acc with a loop counter moves the whole accumulator array to scratch
  // memory. Operands that epilogues read from memory (residual stream, RoPE
  // table) are loaded one accumulator row ahead of the stores: the loads
  // cannot be moved above stores that might alias them, so a load-store-load
  // chain per quad would expose the load latency once per quad.
  // Quad q of row i: token half q>>1 (of 2*TM), feature half q&1.
  AuxT aux[2][TM * 4];
  auto tok = [&](int jt) { return t_base + (jt >> 1) * 128 + wt * 32 + (jt & 1) * 16 + l16; };
  auto fblk = [&](int i) { return f_base + i * 64 + wf * 32; };  // wave-uniform
  auto feat = [&](int i, int ih) { return fblk(i) + ih * 16 + quad * 4; };
  auto load_row = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    static_for<0, TM * 4>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      const int t = tok(q >> 1), f = feat(i, q & 1);
      if constexpr (STAGED) {
        if (t < T && f < N) aux[i & 1][q] = epi.load_staged(stab_lo, stab_hi, t - t_base, TT, f, fblk(i));
      } else {
        if (t < T && f < N) aux[i & 1][q] = AX::load(epi, t, f, fblk(i));
      }
    });
  };
  load_row(std::integral_constant<int, 0>{});
  // EpiRows: the token part of the output addresses once per token, the
  // (feature block, token) part once per 2 quads, both outside the quads'
  // bounds tests (they read no memory)
  constexpr bool ROWS = EpiRows<Epi>::value;
  static_assert(!ROWS || !EpiSumSq<Epi>::value, "row-addressed epilogues return nothing");
  typename EpiRows<Epi>::Tok tkj[ROWS ? 2 * TM : 1];
  if constexpr (ROWS) {
    static_for<0, 2 * TM>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      tkj[j] = epi.tok(tok(j));
    });
  }
  float lane_sq = 0.f;
  static_for<0, FM>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i + 1 < FM) load_row(std::integral_constant<int, i + 1>{});
    static_for<0, 2 * TM>([&](auto jc) {
      constexpr int jt = decltype(jc)::value;
      const int t = tok(jt);
      if constexpr (ROWS) {
        const auto rc = epi.row(tkj[jt], fblk(i));
        static_for<0, 2>([&](auto hc) {
          constexpr int ih = decltype(hc)::value;
          const int f = feat(i, ih);
          if (t < T && f < N)
            epi.store_row(rc, f, acc[i][jt >> 1][ih * 2 + (jt & 1)], aux[i & 1][2 * jt + ih], fblk(i));
        });
      } else {
        static_for<0, 2>([&](auto hc) {
          constexpr int ih = decltype(hc)::value;
          const int f = feat(i, ih);
          if (t < T && f < N) {
            const f32x4 v = acc[i][jt >> 1][ih * 2 + (jt & 1)];
            if constexpr (EpiSumSq<Epi>::value)
              lane_sq += AX::apply(epi, t, f, v, aux[i & 1][2 * jt + ih], fblk(i));
            else
              AX::apply(epi, t, f, v, aux[i & 1][2 * jt + ih], fblk(i));
          }
        });
      }
    });
  });
  if constexpr (EpiSumSq<Epi>::value) {
    float* red = (float*)smem;
    const float s = wave_sum(lane_sq);
    raw_barrier();  // every wave's copies are in: the operand buffers are free
    if (lane == 0) red[wave] = s;
    __syncthreads();
    if (tid == 0) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < NT / 64; ++w) tot += red[w];
      epi.sq_out[tile] = tot;
    }
  }
}

// The small-tile kernel: 4 waves of 32x32x16 MFMAs with register-staged operands.
// Its 128x128 tiles run two to a CU, where gemm_nt_kernel has too little work
// per phase to gain (4096 x 512 x 4096 in two splits: 23.4 against 23.3 us, 600M
// QKV 4608 x 512 x 1536 16.2 against 17.5 us).
//
// Pipeline: two 64-wide K slices are in flight in registers while the MFMAs
// consume a third from LDS. Iteration k computes slice k from LDS buffer k&1,
// issues the global loads of slice k+2 into register set k&1 and writes slice
// k+1 (register set (k+1)&1, loaded one iteration earlier) into LDS buffer
// (k+1)&1; one barrier per slice. The loop is unrolled by two so that both
// register sets have static names. Within an iteration sched_group_barrier
// fixes the order: LDS reads of k-step 0 first, then every MFMA is followed by
// one LDS read of the next k-step (k-steps 0..2), and the global loads are
// spread one per MFMA over k-steps 0..2 while the LDS writes are spread over
// k-steps WSTEP..3 (WSTEP = 2: with the operands read through buffer loads the
// later start gives the loads of every tile shape another k-step to land, 7B
// forward B = 1 9.49-9.53 -> 9.37-9.38 ms, seq 2048 31.4 -> 31.0 ms; WSTEP = 3
// is slower at 4096 tokens). Issuing the loads or the writes as a burst stalls the
// wave's in-order issue behind the memory queues and leaves the MFMA pipe idle
// (one wave per SIMD has nothing else to issue).
// Past the last slice the loads re-read the last slice (clamped), so every
// iteration has the same shape.
template <int FT, int TT, int WF, int WT, class Epi>
__global__ __launch_bounds__(WF* WT * 64, 1) void gemm_nt_kernel_reg(const f16* __restrict__ W,
                                                                 const f16* __restrict__ X, int N,
                                                                 int T, int K, int kw, int kq,
                                                                 Epi epi) {
  constexpr int NT = WF * WT * 64;
  constexpr int WFT = FT / WF, WTT = TT / WT;
  constexpr int FM = WFT / 32, TM = WTT / 32;
  constexpr int WL = FT * 8 / NT, XL = TT * 8 / NT;
  constexpr int RSTEP = NT / 8;
  constexpr int NMF = FM * TM, NRD = FM + TM, NLD = WL + XL;
  static_assert(FM >= 1 && TM >= 1, "wave tile must be at least 32x32");
  static_assert(WL * NT == FT * 8 && XL * NT == TT * 8, "loader coverage");
  static_assert(RSTEP % 16 == 0, "loader passes must keep the LDS swizzle phase");
  static_assert(NLD <= 3 * 3 * NMF, "at most three global loads per MFMA slot");

  __shared__ f16x8 sW[2][FT * 8];
  __shared__ f16x8 sX[2][TT * 8];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int wf = wave / WT, wt = wave - wf * WT;
  int tile, ft, tt;
  tile_of((N + FT - 1) / FT, (T + TT - 1) / TT, tile, ft, tt);
  const int f_base = ft * FT, t_base = tt * TT;

  const int r0 = tid >> 3, c0 = tid & 7;
  const int ldst = r0 * 8 + (c0 ^ lds_swz(r0));
  // Operand tiles are read through raw buffer descriptors with the sc1 (device
  // scope) policy: the loads skip L1 allocation for data this workgroup never
  // re-reads. 7B forward: B = 1 9.49-9.52 -> 9.42 ms, B = 8 56.3 -> 55.9 ms
  // against plain global loads, bit-identical. Byte offsets are 32-bit: the
  // launchers keep N*K and T*K below 2^31 elements.
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void*)W, (short)0, -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc((void*)X, (short)0, -1, 0x00020000);
  constexpr int kSC1 = 16;  // cache policy: sc1
  uint32_t wvo[WL], xvo[XL];  // byte offsets of this thread's 16-byte chunks at column 0
#pragma unroll
  for (int i = 0; i < WL; ++i) wvo[i] = (uint32_t)(c0 * 8 + min(f_base + r0 + RSTEP * i, N - 1) * kw) * 2u;
#pragma unroll
  for (int i = 0; i < XL; ++i) xvo[i] = (uint32_t)(c0 * 8 + min(t_base + r0 + RSTEP * i, T - 1) * K) * 2u;

  using R0 = std::integral_constant<int, 0>;
  using R1 = std::integral_constant<int, 1>;
  f16x8 wreg[2][WL], xreg[2][XL];
  auto gload = [&](auto rs, int k0) {
    constexpr int R = decltype(rs)::value;
    const int kw0 = k0 < kw ? k0 : k0 - kw;  // wave-uniform
    // per-lane row offsets in voffset, the slice's column in soffset
#pragma unroll
    for (int i = 0; i < WL; ++i)
      wreg[R][i] = __builtin_bit_cast(
          f16x8, __builtin_amdgcn_raw_buffer_load_b128(wrs, wvo[i], kw0 * 2, kSC1));
#pragma unroll
    for (int i = 0; i < XL; ++i)
      xreg[R][i] = __builtin_bit_cast(
          f16x8, __builtin_amdgcn_raw_buffer_load_b128(xrs, xvo[i], k0 * 2, kSC1));
  };
  auto sstore = [&](auto rs) {
    constexpr int R = decltype(rs)::value;
#pragma unroll
    for (int i = 0; i < WL; ++i) sW[R][ldst + RSTEP * 8 * i] = wreg[R][i];
#pragma unroll
    for (int i = 0; i < XL; ++i) sX[R][ldst + RSTEP * 8 * i] = xreg[R][i];
  };

  f32x16 acc[FM][TM];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x16{};

  const int khalf = lane >> 5;
  const int arow = wf * WFT + (lane & 31), brow = wt * WTT + (lane & 31);
  const int aswz = lds_swz(arow), bswz = lds_swz(brow);
  struct Frag {
    f16x8 a[FM], b[TM];
  };
  auto fread = [&](Frag& F, int buf, int ks) {
    const int c = ks * 2 + khalf;
    const int aoff = arow * 8 + (c ^ aswz), boff = brow * 8 + (c ^ bswz);
#pragma unroll
    for (int i = 0; i < FM; ++i) F.a[i] = sW[buf][aoff + i * 256];
#pragma unroll
    for (int j = 0; j < TM; ++j) F.b[j] = sX[buf][boff + j * 256];
  };
  auto mfmas = [&](const Frag& F) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(F.a[i], F.b[j], acc[i][j], 0, 0, 0);
  };

  const int kt0 = blockIdx.y * kq;
  const int nk = min(kq, K / 64 - kt0);
  auto kslice = [&](int i) { return (kt0 + min(i, nk - 1)) * 64; };
  Frag F0, F1;
  auto iter = [&](auto rs, int kt) {
    constexpr int R = decltype(rs)::value;
    gload(rs, kslice(kt + 2));
    fread(F0, R, 0);
    fread(F1, R, 1);
    mfmas(F0);
    fread(F0, R, 2);
    mfmas(F1);
    fread(F1, R, 3);
    mfmas(F0);
    mfmas(F1);
    sstore(std::integral_constant<int, R ^ 1>{});
    // MFMA slot s = 0..4*NMF-1 in issue order
    constexpr int WSTEP = 2;
    constexpr int NSLOT = 4 * NMF, GSLOTS = 3 * NMF, WSLOTS = (4 - WSTEP) * NMF;
    __builtin_amdgcn_sched_group_barrier(0x100, NRD, 0);  // DS read, k-step 0
#pragma unroll
    for (int s = 0; s < NSLOT; ++s) {
      const int m = s % NMF;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      if (s < 3 * NMF && m < NRD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
      if (s < GSLOTS) {
        const int g = (s + 1) * NLD / GSLOTS - s * NLD / GSLOTS;
        if (g == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM read
        if (g == 2) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        if (g == 3) __builtin_amdgcn_sched_group_barrier(0x020, 3, 0);
      }
      if (s >= WSTEP * NMF) {
        const int q = s - WSTEP * NMF;
        const int w = (q + 1) * NLD / WSLOTS - q * NLD / WSLOTS;
        if (w == 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // DS write
        if (w == 2) __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);
        if (w == 3) __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);
      }
    }
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };

  using AX = EpiAux<Epi>;
  using AuxT = typename AX::type;
  AuxT aux[2][TM * 4];
  auto tok = [&](int j) { return t_base + wt * WTT + j * 32 + (lane & 31); };
  auto fblk = [&](int i) { return f_base + wf * WFT + i * 32; };  // wave-uniform
  auto feat = [&](int i, int g) { return fblk(i) + 8 * g + 4 * khalf; };
  auto load_row = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    static_for<0, TM * 4>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      const int t = tok(q / 4), f = feat(i, q % 4);
      if (t < T && f < N) aux[i & 1][q] = AX::load(epi, t, f, fblk(i));
    });
  };

  // nk >= 1 for every split (the launcher checks (splits - 1) * kq < K / 64)
  gload(R0{}, kslice(0));
  gload(R1{}, kslice(1));
  sstore(R0{});
  lds_barrier();
  int kt = 0;
  for (; kt + 2 <= nk; kt += 2) {
    iter(R0{}, kt);
    iter(R1{}, kt + 1);
  }
  if (kt < nk) iter(R0{}, kt);
  // Straight-line epilogue with the operands one accumulator row ahead, as in
  // gemm_nt_kernel.
  load_row(std::integral_constant<int, 0>{});
  // EpiRows: the token part of the output addresses once per token, the
  // (feature block, token) part once per 4 quads, both outside the quads'
  // bounds tests (they read no memory)
  constexpr bool ROWS = EpiRows<Epi>::value;
  static_assert(!ROWS || !EpiSumSq<Epi>::value, "row-addressed epilogues return nothing");
  typename EpiRows<Epi>::Tok tkj[ROWS ? TM : 1];
  if constexpr (ROWS) {
    static_for<0, TM>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      tkj[j] = epi.tok(tok(j));
    });
  }
  float lane_sq = 0.f;
  static_for<0, FM>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    if constexpr (i + 1 < FM) load_row(std::integral_constant<int, i + 1>{});
    if constexpr (ROWS) {
      static_for<0, TM>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        const auto rc = epi.row(tkj[j], fblk(i));
        static_for<0, 4>([&](auto gc) {
          constexpr int g = decltype(gc)::value, q = 4 * j + g;
          const int t = tok(j), f = feat(i, g);
          if (t < T && f < N) {
            f32x4 v;
            v.x = acc[i][j][4 * g + 0];
            v.y = acc[i][j][4 * g + 1];
            v.z = acc[i][j][4 * g + 2];
            v.w = acc[i][j][4 * g + 3];
            epi.store_row(rc, f, v, aux[i & 1][q], fblk(i));
          }
        });
      });
    } else {
      static_for<0, TM * 4>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        constexpr int j = q / 4, g = q % 4;
        const int t = tok(j), f = feat(i, g);
        if (t < T && f < N) {
          f32x4 v;
          v.x = acc[i][j][4 * g + 0];
          v.y = acc[i][j][4 * g + 1];
          v.z = acc[i][j][4 * g + 2];
          v.w = acc[i][j][4 * g + 3];
          if constexpr (EpiSumSq<Epi>::value)
            lane_sq += AX::apply(epi, t, f, v, aux[i & 1][q], fblk(i));
          else
            AX::apply(epi, t, f, v, aux[i & 1][q], fblk(i));
        }
      });
    }
  });
  if constexpr (EpiSumSq<Epi>::value) {
    // The main loop ended on a barrier after its last LDS reads, so the
    // operand buffers are free for the per-wave totals.
    float* red = (float*)&sW[0][0];
    const float s = wave_sum(lane_sq);
    if (lane == 0) red[wave] = s;
    __syncthreads();
    if (tid == 0) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < WF * WT; ++w) tot += red[w];
      epi.sq_out[tile] = tot;
    }
  }
}

}  // namespace hb
