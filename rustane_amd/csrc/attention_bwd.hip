// Fused causal attention backward (kernels/sdpa_bwd.rs:46-161), flash style:
//   P = softmax(Q K^T scale) is recomputed from the forward's per-query
//   log-sum-exp, dP = dO V^T, D = rowsum(P * dP), dS = P (dP - D) scale,
//   dQ = dS K, dK = dS^T Q, dV = P^T dO,
// with every score block kept in registers: nothing of size S^2 goes to
// memory. The arithmetic per element is the unfused path's (fp32 scores and
// dP, P and dS rounded to fp16 as MFMA operands, D summed in fp32 from the
// unrounded P and dP), in a different summation order.
//
// Both kernels use the forward kernel's 32x32x16 MFMA layouts (attention.hip):
// a row tile [32][hd] is read as A-operand rows in swap23 slot order (chunk c
// of row r at r*NCH + (c ^ (swap23(r) % NCH))), so the 8 accumulator
// registers 8j..8j+7 of lane half h2 hold the consecutive rows 16j+8h2..+7
// and serve directly as a B operand. The same tile also gives the transposed
// A operand (one feature, 8 consecutive rows) through ds_read_b64_tr_b16
// (TrFrag), so no transposed copies exist in memory or LDS.
//
// Tiles go from global memory straight into LDS (dma_1k) one or two
// iterations ahead, with one barrier per iteration; a workgroup is 4 waves. The
// dQ instances and the wide dK/dV ones (PH = 1) use at most 256 registers, two
// workgroups to a CU, so that one's softmax and waits run under the other's
// MFMAs; dK/dV with two query halves takes 384 at hd = 128, one to a CU, on
// grids that give a CU no second one. The predecessors (register-staged
// double-buffered tiles, transposed copies, one workgroup of 4 waves per CU)
// spent most of an iteration waiting: 20 heads x 2048 of 128, us: dQ 337 ->
// 139, dK/dV 326 -> 118; 32 heads x 4 x 512, 70 -> 58 and 98 -> 49; 32 heads x
// 512, split ranges, 45 -> 34 and 42 -> 31.
//
// attn_bwd_dq_kernel, per (PQ query blocks, head, sequence), PQ x PK waves
// (PK key parts): S^T = K Q^T and dP^T = V dO^T per key block, two passes
// over the keys (D first, then dQ^T += K^T dS^T); with two key halves
// (PQ = 2, as the forward) the halves add their D and dQ through LDS.
//
// attn_bwd_dkv_kernel, per (PB key blocks, sequence and KV head), PB x PH
// waves (PH query parts): the wave's K and V rows stay in registers
// as B operands, S = Q K^T and dP = dO V^T per query block of every head of
// the group (the GQA sum over heads is the loop), dV^T += dO^T P and
// dK^T += Q^T dS; with two query halves (PB = 2) the halves add their
// partials through LDS.
#include "attention_tiles.hpp"
#include "internal.hpp"

namespace hb {

namespace {

// dQKV row and transpose of 4 consecutive features f0..f0+3 of token
// (b, s), column col. Q and K gradients go through the inverse of the
// forward's RoPE rotation at position s (layer.rs:1880-1897
// rope_backward_inplace): dx[2i] = d[2i] c + d[2i+1] s, dx[2i+1] = d[2i+1] c
// - d[2i] s.
HB_DEV void store_grad4(const AttnBwd& p, int b, int s, int col, int f0, f32x4 v, bool rope) {
  f32x4 o = v;
  if (rope) {
    const float4 r = p.rope[(size_t)(f0 >> 2) * p.rope_ld + s];  // f0 % 4 == 0
    const float2 c0 = make_float2(r.x, r.y), c1 = make_float2(r.z, r.w);
    o.x = v.x * c0.x + v.y * c0.y;
    o.y = v.y * c0.x - v.x * c0.y;
    o.z = v.z * c1.x + v.w * c1.y;
    o.w = v.w * c1.x - v.z * c1.y;
  }
  f16x4 h;
  h.x = (f16)o.x;
  h.y = (f16)o.y;
  h.z = (f16)o.z;
  h.w = (f16)o.w;
  const int tok = b * p.S + s;
  *(f16x4*)(p.dqkv + (size_t)tok * p.ld + col) = h;
  p.dqkvT[(size_t)col * p.tld + tok] = h.x;
  p.dqkvT[(size_t)(col + 1) * p.tld + tok] = h.y;
  p.dqkvT[(size_t)(col + 2) * p.tld + tok] = h.z;
  p.dqkvT[(size_t)(col + 3) * p.tld + tok] = h.w;
}

}  // namespace

template <int HD, int PQ, int PK>
__global__ __launch_bounds__(PQ * PK * 64, 2) void attn_bwd_dq_kernel(AttnBwd p) {
  constexpr int PW = PQ * PK;  // waves: query blocks x key parts
  constexpr int KS = HD / 16, MB = HD / 32, NCH = HD / 8, KT8 = 4 * HD;
  constexpr int NB = PK == 1 ? 3 : 2;  // tile buffers: K and V rows of PK key blocks each
  using Dma = TileDma<HD, PW, 2, PK>;
  constexpr int NTILE = 2 * PK * KT8, NMERGE = PK == 2 ? PQ * MB * 16 * 64 * 4 / 16 : 0;
  __shared__ f16x8 s_t[NB * NTILE > NMERGE ? NB * NTILE : NMERGE];
  __shared__ float s_d[PQ][64];

  const int tid = threadIdx.x, lane = tid & 63, h2 = lane >> 5, li = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qs = wave % PQ, kh = wave / PQ;
  const int nqb = (p.S + 31) / 32, ngr = (nqb + PQ - 1) / PQ;
  const int gr = ngr - 1 - blockIdx.x;  // heaviest groups first
  // query blocks gr, gr + ngr, ...: every group spans the sequence, so the
  // groups' causal work is nearly equal
  const int qb = gr + ngr * qs;
  const bool active = qb < nqb;
  const int nkb = gr + ngr * min(PQ - 1, (nqb - 1 - gr) / ngr) + 1;
  const int h = blockIdx.y, b = blockIdx.z;
  const int kvh = h / (p.H / p.KVH), z = b * p.KVH + kvh;
  const int qi = qb * 32 + li;
  const bool qok = active && qi < p.S;
  const size_t qrow = ((size_t)b * p.H + h) * p.Sp;

  f16x8 qf[KS], df[KS];
  float L2 = 0.f;
  if (active) {
    const size_t qo = (qrow + qi) * HD + 8 * h2;
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      qf[j] = *(const f16x8*)(p.q + qo + 16 * j);
      df[j] = *(const f16x8*)(p.dO + qo + 16 * j);
    }
    if (qi < p.S) L2 = p.lse[qrow + qi];
  }
  settle(qf);
  settle(df);
  asm volatile("" : "+v"(L2));

  const Dma dma({p.k + (size_t)z * p.Sp * HD, p.v + (size_t)z * p.Sp * HD}, lds_addr(s_t), wave, lane);
  const TrFrag<HD> tr(lane);
  const float sl2 = p.scale * HB_LOG2E;
  const int krow = swap23(li);
  const int niter = (nkb + PK - 1) / PK;
  auto issue = [&](int n, int buf) {
    dma.issue(buf, [&](int part) { return min(n * PK + part, nkb - 1) * 32; });
  };
  // the key loop of one pass: body(n, tiles) on every iteration's tiles, the
  // copies NB - 1 iterations ahead. The barrier of iteration n follows every
  // wave's wait for its own copies of n and its last read of n - 1, whose
  // buffer the new copies go into.
  auto keyloop = [&](auto&& body) {
    raw_barrier();  // the other waves are done with LDS
    issue(0, 0);
    if (NB == 3 && niter > 1) issue(1, 1);
    int buf = 0;
    for (int n = 0; n < niter; ++n) {
      if (NB == 3 && n + 1 < niter)
        dma_wait<Dma::NI>();
      else
        dma_wait<0>();
      raw_barrier();
      if (n + NB - 1 < niter) issue(n + NB - 1, buf == 0 ? NB - 1 : buf - 1);
      body(n, s_t + buf * NTILE);
      buf = buf == NB - 1 ? 0 : buf + 1;
    }
  };
  // S^T and dP^T of key block kb against this wave's queries; s becomes P
  auto block = [&](const f16x8* st, int kb, f32x16& s, f32x16& dp) {
    const f16x8* sk = st + kh * KT8;
    const f16x8* sv = st + (PK + kh) * KT8;
    s = f32x16{};
    dp = f32x16{};
    f16x8 kf[KS];
#pragma unroll
    for (int j = 0; j < KS; ++j) kf[j] = sk[krow * NCH + ((2 * j + h2) ^ (li % NCH))];
#pragma unroll
    for (int j = 0; j < KS; ++j) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j], qf[j], s, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < KS; ++j) kf[j] = sv[krow * NCH + ((2 * j + h2) ^ (li % NCH))];
#pragma unroll
    for (int j = 0; j < KS; ++j) dp = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j], df[j], dp, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = s[r] * sl2 - L2;
    // keys after the query exist in its diagonal block only (padding keys
    // come after every valid query); queries past S are never stored
    if (kb == qb) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (kb * 32 + swap23(8 * (r >> 2) + 4 * h2 + (r & 3)) > qi) s[r] = -INFINITY;
    }
    // v_exp_f32 itself: what exp2f's range scaling would add, results below
    // 2^-126, is 0 in every use
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(s[r]);
  };

  // pass 1: D = rowsum(P * dP) over this wave's key half, then over both
  float dsum = 0.f;
  keyloop([&](int n, const f16x8* st) {
    const int kb = n * PK + kh;
    if (!active || kb > qb) return;  // wave-uniform
    f32x16 s, dp;
    block(st, kb, s, dp);
#pragma unroll
    for (int r = 0; r < 16; ++r) dsum += s[r] * dp[r];
  });
  dsum += __shfl_xor(dsum, 32, 64);  // both lanes of a query pair
  float D = dsum;
  if constexpr (PK == 2) {
    if (kh == 1) s_d[qs][lane] = dsum;
    lds_barrier();
    const float Dq = kh == 0 ? dsum + s_d[qs][lane] : 0.f;
    lds_barrier();
    if (kh == 0) s_d[qs][lane] = Dq;
    lds_barrier();
    D = s_d[qs][lane];
  }
  if (kh == 0 && qok && h2 == 0) p.D[qrow + qi] = D;

  // pass 2: dS^T = P (dP - D) scale, dQ^T += K^T dS^T
  f32x16 o[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) o[m] = f32x16{};
  keyloop([&](int n, const f16x8* st) {
    const int kb = n * PK + kh;
    if (!active || kb > qb) return;
    f32x16 s, dp;
    block(st, kb, s, dp);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = s[r] * (dp[r] - D) * p.scale;
    const f16x8* sk = st + kh * KT8;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f16x8 db;
#pragma unroll
      for (int i = 0; i < 8; ++i) db[i] = (f16)s[8 * j + i];
#pragma unroll
      for (int m = 0; m < MB; ++m)
        o[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(tr.read(sk, m, j), db, o[m], 0, 0, 0);
    }
  });

  // with two key halves, half 1 hands its dQ^T to half 0 (same lane, same
  // slots) through the tile buffers
  if constexpr (PK == 2) {
    raw_barrier();  // every wave's copies were waited for, its reads are done
    float* s_o = (float*)s_t + qs * (MB * 16 * 64);
    if (kh == 1) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) s_o[(m * 16 + r) * 64 + lane] = o[m][r];
    }
    lds_barrier();
    if (kh == 1) return;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[m][r] += s_o[(m * 16 + r) * 64 + lane];
  }
  if (!qok) return;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int f0 = m * 32 + 8 * g + 4 * h2;
      f32x4 v;
      v.x = o[m][4 * g + 0];
      v.y = o[m][4 * g + 1];
      v.z = o[m][4 * g + 2];
      v.w = o[m][4 * g + 3];
      store_grad4(p, b, qi, h * HD + f0, f0, v, true);
    }
}

template <int HD, int PB, int PH>
__global__ __launch_bounds__(PB * PH * 64, PH == 1 ? 2 : 1) void attn_bwd_dkv_kernel(AttnBwd p) {
  constexpr int PW = PB * PH;  // waves: key blocks x query parts
  constexpr int KS = HD / 16, MB = HD / 32, NCH = HD / 8, KT8 = 4 * HD;
  constexpr int NB = 2;  // tile buffers: Q and dO rows of PH query blocks each
  // The K and V rows, dK, dV, S and dP are 224 registers at hd = 128: with two
  // workgroups per CU (PH = 1) each wave keeps its V rows in LDS instead.
  constexpr bool VLDS = PH == 1 && HD == 128;
  using Dma = TileDma<HD, PW, 2, PH>;
  constexpr int NTILE = 2 * PH * KT8, NMERGE = PH == 2 ? PB * 2 * MB * 16 * 64 * 4 / 16 : 0;
  __shared__ f16x8 s_t[NB * NTILE > NMERGE ? NB * NTILE : NMERGE];
  // log-sum-exp and D of the iteration's query blocks: [part][lse, D][64], the
  // upper 32 of each a copy of the lower
  __shared__ __align__(16) float s_ld[NB][PH][2][64];
  static_assert(PW >= 2 * PH, "a wave copies one row of s_ld");
  __shared__ f16x8 s_v[VLDS ? PB * KT8 : 1];

  const int tid = threadIdx.x, lane = tid & 63, h2 = lane >> 5, li = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kbi = wave % PB, qh = wave / PB;
  const int nb = (p.S + 31) / 32;  // key blocks = query blocks
  const int grp = blockIdx.x;      // group 0 sees the most query blocks: launched first
  // key blocks grp, grp + ngr, ...: every group spans the sequence, so the
  // groups' causal work is nearly equal
  const int ngr = (nb + PB - 1) / PB;
  const int kb = grp + ngr * kbi;
  const bool active = kb < nb;
  const int z = blockIdx.y, b = z / p.KVH, g = z - b * p.KVH;
  const int rep = p.H / p.KVH;
  const int ki = kb * 32 + li;
  const int qstart = grp;              // first query block that sees the group's keys
  const int nq = nb - qstart;           // query blocks per head
  const int npairs = rep * nq;          // (head, query block) pairs
  const int niter = (npairs + PH - 1) / PH;

  f16x8 kf[KS], vf[VLDS ? 1 : KS];
  if (active) {
    const size_t ko = ((size_t)z * p.Sp + ki) * HD + 8 * h2;
#pragma unroll
    for (int j = 0; j < KS; ++j) {
      kf[j] = *(const f16x8*)(p.k + ko + 16 * j);
      if constexpr (!VLDS) vf[j] = *(const f16x8*)(p.v + ko + 16 * j);
    }
    if constexpr (VLDS) {  // this wave's own rows: its first dma_wait covers them
      const i32x4 vrs = dma_rsrc(p.v + (size_t)z * p.Sp * HD);
#pragma unroll
      for (int n = 0; n < HD / 16; ++n) {
        const int row = n * (64 / NCH) + lane / NCH;
        dma_1k(lds_addr(s_v) + kbi * (HD * 64) + n * 1024,
               (uint32_t)(row * HD + ((lane % NCH) ^ (swap23(row) % NCH)) * 8) * 2u, vrs,
               (uint32_t)kb * (uint32_t)(HD * 64));
      }
    }
  }
  // LDS chunks of fragment j: base ^ 2j. The bases are made opaque in each
  // iteration: hoisted out of the loop, the 16 addresses would spill.
  const int qbase = swap23(li) * NCH + (h2 ^ (li % NCH)), vbase = li * NCH + (h2 ^ (swap23(li) % NCH));
  auto vfrag = [&](int j, int vo) -> f16x8 {
    if constexpr (VLDS)
      return s_v[kbi * KT8 + (vo ^ (2 * j))];
    else
      return vf[j];
  };

  // rows of the group's heads: row r*Sp + q of head g*rep + r, query q
  const size_t grow = ((size_t)b * p.H + (size_t)g * rep) * p.Sp;
  const Dma dma({p.q + grow * HD, p.dO + grow * HD}, lds_addr(s_t), wave, lane);
  const TrFrag<HD> tr(lane);
  auto pair_row = [&](int n, int hq) {  // first row of the iteration's query block
    const int pi = min(n * PH + hq, npairs - 1), r = pi / nq;
    return r * p.Sp + (qstart + (pi - r * nq)) * 32;
  };
  // s_ld: waves beyond 2 * PH repeat the copy of wave % (2 * PH)
  const int ldw = wave % (2 * PH);
  const i32x4 ldrs = dma_rsrc((ldw & 1 ? p.D : p.lse) + grow);
  const uint32_t ld_lds = lds_addr(&s_ld[0][0][0][0]) + ldw * 256;
  auto issue = [&](int n, int buf) {
    dma.issue(buf, [&](int part) { return pair_row(n, part); });
    dma_256(ld_lds + buf * (uint32_t)sizeof(s_ld[0]), (uint32_t)li * 4u, ldrs,
            (uint32_t)pair_row(n, ldw >> 1) * 4u);
  };

  const float sl2 = p.scale * HB_LOG2E;
  f32x16 dk[MB], dv[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    dk[m] = f32x16{};
    dv[m] = f32x16{};
  }
  auto body = [&](int n, int buf) {
    const int pi = n * PH + qh;
    if (!active || pi >= npairs) return;  // wave-uniform
    const int qb = qstart + pi % nq;
    if (qb < kb) return;  // every query of the block precedes every key
    const f16x8* sq = s_t + buf * NTILE + qh * KT8;
    const f16x8* sd = s_t + buf * NTILE + (PH + qh) * KT8;
    f32x16 s = {}, dp = {};
    int qo = qbase, vo = vbase;
    asm volatile("" : "+v"(qo), "+v"(vo));
    constexpr int KH = KS / 2;  // fragments at a time: the registers are full
#pragma unroll
    for (int j0 = 0; j0 < KS; j0 += KH) {
      f16x8 f[KH];
#pragma unroll
      for (int j = 0; j < KH; ++j) f[j] = sq[qo ^ (2 * (j0 + j))];
#pragma unroll
      for (int j = 0; j < KH; ++j) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[j], kf[j0 + j], s, 0, 0, 0);
    }
#pragma unroll
    for (int j0 = 0; j0 < KS; j0 += KH) {
      f16x8 f[KH];
#pragma unroll
      for (int j = 0; j < KH; ++j) f[j] = sd[qo ^ (2 * (j0 + j))];
#pragma unroll
      for (int j = 0; j < KH; ++j) dp = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[j], vfrag(j0 + j, vo), dp, 0, 0, 0);
    }
    // rows are the queries qb*32 + 16j + 8h2 + i (registers 8j + i), columns
    // this lane's key ki
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const f32x4 l = *(const f32x4*)&s_ld[buf][qh][0][16 * (e >> 3) + 8 * h2 + (e & 7)];
#pragma unroll
      for (int i = 0; i < 4; ++i) s[e + i] = s[e + i] * sl2 - l[i];
    }
    // masked entries only in the diagonal block and where the sequence ends
    if (qb == kb || (qb + 1) * 32 > p.S) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int qpos = qb * 32 + 16 * (e >> 3) + 8 * h2 + (e & 7);
        if (ki > qpos || qpos >= p.S) s[e] = -INFINITY;
      }
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = __builtin_amdgcn_exp2f(s[e]);
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const f32x4 d = *(const f32x4*)&s_ld[buf][qh][1][16 * (e >> 3) + 8 * h2 + (e & 7)];
#pragma unroll
      for (int i = 0; i < 4; ++i) dp[e + i] = s[e + i] * (dp[e + i] - d[i]) * p.scale;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f16x8 pb, db;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        pb[i] = (f16)s[8 * j + i];
        db[i] = (f16)dp[8 * j + i];
      }
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        dv[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(tr.read(sd, m, j), pb, dv[m], 0, 0, 0);
        dk[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(tr.read(sq, m, j), db, dk[m], 0, 0, 0);
      }
    }
  };
  // as the dQ kernel's key loop, one iteration ahead
  issue(0, 0);
  settle(kf);
  settle(vf);
  for (int n = 0; n < niter; ++n) {
    dma_wait<0>();
    raw_barrier();
    if (n + 1 < niter) issue(n + 1, (n + 1) & 1);
    body(n, n & 1);
  }

  // with two query halves, half 1 hands its dK^T and dV^T to half 0 of the
  // same key block through the tile buffers
  if constexpr (PH == 2) {
    raw_barrier();  // every wave's copies were waited for, its reads are done
    float* s_o = (float*)s_t + kbi * (2 * MB * 16 * 64);
    if (qh == 1) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          s_o[(m * 16 + e) * 64 + lane] = dk[m][e];
          s_o[((MB + m) * 16 + e) * 64 + lane] = dv[m][e];
        }
    }
    lds_barrier();
    if (qh == 1) return;
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        dk[m][e] += s_o[(m * 16 + e) * 64 + lane];
        dv[m][e] += s_o[((MB + m) * 16 + e) * 64 + lane];
      }
  }
  if (!active || ki >= p.S) return;
  const int colk = p.q_dim + g * HD, colv = p.q_dim + p.kv_dim + g * HD;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int f0 = m * 32 + 8 * q4 + 4 * h2;
      f32x4 a, c;
      a.x = dk[m][4 * q4 + 0];
      a.y = dk[m][4 * q4 + 1];
      a.z = dk[m][4 * q4 + 2];
      a.w = dk[m][4 * q4 + 3];
      c.x = dv[m][4 * q4 + 0];
      c.y = dv[m][4 * q4 + 1];
      c.z = dv[m][4 * q4 + 2];
      c.w = dv[m][4 * q4 + 3];
      store_grad4(p, b, ki, colk + f0, f0, a, true);
      store_grad4(p, b, ki, colv + f0, f0, c, false);
    }
}

namespace {
// Four query (dQ) or key (dK/dV) blocks per workgroup share each staged tile
// once that gives every CU a workgroup; otherwise two blocks, with the key or
// query range split in halves.
constexpr long HB_BWD_WIDE_MIN = 256;
template <int HD>
void launch_bwd(const AttnBwd& p, hipStream_t st) {
  const int nb = (p.S + 31) / 32;
  const long hb = (long)p.H * p.B, zb = (long)p.KVH * p.B;
  if ((long)((nb + 3) / 4) * hb >= HB_BWD_WIDE_MIN)
    hipLaunchKernelGGL((attn_bwd_dq_kernel<HD, 4, 1>), dim3((nb + 3) / 4, p.H, p.B), dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((attn_bwd_dq_kernel<HD, 2, 2>), dim3((nb + 1) / 2, p.H, p.B), dim3(256), 0, st, p);
  if ((long)((nb + 3) / 4) * zb >= HB_BWD_WIDE_MIN)
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<HD, 4, 1>), dim3((nb + 3) / 4, p.B * p.KVH), dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<HD, 2, 2>), dim3((nb + 1) / 2, p.B * p.KVH), dim3(256), 0, st, p);
}
}  // namespace

hipError_t attention_backward_fused(const AttnBwd& p, hipStream_t st) {
  if (p.S < 1 || p.Sp < p.S || p.Sp % 32 || p.H % p.KVH || (p.hd != 64 && p.hd != 128) || !p.lse || !p.D)
    return hipErrorInvalidValue;
  if (p.hd == 128)
    launch_bwd<128>(p, st);
  else
    launch_bwd<64>(p, st);
  return hipGetLastError();
}

}  // namespace hb
