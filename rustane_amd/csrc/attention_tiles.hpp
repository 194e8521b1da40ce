// Row tiles of the attention kernels: 32 rows of HD halves in LDS, 16-byte
// chunk c of row r at chunk r*NCH + (c ^ (swap23(r) % NCH)), NCH = HD / 8.
#pragma once
#include "common.hpp"

namespace hb {

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Transposed A fragments of a row tile. ds_read_b64_tr_b16: in each group of
// 16 lanes, lane s supplies 4 halves of its own address and lane i receives,
// as element e, half i%4 of lane 4e + i/4. With lane s at row base + s/4,
// features F + 4(s%4)..+3, lane i gets feature F + i of rows base..base+3.
// The fragment (m, j) of lane (h2, li) is feature m*32 + li of rows 16j + 8h2
// .. +7: two reads. The tile's chunk swizzle enters through the two lane
// bases (m even, odd); everything else is an immediate offset.
template <int HD>
struct TrFrag {
  static constexpr int NCH = HD / 8;
  int base[2];
  HB_DEV explicit TrFrag(int lane) {
    const int s = lane & 15, g = lane >> 4, h2 = lane >> 5;
#pragma unroll
    for (int mm = 0; mm < 2; ++mm) {
      const int c = mm * 4 + 2 * (g & 1) + ((s & 3) >> 1), x = (4 * h2 + (s >> 2)) % NCH;
      base[mm] = ((8 * h2 + (s >> 2)) * NCH + (c ^ x)) * 8 + 4 * (s & 1);
    }
  }
  HB_DEV f16x8 read(const f16x8* tile, int m, int j) const {
    const f16* t = (const f16*)tile + base[m & 1];
    s16x4 v[2];
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int off = (16 * j + 4 * hh) * NCH * 8 + (NCH == 16 ? ((hh ^ (m >> 1)) & 1) * 64 : 0);
      v[hh] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(__attribute__((address_space(3))) void*)(t + off));
    }
    const auto w = __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(f16x8, w);
  }
};

// Copies of one iteration's tiles by PW waves: tile kind * PARTS + part holds
// the 32 rows from row0(part) of base[kind]; NI instructions of 1 KB per wave.
template <int HD, int PW, int KINDS, int PARTS>
struct TileDma {
  static constexpr int NCH = HD / 8, IPT = HD / 16;  // instructions per tile
  static constexpr int NI = KINDS * PARTS * IPT / PW;
  static constexpr uint32_t BYTES = KINDS * PARTS * HD * 64;
  // instruction slot u of a wave belongs to one tile (PW <= IPT), or slot u of
  // PW / IPT groups of waves to as many parts of one kind
  static constexpr int NV = PW <= IPT ? IPT / PW : 1, TPS = PW <= IPT ? 1 : PW / IPT;
  static_assert(PW <= IPT ? IPT % PW == 0 : PW % IPT == 0 && PARTS % TPS == 0, "slots and tiles nest");
  struct Bases {
    const f16* p[KINDS];
  };
  uint32_t voff[NV];
  uint32_t lds;
  int wpart;
  i32x4 rs[KINDS];
  HB_DEV TileDma(const Bases& b, uint32_t lds0, int wave, int lane)
      : lds(lds0 + wave * 1024), wpart(PW <= IPT ? 0 : wave / IPT) {
#pragma unroll
    for (int k = 0; k < KINDS; ++k) rs[k] = dma_rsrc(b.p[k]);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int row = (PW <= IPT ? wave + PW * u : wave % IPT) * (64 / NCH) + lane / NCH;
      voff[u] = (uint32_t)(row * HD + ((lane % NCH) ^ (swap23(row) % NCH)) * 8) * 2u;
    }
  }
  // row0: part -> first row, wave-uniform
  template <class F>
  HB_DEV void issue(int buf, F&& row0) const {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int tile = PW <= IPT ? u * PW / IPT : u * TPS, kind = tile / PARTS;
      dma_1k(lds + buf * BYTES + u * PW * 1024, voff[u % NV], rs[kind],
             (uint32_t)row0(tile % PARTS + wpart) * (uint32_t)(HD * 2));
    }
  }
};

}  // namespace hb
