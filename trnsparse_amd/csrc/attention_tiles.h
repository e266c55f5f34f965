// LDS tiles of the attention kernels' MFMA operands: bf16 rows (abw) and fp32
// rows (abf) of head_dim D, read as the operand of products over head_dim
// (rows) and of products over rows (bf16: transpose reads).
#pragma once

#include "common.h"

#include "lds_dma.h"

namespace tsp {

namespace abw {
constexpr int BS = 128;             // block size served by the MFMA kernels
constexpr int HR = 64;              // rows (keys in the row pass, queries in the column pass) per ring stage
constexpr int SEG_MAX = 64;         // most block rows one column-pass item walks
template <int D>
struct Geo {
  static constexpr int ROWB = D * 2;                // bytes per row
  static constexpr int HBYTES = HR * ROWB;          // a half: 64 rows
  static constexpr int KS = D / 16;                 // k-steps over head_dim
  static constexpr int NU = D / 32;                 // 32-wide head_dim subtiles
  static constexpr int LOADS = 2 * HBYTES / 4096;   // 1-KiB loads per wave of two operands' halves
};
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

// The 16-byte chunk c of stage row r sits in slot c ^ swz(r). Rows are read
// as 16-byte pieces of 16 consecutive rows (one chunk) and through transpose
// reads of 4 consecutive rows (4 chunks). At d = 128 (256-byte rows, 16
// chunks) swz is a bijection on r % 16 whose low two bits follow r / 4 and
// high two bits r % 4; at d = 64 two rows share the 64 banks and the 8 chunks
// of a row follow r / 2: its parity in the high bit, r / 4 in the low two. So
// both access forms hit 16 (resp. 4 x 4) distinct slots.
template <int D>
__host__ __device__ constexpr int swz(int r) {
  return D == 128 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
}

// One wave's share (rows [16w, 16w + 16)) of a 64-row half starting at global
// row row0 of the buffer `rs`, into the stage at LDS address dst.
template <int D>
__device__ inline void dma_half(tsp::dma::i32x4 rs, int64_t row0, uint32_t dst, int w, int lane) {
  constexpr int ROWB = Geo<D>::ROWB, CPR = ROWB / 16, RPI = 64 / CPR;  // chunks per row, rows per instruction
#pragma unroll
  for (int qq = 0; qq < Geo<D>::LOADS / 2; ++qq) {
    const int j = Geo<D>::LOADS / 2 * w + qq;
    const int rr = RPI * j + lane / CPR;
    const int p = lane % CPR;
    tsp::dma::buffer16(rs, (uint32_t)((row0 + rr) * ROWB + ((p ^ swz<D>(rr)) << 4)), dst + j * 1024);
  }
}

// A operand holding the transpose: rows (MFMA i) are head_dim 32u + l32 and
// the 8 k values are stage rows r0 + 4h + {0..3} and r0 + 8 + 4h + {0..3}
// (the k order of the lane's own accumulator rows), from two
// ds_read_b64_tr_b16: lane j of 16-lane group gq points at row
// r0 + 8 rr + 4 (gq / 2) + j / 4, column 32u + 16 (gq % 2) + 4 (j % 4).
struct TrLane {
  int off[2];
  int xu;
};
template <int D>
__device__ inline TrLane tr_lane(int lane) {
  const int gq = lane >> 4, jq = lane & 15;
  const int c0 = 2 * (gq & 1) + ((jq & 3) >> 1);
  TrLane t;
#pragma unroll
  for (int rr = 0; rr < 2; ++rr) {
    const int row = 8 * rr + 4 * (gq >> 1) + (jq >> 2);
    t.off[rr] = row * Geo<D>::ROWB + ((c0 ^ (swz<D>(row) & 3)) << 4) + 8 * (jq & 1);
  }
  t.xu = D == 128 ? jq >> 2 : jq >> 3;  // swz(row) >> 2
  return t;
}
// Address form of the two reads for the slot kernels. A stage starts at an
// LDS address that is a multiple of 256 and rows are 256 (d = 64: 128) bytes,
// so the swizzled chunk bits (4-7, 4-6) of a lane's address are free in the stage base:
// per step one base per access kind is formed (row reads: stage + l32 * ROWB
// + swz(l32)^h in bits 4-7; transpose reads: stage + off[rr] + xu in bits
// 6-7) and each read is base ^ (k-step or subtile bits) plus a constant row
// offset that the ds_read immediate absorbs.
// Round 4 floats to bf16 (round to nearest even, v_cvt_pk_bf16_f32) as 4 halfwords.
__device__ inline u16x4 bf16x4_rne(f32x4 v) {
  return __builtin_bit_cast(u16x4, __builtin_convertvector(v, bf16x4));
}


typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
__device__ inline bf16x8 lds_row(uint32_t rb, int ks, uint32_t off) {
  return *(const lds_bf16x8*)(uintptr_t)((rb ^ (uint32_t)(ks << 5)) + off);
}
__device__ inline bf16x8 lds_trp(uint32_t tb0, uint32_t tb1, int u, uint32_t off) {
  const s16x4 r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)((tb0 ^ (uint32_t)(u << 6)) + off));
  const s16x4 r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)((tb1 ^ (uint32_t)(u << 6)) + off));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(r0, r1, 0, 1, 2, 3, 4, 5, 6, 7));
}
}  // namespace abw

namespace abf {
template <int D>
struct Cfg {
  static constexpr int BS = 128;
  static constexpr int HR = 4096 / D;       // rows per ring stage
  static constexpr int ROWB = D * 4;        // bytes per row
  static constexpr int HBYTES = HR * ROWB;  // 16 KiB
  static constexpr int NT = HR / 32;        // 32-row tiles per stage
  static constexpr int NU = D / 32;         // head_dim subtiles of row products
  static constexpr int KT = D / 8;          // b128 chunk reads per 32-row tile
  static constexpr int SPB = BS / HR;       // stages per block
};
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int NU> struct VRow;
template <> struct VRow<4> { typedef f32x4 type; };
template <> struct VRow<2> { typedef f32x2 type; };

// One wave's share of a stage: rows [row0, row0 + HR) of the buffer rs into
// LDS dst, 16 instructions of 1 KiB, 4 per wave.
template <int D>
__device__ inline void dma_rows(tsp::dma::i32x4 rs, int64_t row0, uint32_t dst, int w, int lane) {
  constexpr int LPR = D / 4, RPI = 64 / LPR, ROWB = D * 4;
#pragma unroll
  for (int qq = 0; qq < 4; ++qq) {
    const int j = 4 * w + qq;
    const int rr = RPI * j + lane / LPR;
    const int p = lane % LPR;
    tsp::dma::buffer16(rs, (uint32_t)((row0 + rr) * ROWB + ((p ^ (rr & 15)) << 4)), dst + j * 1024);
  }
}
// chunk read: logical chunk c of stage row `row` (row % 16 == kx)
template <int D>
__device__ inline f32x4 chunk_read(const uint8_t* base, int row, int c, int kx) {
  return *(const f32x4*)(base + row * (D * 4) + ((c ^ kx) << 4));
}
// row read: floats [NU * l32, NU * l32 + NU) of stage row `row`
template <int D>
__device__ inline typename VRow<D / 32>::type row_read(const uint8_t* base, int row, int l32) {
  constexpr int NU = D / 32;
  const int byte = NU * 4 * l32;
  return *(const typename VRow<NU>::type*)(base + row * (D * 4) + ((((byte >> 4) ^ (row & 15))) << 4) + (byte & 15));
}
// Store a 32-row x D tile held as NU accumulators (element v of subtile u is
// head_dim NU * (8 (v / 4) + 4 h + v % 4) + u of the lane's row) to dst, times f.
template <int D>
__device__ inline void store_rows(float* dst, const f32x16* acc, int h, float f) {
  constexpr int NU = D / 32;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    float* d = dst + NU * (8 * a + 4 * h);
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      f32x4 t;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int idx = 4 * k + e;
        t[e] = acc[idx % NU][4 * a + idx / NU] * f;
      }
      *(f32x4*)(d + 4 * k) = t;
    }
  }
}
}  // namespace abf

}  // namespace tsp
