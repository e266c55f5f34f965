// fp32 MFMA products of any alignment and size on small output tiles.
//
// A 512-thread workgroup forms a 64x64 tile of X Y over a sequence of 64-wide
// k-slabs: four wavefronts of 32x32, twice, the two sets taking half of each
// slab's k and adding their sums through LDS at the end. The caller's slab
// source loads slab s into registers (two 16-byte pieces of each operand per
// thread) and run() stages them through a 2-stage LDS ring, the loads
// three slabs ahead of the MFMAs. Unlike the direct-to-LDS kernels, which need 16-byte aligned
// rows and own a CU with 128x128 tiles, the loads take any 4-byte alignment
// and four times as many tiles fill the chip; the k split keeps two
// wavefronts on every SIMD where a CU gets a single tile, and two workgroups
// (72 KiB of LDS each) share a CU where it gets more.
//
// An operand has one of two forms (`i` is its row or column of the output):
//   ROW: k contiguous in memory, staged as [64 i][64 k]: one 16-byte LDS read
//        per 8 k;
//   COL: i contiguous in memory, staged as [64 k][64 i]: four 4-byte reads.
// Row strides in LDS are padded so that the reads are conflict-free. (COL
// tiles transposed in registers, so that their reads are 16-byte ones too,
// were no faster: with 8-byte loads 73 against 105 TF on 4096^3, as a
// vector-memory instruction waits for a gap between the SIMD's MFMAs and
// their number counts; with 16-byte loads of one operand per wavefront 90.)
#pragma once

#include "common.h"
#include "lds_dma.h"

namespace tsp {
namespace flex {

constexpr int TM = 64;           // output tile: TM x TM
constexpr int KC = 64;           // k-slab width
constexpr int NTHR = 512;
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// p[0..3] where the first `left` elements exist; the rest read as zero.
__device__ inline f32x4 load4(const float* __restrict__ p, int64_t left) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (left >= 4) {
    v = *(const f32x4_u*)p;
  } else {
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (e < left) v[e] = p[e];
  }
  return v;
}

// An operand form: this thread's part of a slab, two pieces v[j] of 4
// elements along the contiguous dimension, and where it is staged.
struct Row {  // v[j] = k() .. + 3 of row i() + 32 j
  static constexpr int LD = KC + 4;  // floats per staged row
  f32x4 v[2];
  static __device__ int i() { return (int)threadIdx.x >> 4; }
  static __device__ int k() { return ((int)threadIdx.x & 15) * 4; }
  // rows i0 .. and columns k0 .. of a row-major matrix (row stride ld); rows
  // at or past iend and columns at or past kend read as zero
  __device__ void load(const float* __restrict__ p, int64_t ld, int64_t i0, int64_t iend, int64_t k0, int64_t kend) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t r = i0 + i() + 32 * j;
      v[j] = load4(p + r * ld + k0 + k(), r < iend ? kend - k0 - k() : 0);
    }
  }
  __device__ void store(float* tile) const {
#pragma unroll
    for (int j = 0; j < 2; ++j) *(f32x4*)(tile + (i() + 32 * j) * LD + k()) = v[j];
  }
  // the operand of row i over the 8 k from 8 g, lane half h's four
  static __device__ f32x4 read(const float* tile, int i, int g, int h) {
    return *(const f32x4*)(tile + i * LD + 8 * g + 4 * h);
  }
};
struct Col {  // v[j] = i() .. + 3 of k row k() + 32 j
  static constexpr int LD = TM + 8;  // floats per staged k: the lane halves' rows, 4 apart, use different banks
  f32x4 v[2];
  static __device__ int k() { return (int)threadIdx.x >> 4; }
  static __device__ int i() { return ((int)threadIdx.x & 15) * 4; }
  // columns i0 .. of rows k0 .. of a row-major matrix (row stride ld); rows
  // at or past kend and columns at or past iend read as zero
  __device__ void load(const float* __restrict__ p, int64_t ld, int64_t k0, int64_t kend, int64_t i0, int64_t iend) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t r = k0 + k() + 32 * j;
      v[j] = load4(p + r * ld + i0 + i(), r < kend ? iend - i0 - i() : 0);
    }
  }
  __device__ void store(float* tile) const {
#pragma unroll
    for (int j = 0; j < 2; ++j) *(f32x4*)(tile + (k() + 32 * j) * LD + i()) = v[j];
  }
  static __device__ f32x4 read(const float* tile, int i, int g, int h) {
    f32x4 r;
#pragma unroll
    for (int t = 0; t < 4; ++t) r[t] = tile[(8 * g + 4 * h + t) * LD + i];
    return r;
  }
};
constexpr int TILE_F = KC * Col::LD;  // floats per staged operand (the larger form)
constexpr int LDS_FLOATS = 4 * TILE_F;

// Position of this lane in the output tile: column `col`, and element v of
// its 8 results is row row(v).
struct Out {
  int rbase, col;
  __device__ Out() {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    rbase = (w & 1) * 32 + 4 * (lane >> 5) + 16 * (w >> 2);
    col = ((w >> 1) & 1) * 32 + (lane & 31);
  }
  __device__ int row(int v) const { return rbase + 8 * (v >> 2) + (v & 3); }
};

// out = the product over `nsteps` slabs, this lane's 8 elements (Out).
// src.load(s, r) fetches slab s into r.x and r.y (Row or Col; called once for
// every slab, in order) and src.finish(r) is called on it before it is
// staged, when the loads have landed.
template <class Src>
__device__ inline void run(Src& src, int nsteps, float* lds, float (&out)[8]) {
  typedef decltype(Src::Regs::x) XF;
  typedef decltype(Src::Regs::y) YF;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int h = lane >> 5, l32 = lane & 31, kg = w >> 2;
  const int xi = (w & 1) * 32 + l32, yi = ((w >> 1) & 1) * 32 + l32;
  constexpr int NG = KC / 16;  // 8-k groups of this wave's half
  f32x16 acc = {};

  auto store = [&](int stage, typename Src::Regs& r) {
    src.finish(r);
    r.x.store(lds + stage * 2 * TILE_F);
    r.y.store(lds + stage * 2 * TILE_F + TILE_F);
  };
  // One slab: its operand reads are issued first, then the next slab's stage
  // is written and the loads of a later one are issued, so that both run
  // under the MFMAs. Lane half h takes k = 8g + 4h + t at k-step t on both
  // operands, so the sum is over the same k pairs.
  auto step = [&](int s, int stage, typename Src::Regs& next) {
    f32x4 a[NG], b[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      a[g] = XF::read(lds + stage * 2 * TILE_F, xi, kg * NG + g, h);
      b[g] = YF::read(lds + stage * 2 * TILE_F + TILE_F, yi, kg * NG + g, h);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (s + 1 < nsteps) store(stage ^ 1, next);
    if (s + 3 < nsteps) src.load(s + 3, next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g][t], b[g][t], acc, 0, 0, 0);
    tsp::dma::barrier();
  };

  if (nsteps > 0) {
    // slab s + 1 waits in r1, slab s + 2 in r0 (s even; swapped for s odd)
    typename Src::Regs r0, r1;
    src.load(0, r0);
    if (nsteps > 1) src.load(1, r1);
    store(0, r0);
    if (nsteps > 2) src.load(2, r0);
    tsp::dma::barrier();
    for (int s = 0; s < nsteps; s += 2) {
      step(s, 0, r1);
      if (s + 1 < nsteps) step(s + 1, 1, r0);
    }
  }
  // the two k halves: each wave gives its partner (w ^ 4) half of its sums
  // and adds the partner's to the other half
  // (the last slab ended with a barrier, so the ring is free)
  float* const mine = lds + w * 512 + lane;
  const float* const other = lds + (w ^ 4) * 512 + lane;
#pragma unroll
  for (int v = 0; v < 8; ++v) mine[64 * v] = kg ? acc[v] : acc[8 + v];
  tsp::dma::barrier();
#pragma unroll
  for (int v = 0; v < 8; ++v) out[v] = (kg ? acc[8 + v] : acc[v]) + other[64 * v];
}

}  // namespace flex
}  // namespace tsp
