// fp32 MFMA products of any alignment and size on small output tiles, shared
// by the screened products (screened.hip) and the BSR products (bsr_flex.hip).
//
// A 512-thread workgroup forms an output tile of at most 64x64 over a
// sequence of 64-wide k-slabs. Its 8 wavefronts split the tile and each
// slab's k (Split below) and add their sums through LDS at the end. The
// caller's slab source loads slab s into registers and run() stages them
// through a 2-stage LDS ring, the loads three slabs ahead of the MFMAs.
// Unlike the direct-to-LDS kernels, which need 16-byte aligned rows and own a
// CU with 128x128 tiles, the loads take any element alignment and four times
// as many tiles fill the chip; the k split keeps two wavefronts on every SIMD
// where a CU gets a single tile, and two workgroups (72 KiB of LDS each)
// share a CU where it gets more.
//
// An operand has one of two forms (`i` is its row or column of the output):
//   ROW: k contiguous in memory, staged as [i][64 k]: one 16-byte LDS read
//        per 4 k of a lane;
//   COL: i contiguous in memory, staged as [64 k][i]: four 4-byte reads.
// Row strides in LDS are padded so that the reads are conflict-free. (COL
// tiles transposed in registers, so that their reads are 16-byte ones too,
// were no faster: with 8-byte loads 73 against 105 TF on 4096^3, as a
// vector-memory instruction waits for a gap between the SIMD's MFMAs and
// their number counts; with 16-byte loads of one operand per wavefront 90.)
// bf16 operands are widened exactly when they are staged.
#pragma once

#include "common.h"
#include "lds_dma.h"

namespace tsp {
namespace flex {

constexpr int KC = 64;    // k-slab width
constexpr int NTHR = 512;

// How the 8 wavefronts share the output tile and each slab's k: MS x MS
// MFMAs (32 or 16), WM x WN of them, the rest splitting k. DIAG: only the
// tile's diagonal MS x MS squares are formed (WM == WN, one wave each).
template <int MS_, int XN_, int YN_, bool DIAG_ = false>
struct Split {
  static constexpr int MS = MS_, XN = XN_, YN = YN_;
  static constexpr bool DIAG = DIAG_;
  static constexpr int WM = XN / MS, WN = DIAG ? 1 : YN / MS, KG = 8 / (WM * WN);
  static constexpr int NV = MS * MS / 64;  // accumulator elements per lane
  static constexpr int NOUT = NV / KG;     // results per lane
  static_assert(WM * WN * KG == 8 && NOUT * KG == NV, "");
  static __device__ int wave() { return (int)threadIdx.x >> 6; }
  static __device__ int x0() { return wave() % WM * MS; }
  static __device__ int y0() { return DIAG ? x0() : wave() / WM % WN * MS; }
  static __device__ int kg() { return wave() / (WM * WN); }
  // this lane's results out[v] of run(): column col() and row row(v) of the tile
  static __device__ int col() { return y0() + ((int)threadIdx.x & (MS - 1)); }
  static __device__ int row(int v) {
    const int e = kg() * NOUT + v, h = ((int)threadIdx.x & 63) / MS;
    return x0() + (MS == 32 ? 8 * (e >> 2) + 4 * h + (e & 3) : 4 * h + e);
  }
};

// Four elements at p of which the first `left` exist (the rest are zero), as
// loaded (wide loads at element alignment) and widened to fp32.
template <typename T>
struct Quad;
template <>
struct Quad<float> {
  typedef float v4 __attribute__((ext_vector_type(4), aligned(4)));
  f32x4 v;
  __device__ void load(const float* __restrict__ p, int64_t left) {
    v = f32x4{0.f, 0.f, 0.f, 0.f};
    if (left >= 4) {
      v = *(const v4*)p;
    } else {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (e < left) v[e] = p[e];
    }
  }
  __device__ f32x4 f32() const { return v; }
};
template <>
struct Quad<uint16_t> {
  typedef uint32_t v2 __attribute__((ext_vector_type(2), aligned(2)));
  u32x2 v;
  __device__ void load(const uint16_t* __restrict__ p, int64_t left) {
    v = u32x2{0u, 0u};
    if (left >= 4) {
      v = *(const v2*)p;
    } else {
      if (left > 0) v[0] = p[0];
      if (left > 1) v[0] |= (uint32_t)p[1] << 16;
      if (left > 2) v[1] = p[2];
    }
  }
  __device__ f32x4 f32() const {
    return f32x4{__builtin_bit_cast(float, v[0] << 16), __builtin_bit_cast(float, v[0] & 0xFFFF0000u),
                 __builtin_bit_cast(float, v[1] << 16), __builtin_bit_cast(float, v[1] & 0xFFFF0000u)};
  }
};

// An operand form: this thread's pieces of a slab and where they are staged.
template <typename T, int N>
struct Row {  // q[j] = k() .. + 3 of row i() + 32 j
  static constexpr int LD = KC + 4, FLOATS = N * LD, PIECES = N < 32 ? 1 : N / 32;
  Quad<T> q[PIECES];
  static __device__ int i() { return (int)threadIdx.x >> 4; }
  static __device__ int k() { return ((int)threadIdx.x & 15) * 4; }
  static __device__ bool idle() { return N < 32 && i() >= N; }
  // rows i0 .. and columns k0 .. of a row-major matrix (row stride ld); rows
  // at or past iend and columns at or past kend read as zero
  __device__ void load(const T* __restrict__ p, int64_t ld, int64_t i0, int64_t iend, int64_t k0, int64_t kend) {
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      const int64_t r = i0 + i() + 32 * j;
      q[j].load(p + r * ld + k0 + k(), r < iend && !idle() ? kend - k0 - k() : 0);
    }
  }
  __device__ void store(float* tile) const {
    if (idle()) return;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) *(f32x4*)(tile + (i() + 32 * j) * LD + k()) = q[j].f32();
  }
  // the operand of row i at k .. + 3
  static __device__ f32x4 read(const float* tile, int i, int k) { return *(const f32x4*)(tile + i * LD + k); }
};
template <typename T, int N, int MS>
struct Col {  // q[j] = i() .. + 3 of k row k() + KSTEP j
  // lane groups of a read take k rows 4 apart: they fall into different banks
  static constexpr int LD = N + (MS == 32 ? 8 : 4), FLOATS = KC * LD;
  static constexpr int TPR = N / 4, KSTEP = NTHR / TPR, PIECES = KSTEP >= KC ? 1 : KC / KSTEP;
  Quad<T> q[PIECES];
  static __device__ int k() { return (int)threadIdx.x / TPR; }
  static __device__ int i() { return (int)threadIdx.x % TPR * 4; }
  static __device__ bool idle() { return KSTEP > KC && k() >= KC; }
  // columns i0 .. of rows k0 .. of a row-major matrix (row stride ld); rows
  // at or past kend and columns at or past iend read as zero
  __device__ void load(const T* __restrict__ p, int64_t ld, int64_t k0, int64_t kend, int64_t i0, int64_t iend) {
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      const int64_t r = k0 + k() + KSTEP * j;
      q[j].load(p + r * ld + i0 + i(), r < kend && !idle() ? iend - i0 - i() : 0);
    }
  }
  __device__ void store(float* tile) const {
    if (idle()) return;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) *(f32x4*)(tile + (k() + KSTEP * j) * LD + i()) = q[j].f32();
  }
  static __device__ f32x4 read(const float* tile, int i, int k) {
    f32x4 r;
#pragma unroll
    for (int t = 0; t < 4; ++t) r[t] = tile[(k + t) * LD + i];
    return r;
  }
};

template <class XF, class YF>
constexpr int lds_floats() {
  return 2 * (XF::FLOATS + YF::FLOATS) < 8192 ? 8192 : 2 * (XF::FLOATS + YF::FLOATS);
}

// out = the product over `nsteps` slabs, this lane's elements (S::row,
// S::col). src.load(s, r) fetches slab s into r.x and r.y (Row or Col; called
// once for every slab, in order) and src.finish(r) is called on it before it
// is staged, when the loads have landed. lds: lds_floats() floats.
template <class S, class Src>
__device__ inline void run(Src& src, int nsteps, float* lds, float (&out)[S::NOUT]) {
  typedef decltype(Src::Regs::x) XF;
  typedef decltype(Src::Regs::y) YF;
  constexpr int STAGE = XF::FLOATS + YF::FLOATS;
  constexpr int MS = S::MS, GK = 256 / MS;    // k per group: one f32x4 per lane and operand
  constexpr int NG = KC / GK / S::KG;         // groups of this wave's part of a slab
  typedef float acc_t __attribute__((ext_vector_type(S::NV)));
  const int lane = threadIdx.x & 63, l = lane % MS, h = lane / MS;
  const int xi = S::x0() + l, yi = S::y0() + l, k0 = S::kg() * NG * GK + 4 * h;
  acc_t acc = {};

  auto store = [&](int stage, typename Src::Regs& r) {
    src.finish(r);
    r.x.store(lds + stage * STAGE);
    r.y.store(lds + stage * STAGE + XF::FLOATS);
  };
  // One slab: its operand reads are issued first, then the next slab's stage
  // is written and the loads of a later one are issued, so that both run
  // under the MFMAs. A group's k-step t takes k = 4 h + t of lane group h on
  // both operands, so the sum is over the same k pairs.
  auto step = [&](int s, int stage, typename Src::Regs& next) {
    f32x4 a[NG], b[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      a[g] = XF::read(lds + stage * STAGE, xi, k0 + GK * g);
      b[g] = YF::read(lds + stage * STAGE + XF::FLOATS, yi, k0 + GK * g);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (s + 1 < nsteps) store(stage ^ 1, next);
    if (s + 3 < nsteps) src.load(s + 3, next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if constexpr (MS == 32)
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g][t], b[g][t], acc, 0, 0, 0);
        else
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[g][t], b[g][t], acc, 0, 0, 0);
      }
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
  // the k parts: each wave keeps its own share of its elements and adds the
  // other parts' in their order (the last slab ended with a barrier, so the
  // ring is free)
  float* const part = lds + lane;
  constexpr int WS = 64 * S::NV, PS = S::WM * S::WN * WS;  // floats of a wave, of a k part
  const int wt = S::wave() % (S::WM * S::WN);
#pragma unroll
  for (int v = 0; v < S::NV; ++v) part[S::kg() * PS + wt * WS + 64 * v] = acc[v];
  tsp::dma::barrier();
#pragma unroll
  for (int v = 0; v < S::NOUT; ++v) {
    float sum = 0.f;
#pragma unroll
    for (int kg = 0; kg < S::KG; ++kg) sum += part[kg * PS + wt * WS + 64 * (S::kg() * S::NOUT + v)];
    out[v] = sum;
  }
}

}  // namespace flex
}  // namespace tsp
