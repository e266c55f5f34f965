// BSR products on small output tiles (f32_flex.h): C = A B, its gradients
// dA = dC B^T on the pattern and dB = A^T dC (reference
// trnsparse/ops.py:162-192, nki/dispatch.py:290-369), for fp32 and bf16
// operands (accumulated and multiplied in fp32) of any alignment.
//
// A 64-wide k-slab is a part of a block (b = 128), one block (64) or several
// (32, 16), so the walk over a block row's stored blocks is one stream of
// slabs: no block starts or drains a pipeline of its own. Output tiles are
// min(b, 64) rows x YN columns, and for dA 64x64 parts of a block (b >= 64)
// or the diagonal squares of a tile of several blocks (b = 32, 16). Bound by
// the MFMAs where the tiles fill the chip (8192^2, 10 % blocks of 64, N = 512:
// forward 76 us = 90 TFLOP/s, dA 76, dB 81; a wavefront per 64 columns or per
// block with operands straight from memory, the form before this one, took
// 132, 92 and 177), by the longest list of slabs, about 1.5 us each, where they
// do not (1024^2, 19 blocks of 128, N = 256: 12 us, from 28 on 128x128 tiles),
// and by the start and end of a workgroup, 4 us together, where lists are one
// slab (256 rows of one block of 32, N = 512: 18 us, a wavefront per tile 11).
#include "f32_flex.h"
#include "tile_item.h"

namespace {

namespace X = tsp::flex;

// A list walked in order, 64 entries at a time in the lanes of a wavefront;
// AHEAD: the next 64 loaded ahead. (Not for dB at b >= 64, whose registers are
// short: two spilled there, 94 against 86 us on 8192^2, 10 % blocks of 128, N =
// 512, and 64 entries last 64 slabs or more, where a wait for the next is
// little.)
template <bool AHEAD>
struct Walk {
  const int64_t* p;
  int n, base;
  int cur, next;
  __device__ Walk(const int64_t* p_, int n_) : p(p_), n(n_), base(0), cur(fetch(0)), next(AHEAD ? fetch(64) : 0) {}
  __device__ int fetch(int at) const {
    const int i = at + ((int)threadIdx.x & 63);
    return i < n ? (int)p[i] : 0;
  }
  // brings in entry q and the PER - 1 after it (q a multiple of PER and
  // ascending from call to call; PER divides 64)
  __device__ void to(int q) {
    if (q - base >= 64) {
      base += 64;
      cur = AHEAD ? next : fetch(base);
      if (AHEAD) next = fetch(base + 64);
    }
  }
  // entry q + e; e may differ between lanes. Selected from scalars: as an array
  // the PER of them lived in scratch memory, which costs a launch some 13 us
  // (b = 16, 512 rows of 3 blocks, N = 8: 18.4 -> 4.7 us, its dB 19.6 -> 5.6; a
  // wavefront per 64 columns took 6.2).
  template <int PER>
  __device__ int get(int q, int e) const {
    int x = __builtin_amdgcn_readlane(cur, q - base);
#pragma unroll
    for (int i = 1; i < PER; ++i) {
      const int v = __builtin_amdgcn_readlane(cur, q - base + i);
      x = e == i ? v : x;
    }
    return x;
  }
};

constexpr int part(int b) { return b < 64 ? b : 64; }  // rows of an output tile
// Columns of an output tile: 128 were slower for 32-row tiles (107 against 95 us
// where the chip is full) and for 16-row ones where it is not (8192^2, 10 %
// blocks, N = 509: 136 against 124; 2992^2, 20 %, N = 80: 22 against 16).
constexpr int YN = 64;

// The slab stream of one list of stored blocks. TA: the blocks enter
// transposed (dB); ids[q] is then entry q's block, else its block is p0 + q.
// dense rows of entry q start at cols[q] * b.
template <typename T, int B_, bool TA>
struct Stream {
  static constexpr int B = B_, MS = B < 32 ? 16 : 32, XN = part(B), PER = B < 64 ? 64 / B : 1;
  typedef X::Split<MS, XN, YN> Split;
  typedef X::Row<T, XN> XRow;
  typedef X::Col<T, XN, MS> XCol;
  typedef std::conditional_t<TA, XCol, XRow> XF;
  typedef X::Col<T, YN, MS> YF;
  const T *blocks, *dense;
  int64_t ldd, rows, ncols, n0, p0;
  int nblk, off;  // off: first row (TA: column) of the block in this tile
  Walk<(B < 64 || !TA)> cols, ids;
  struct Regs {
    XF x;
    YF y;
  };
  __device__ int slabs() const { return (int)(((int64_t)nblk * B + X::KC - 1) / X::KC); }
  __device__ void load(int s, Regs& r) {
    // the slab's blocks: entry q0 + e holds its k from e * B (B < 64), or the
    // slab is k kk .. of entry q0
    const int q0 = B < 64 ? s * PER : s / (B / 64), kk = B < 64 ? 0 : s % (B / 64) * 64;
    cols.to(q0);
    if constexpr (TA) ids.to(q0);
    auto block = [&](int e) -> const T* {
      if constexpr (TA)
        return blocks + (int64_t)ids.template get<PER>(q0, e) * (B * B);
      else
        return blocks + (p0 + q0 + e) * (B * B);
    };
#pragma unroll
    for (int j = 0; j < XF::PIECES; ++j) {
      const int i = XF::i() + (TA ? 0 : 32 * j), k = XF::k() + (TA ? XCol::KSTEP * j : 0);
      const int e = B < 64 ? k / B : 0, kb = B < 64 ? k % B : kk + k;
      const bool there = !XF::idle() && q0 + e < nblk;
      r.x.q[j].load(block(e) + (TA ? kb * B + off + i : (off + i) * B + kb), there ? 4 : 0);
    }
#pragma unroll
    for (int j = 0; j < YF::PIECES; ++j) {
      const int k = YF::k() + YF::KSTEP * j, e = B < 64 ? k / B : 0;
      const int64_t row = (int64_t)cols.template get<PER>(q0, e) * B + (B < 64 ? k % B : kk + k), c = n0 + YF::i();
      r.y.q[j].load(dense + row * ldd + c, !YF::idle() && q0 + e < nblk && row < rows ? ncols - c : 0);
    }
  }
  __device__ void finish(Regs&) {}
};

// out tile = sum over the entries [ptr[i], ptr[i + 1]) of list i of block
// (TA: transposed) times dense rows. C = A B: lists are block rows, `cols`
// the block columns; dB = A^T dC: lists are block columns, `cols` the block
// rows and `ids` the block numbers.
template <typename T, typename OutT, int B, bool TA>
__global__ __launch_bounds__(X::NTHR, 4) void bsr_flex(const T* __restrict__ blocks, const int64_t* __restrict__ ptr,
                                                       const int64_t* __restrict__ cols,
                                                       const int64_t* __restrict__ ids, int64_t lists, int nnt,
                                                       int64_t out_rows, int64_t dense_rows,
                                                       const T* __restrict__ dense, int64_t ldd, int64_t ncols,
                                                       OutT* __restrict__ out, int64_t ldo,
                                                       const int32_t* __restrict__ order) {
  typedef Stream<T, B, TA> S;
  __shared__ __attribute__((aligned(16))) float lds[X::lds_floats<typename S::XF, typename S::YF>()];
  constexpr int PARTS = B / S::XN;
  int64_t li;
  int item;
  if (!tsp::tile_item(blockIdx.x, lists, (int64_t)nnt * PARTS, order, li, item)) return;
  const int off = item % PARTS * S::XN;
  const int64_t n0 = (int64_t)(item / PARTS) * YN;
  const int64_t p0 = ptr[li];
  const int nblk = (int)(ptr[li + 1] - p0);
  S src{blocks, dense, ldd, dense_rows, ncols, n0, p0, nblk, off, {cols + p0, nblk}, {TA ? ids + p0 : cols, TA ? nblk : 0}};
  float acc[S::Split::NOUT];
  X::run<typename S::Split>(src, src.slabs(), lds, acc);
  const int64_t c = n0 + S::Split::col();
  if (c < ncols) {
#pragma unroll
    for (int v = 0; v < S::Split::NOUT; ++v) {
      const int64_t r = li * B + off + S::Split::row(v);
      if (r < out_rows) out[r * ldo + c] = tsp::from_acc<OutT>(acc[v]);
    }
  }
}

// dA: tile = 64x64 part of one block, or the diagonal of 64 / b blocks.
template <typename T, int B_>
struct Pairs {
  static constexpr int B = B_, MS = B < 32 ? 16 : 32, PER = B < 64 ? 64 / B : 1;
  typedef X::Split<MS, 64, 64, (B < 64)> Split;
  typedef X::Row<T, 64> XF;
  const T *G, *D;
  int64_t ldg, ldd, m, n, ncols;
  int64_t gr[2], dr[2];  // this thread's rows of dC and of B (-1: none)
  struct Regs {
    XF x, y;
  };
  __device__ void load(int s, Regs& r) {
    const int64_t k = (int64_t)s * X::KC + XF::k();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      r.x.q[j].load(G + gr[j] * ldg + k, gr[j] >= 0 ? ncols - k : 0);
      r.y.q[j].load(D + dr[j] * ldd + k, dr[j] >= 0 ? ncols - k : 0);
    }
  }
  __device__ void finish(Regs&) {}
};

template <typename T, int B>
__global__ __launch_bounds__(X::NTHR, 4) void bsr_flex_sddmm(const T* __restrict__ G, int64_t ldg, int64_t m,
                                                             const T* __restrict__ D, int64_t ldd, int64_t n,
                                                             int64_t ncols, const int64_t* __restrict__ brow,
                                                             const int64_t* __restrict__ bcol, int64_t nnzb,
                                                             T* __restrict__ out) {
  typedef Pairs<T, B> S;
  __shared__ __attribute__((aligned(16))) float lds[X::lds_floats<typename S::XF, typename S::XF>()];
  // XCD-aware: XCD x takes a contiguous range of blocks (shared dC rows)
  constexpr int PARTS = B < 64 ? 1 : (B / 64) * (B / 64);
  const int64_t items = tsp::ceil_div(nnzb, S::PER) * PARTS, per = tsp::ceil_div(items, 8);
  const int64_t slot = blockIdx.x >> 3, item = (blockIdx.x & 7) * per + slot;
  if (slot >= per || item >= items) return;
  const int64_t p0 = item / PARTS * S::PER;
  const int ro = B < 64 ? 0 : (int)(item % PARTS) / (B / 64) * 64, co = B < 64 ? 0 : (int)(item % PARTS) % (B / 64) * 64;
  S src{G, D, ldg, ldd, m, n, ncols, {}, {}};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = S::XF::i() + 32 * j;
    const int64_t p = p0 + (B < 64 ? i / B : 0);
    const int ib = B < 64 ? i % B : i;
    const int64_t r = p < nnzb ? brow[p] * B + ro + ib : m, c = p < nnzb ? bcol[p] * B + co + ib : n;
    src.gr[j] = r < m ? r : -1;
    src.dr[j] = c < n ? c : -1;
  }
  float acc[S::Split::NOUT];
  X::run<typename S::Split>(src, (int)tsp::ceil_div(ncols, X::KC), lds, acc);
  const int64_t p = p0 + (B < 64 ? S::Split::x0() / B : 0);
  if (p >= nnzb) return;
  const int cb = co + (B < 64 ? S::Split::col() % B : S::Split::col());
#pragma unroll
  for (int v = 0; v < S::Split::NOUT; ++v) {
    const int rb = ro + (B < 64 ? S::Split::row(v) % B : S::Split::row(v));
    out[p * (B * B) + rb * B + cb] = tsp::from_acc<T>(acc[v]);
  }
}

template <typename T, typename OutT, int B, bool TA>
int launch_product(const void* blocks, const int64_t* ptr, const int64_t* cols, const int64_t* ids, int64_t lists,
                   int64_t out_rows, int64_t dense_rows, const void* dense, int64_t ldd, int64_t ncols, void* out,
                   int64_t ldo, const int32_t* order, hipStream_t st) {
  const int64_t nnt = tsp::ceil_div(ncols, YN), parts = B / part(B);
  const int64_t grid = tsp::ceil_div(lists, 8) * 8 * nnt * parts;
  if (grid > INT32_MAX) return tsp::fail(TSP_EUNSUPPORTED, "bsr_flex: problem too large");
  hipLaunchKernelGGL((bsr_flex<T, OutT, B, TA>), dim3((unsigned)grid), dim3(X::NTHR), 0, st, (const T*)blocks, ptr,
                     cols, ids, lists, (int)nnt, out_rows, dense_rows, (const T*)dense, ldd, ncols, (OutT*)out, ldo,
                     order);
  return tsp::check_launch("bsr_flex launch");
}

template <typename T, typename OutT, bool TA, typename... Args>
int by_size(int64_t b, Args... a) {
  if (b == 16) return launch_product<T, OutT, 16, TA>(a...);
  if (b == 32) return launch_product<T, OutT, 32, TA>(a...);
  if (b == 64) return launch_product<T, OutT, 64, TA>(a...);
  return launch_product<T, OutT, 128, TA>(a...);
}

template <typename T, int B>
int launch_sddmm(const void* G, int64_t ldg, int64_t m, const void* D, int64_t ldd, int64_t n, int64_t ncols,
                 const int64_t* brow, const int64_t* bcol, int64_t nnzb, void* out, hipStream_t st) {
  const int64_t items = B < 64 ? tsp::ceil_div(nnzb, 64 / B) : nnzb * (B / 64) * (B / 64);
  const int64_t grid = tsp::ceil_div(items, 8) * 8;
  if (grid > INT32_MAX) return tsp::fail(TSP_EUNSUPPORTED, "bsr_flex_sddmm: too many blocks");
  hipLaunchKernelGGL((bsr_flex_sddmm<T, B>), dim3((unsigned)grid), dim3(X::NTHR), 0, st, (const T*)G, ldg, m,
                     (const T*)D, ldd, n, ncols, brow, bcol, nnzb, (T*)out);
  return tsp::check_launch("bsr_flex_sddmm launch");
}

}  // namespace

int tsp::launch_bsr_flex(int dtype, int out_dtype, int64_t b, const void* blocks, const int64_t* rp, const int64_t* ci,
                         int64_t mb, int64_t m, int64_t n, const void* B, int64_t ldb, int64_t ncols, void* C,
                         int64_t ldc, const int32_t* order, hipStream_t st) {
  const int64_t* none = nullptr;
  if (dtype == TSP_F32)
    return by_size<float, float, false>(b, blocks, rp, ci, none, mb, m, n, B, ldb, ncols, C, ldc, order, st);
  if (out_dtype == TSP_F32)
    return by_size<uint16_t, float, false>(b, blocks, rp, ci, none, mb, m, n, B, ldb, ncols, C, ldc, order, st);
  return by_size<uint16_t, uint16_t, false>(b, blocks, rp, ci, none, mb, m, n, B, ldb, ncols, C, ldc, order, st);
}

int tsp::launch_bsr_flex_t(int dtype, int64_t b, const void* blocks, const int64_t* col_ptrs,
                           const int64_t* col_block_rows, const int64_t* col_block_ids, int64_t n_block_cols,
                           int64_t m, int64_t n, const void* G, int64_t ldg, int64_t ncols, void* out, int64_t ldo,
                           const int32_t* order, hipStream_t st) {
  if (dtype == TSP_F32)
    return by_size<float, float, true>(b, blocks, col_ptrs, col_block_rows, col_block_ids, n_block_cols, n, m, G, ldg,
                                       ncols, out, ldo, order, st);
  return by_size<uint16_t, uint16_t, true>(b, blocks, col_ptrs, col_block_rows, col_block_ids, n_block_cols, n, m, G,
                                           ldg, ncols, out, ldo, order, st);
}

int tsp::launch_bsr_flex_sddmm(int dtype, int64_t b, const void* G, int64_t ldg, int64_t m, const void* B, int64_t ldb,
                               int64_t n, int64_t ncols, const int64_t* brow, const int64_t* bcol, int64_t nnzb,
                               void* out, hipStream_t st) {
  auto go = [&](auto t) {
    typedef decltype(t) T;
    if (b == 16) return launch_sddmm<T, 16>(G, ldg, m, B, ldb, n, ncols, brow, bcol, nnzb, out, st);
    if (b == 32) return launch_sddmm<T, 32>(G, ldg, m, B, ldb, n, ncols, brow, bcol, nnzb, out, st);
    if (b == 64) return launch_sddmm<T, 64>(G, ldg, m, B, ldb, n, ncols, brow, bcol, nnzb, out, st);
    return launch_sddmm<T, 128>(G, ldg, m, B, ldb, n, ncols, brow, bcol, nnzb, out, st);
  };
  return dtype == TSP_F32 ? go(float{}) : go(uint16_t{});
}
