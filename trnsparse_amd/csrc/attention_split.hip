// Block-sparse attention on grids that leave compute units idle: the forward,
// the dQ pass and the dK / dV pass of attention.hip and attention_bwd.hip
// (semantics there; reference trnsparse/ops.py:280-473) with four times the
// workgroups. fp32 and bf16, 128-blocks, head_dim 64 and 128.
//
// The full-grid kernels give a workgroup 128 queries (or keys), 32 to a
// wavefront, and stream the other operand's rows through LDS for all four.
// Few heads on a short sequence then fill a fraction of the 256 CUs, each
// walking its row's blocks one after the other. Here a workgroup has 32
// queries (keys) and wavefront w takes rows 32 w .. 32 w + 31 of every block it
// walks, streamed through LDS of its own: no barrier until the end, where the
// four partial results are added through LDS in wavefront order (the forward
// weighs them by their maxima). Every byte of a block is still loaded by each
// workgroup, so the loads per MFMA are four times the full-grid kernels'; that
// is what a full chip would be bound by, and why those stay.
//
// fp32 tiles are single-buffered: each operand's next tile is loaded as soon as
// its last product is done, under the products of the other. bf16 products are
// too short for that: two buffers, the next tiles loaded first.
#include "attention_tiles.h"
#include "lds_dma.h"
#include "tile_item.h"

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.69314718055994531f;
constexpr int BS = 128;

// One 32-row tile and the products with it.
template <typename T, int D>
struct Tile;

template <int D>
struct Tile<float, D> {
  static constexpr int NBUF = 1, ROWB = D * 4, BYTES = 32 * ROWB, LOADS = BYTES / 1024, NU = D / 32, KT = D / 8;
  struct Own {
    f32x4 v[KT];
  };
  __device__ static void load_own(const float* row, int h, bool valid, Own& o) {
#pragma unroll
    for (int t = 0; t < KT; ++t) o.v[t] = valid ? *(const f32x4*)(row + 8 * t + 4 * h) : f32x4{};
  }
  __device__ static float dot(const Own& a, const Own& b) {
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c) s += a.v[t][c] * b.v[t][c];
    return s;
  }
  // rows row0 .. + 31 of rs into LDS dst (rows past the buffer read as zero)
  __device__ static void fetch(tsp::dma::i32x4 rs, int64_t row0, uint32_t dst, int lane) {
    constexpr int LPR = D / 4, RPI = 64 / LPR;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int rr = RPI * j + lane / LPR, p = lane % LPR;
      tsp::dma::buffer16(rs, (uint32_t)((row0 + rr) * ROWB + ((p ^ (rr & 15)) << 4)), dst + j * 1024);
    }
  }
  // element v: tile row 8 (v / 4) + 4 h + v % 4 times the lane's own row
  __device__ static f32x16 scores(const uint8_t* tile, const Own& own, int h, int l32) {
    f32x16 s = {};
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      const f32x4 a = tsp::abf::chunk_read<D>(tile, l32, 2 * t + h, l32 & 15);
#pragma unroll
      for (int c = 0; c < 4; ++c) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c], own.v[t][c], s, 0, 0, 0);
    }
    return s;
  }
  // acc += tile^T p (p as scores() lays it out)
  __device__ static void add(const uint8_t* tile, const f32x16& p, f32x16 (&acc)[NU], int h, int l32) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const auto r = tsp::abf::row_read<D>(tile, 8 * (i >> 2) + 4 * h + (i & 3), l32);
#pragma unroll
      for (int u = 0; u < NU; ++u) acc[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(r[u], p[i], acc[u], 0, 0, 0);
    }
  }
  // elements v = 4 a .. 4 a + 3 of every subtile: 4 NU consecutive values
  template <typename OutT>
  __device__ static void store(OutT* row, const float (&r)[NU][4], int a, int h) {
#pragma unroll
    for (int k = 0; k < NU; ++k) {
      f32x4 t;
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = r[(4 * k + e) % NU][(4 * k + e) / NU];
      *(f32x4*)(row + NU * (8 * a + 4 * h) + 4 * k) = t;
    }
  }
};

template <int D>
struct Tile<uint16_t, D> {
  typedef tsp::abw::Geo<D> G;
  static constexpr int NBUF = 2, ROWB = D * 2, BYTES = 32 * ROWB, LOADS = BYTES / 1024, NU = D / 32, KS = D / 16;
  struct Own {
    bf16x8 v[KS];
  };
  __device__ static void load_own(const uint16_t* row, int h, bool valid, Own& o) {
#pragma unroll
    for (int s = 0; s < KS; ++s) o.v[s] = valid ? *(const bf16x8*)(row + 16 * s + 8 * h) : bf16x8{};
  }
  __device__ static float dot(const Own& a, const Own& b) {
    float s = 0.f;
#pragma unroll
    for (int t = 0; t < KS; ++t)
#pragma unroll
      for (int c = 0; c < 8; ++c) s += (float)a.v[t][c] * (float)b.v[t][c];
    return s;
  }
  __device__ static void fetch(tsp::dma::i32x4 rs, int64_t row0, uint32_t dst, int lane) {
    constexpr int CPR = ROWB / 16, RPI = 64 / CPR;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      const int rr = RPI * j + lane / CPR, p = lane % CPR;
      tsp::dma::buffer16(rs, (uint32_t)((row0 + rr) * ROWB + ((p ^ tsp::abw::swz<D>(rr)) << 4)), dst + j * 1024);
    }
  }
  __device__ static f32x16 scores(const uint8_t* tile, const Own& own, int h, int l32) {
    const uint32_t rb = tsp::dma::lds_addr(tile) + (uint32_t)(l32 * ROWB + ((tsp::abw::swz<D>(l32) ^ h) << 4));
    f32x16 s = {};
#pragma unroll
    for (int k = 0; k < KS; ++k)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tsp::abw::lds_row(rb, k, 0), own.v[k], s, 0, 0, 0);
    return s;
  }
  __device__ static void add(const uint8_t* tile, const f32x16& p, f32x16 (&acc)[NU], int h, int l32) {
    const tsp::abw::TrLane t = tsp::abw::tr_lane<D>(32 * h + l32);
    const uint32_t base = tsp::dma::lds_addr(tile) + (uint32_t)(t.xu << 6);
    const uint32_t tb0 = base + t.off[0], tb1 = base + t.off[1];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      tsp::abw::f32x8 x;
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = p[8 * a + i];
      const bf16x8 pb = __builtin_convertvector(x, bf16x8);
#pragma unroll
      for (int u = 0; u < NU; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tsp::abw::lds_trp(tb0, tb1, u, 16 * a * ROWB), pb, acc[u], 0,
                                                         0, 0);
    }
  }
  __device__ static void store(uint16_t* row, const float (&r)[NU][4], int a, int h) {
#pragma unroll
    for (int u = 0; u < NU; ++u)
      *(tsp::abw::u16x4*)(row + 32 * u + 8 * a + 4 * h) = tsp::abw::bf16x4_rne(f32x4{r[u][0], r[u][1], r[u][2], r[u][3]});
  }
  __device__ static void store(float* row, const float (&r)[NU][4], int a, int h) {
#pragma unroll
    for (int u = 0; u < NU; ++u) *(f32x4*)(row + 32 * u + 8 * a + 4 * h) = f32x4{r[u][0], r[u][1], r[u][2], r[u][3]};
  }
};

// Block indices of a row (or column), 64 at a time in one VGPR.
struct List {
  const int64_t* p;
  int n, base, v;
  __device__ List(const int64_t* p_, int n_, int lane) : p(p_), n(n_), base(0), v(0) {
    if (n > 0) v = load(0, lane);
  }
  __device__ int load(int at, int lane) const {
    const int i = at + lane < n ? at + lane : n - 1;
    return tsp::dma::load_lo32_sync(p + i);
  }
  __device__ int get(int i, int lane) {
    if (i - base >= 64) {
      base = i & ~63;
      v = load(base, lane);
    }
    return __builtin_amdgcn_readlane(v, i - base);
  }
};

__device__ inline void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Streams two operands' tiles (rows 32 w .. of block get(i)) through this
// wavefront's LDS. FIRST is the operand whose tile is needed first and freed
// first. `extra` loads ride with it.
//   fp32: first(i) ... free_first(i) ... second(i) ... free_second(i)
//   bf16: first(i) issues both operands of i + 1 and waits for those of i.
// Both return the tile's LDS address.
template <typename T, int D, int EXTRA, class Issue>
struct Stream {
  typedef Tile<T, D> TL;
  static constexpr int A = TL::BYTES + (EXTRA ? 1024 : 0), BUF = A + TL::BYTES;
  static constexpr int WAVE = TL::NBUF * BUF;  // LDS of a wavefront
  Issue issue;  // issue(i, which, dst): which = 0 first (+ extra), 1 second
  uint32_t lds;
  int n;
  __device__ void start() {
    if (n > 0) {
      issue(0, 0, lds);
      issue(0, 1, lds + A);
    }
  }
  __device__ uint32_t first(int i) {
    if constexpr (TL::NBUF == 2) {
      if (i + 1 < n) {
        lds_reads_done();  // of tile i - 1, in the buffer that i + 1 takes
        const uint32_t b = lds + ((i + 1) & 1) * BUF;
        issue(i + 1, 0, b);
        issue(i + 1, 1, b + A);
        tsp::dma::wait_vm<2 * TL::LOADS + EXTRA>();
      } else {
        tsp::dma::wait_vm<0>();
      }
      return lds + (i & 1) * BUF;
    } else {
      tsp::dma::wait_vm<TL::LOADS>();  // all but the second operand's tile i
      return lds;
    }
  }
  __device__ void free_first(int i) {
    if (TL::NBUF == 1 && i + 1 < n) {
      lds_reads_done();
      issue(i + 1, 0, lds);
    }
  }
  // early: free_first(i) has been called
  template <bool EARLY>
  __device__ uint32_t second(int i) {
    if constexpr (TL::NBUF == 2) {
      return lds + (i & 1) * BUF + A;
    } else {
      if (EARLY && i + 1 < n)
        tsp::dma::wait_vm<TL::LOADS + EXTRA>();
      else
        tsp::dma::wait_vm<0>();
      return lds + A;
    }
  }
  __device__ void free_second(int i) {
    if (TL::NBUF == 1 && i + 1 < n) {
      lds_reads_done();
      issue(i + 1, 1, lds + A);
    }
  }
};
template <typename T, int D, int EXTRA, class Issue>
__device__ inline Stream<T, D, EXTRA, Issue> make_stream(Issue issue, uint32_t lds, int n) {
  return Stream<T, D, EXTRA, Issue>{issue, lds, n};
}

__device__ inline const uint8_t* lds_ptr(uint32_t a) {
  return (const uint8_t*)(__attribute__((address_space(3))) const uint8_t*)(uintptr_t)a;
}

// r[u][c] = sum over the wavefronts of acc[u][4 w + c] of wavefront w's lanes.
template <int NU>
__device__ inline void sum_waves(float* red, const f32x16 (&acc)[NU], float f, float (&r)[NU][4], int w, int lane) {
  constexpr int PER = NU * 16 * 64;
  tsp::dma::barrier();
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int v = 0; v < 16; ++v) red[w * PER + (u * 16 + v) * 64 + lane] = acc[u][v] * f;
  tsp::dma::barrier();
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float s = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) s += red[k * PER + (u * 16 + 4 * w + c) * 64 + lane];
      r[u][c] = s;
    }
}

// Head, block row and 32-row part of a workgroup.
__device__ inline bool item_of(int64_t Mt, int64_t H, int64_t& head, int64_t& m, int& sub) {
  int64_t i;
  if (!tsp::head_item(blockIdx.x, 4 * Mt, H, head, i)) return false;
  m = i >> 2;
  sub = (int)(i & 3);
  return true;
}

template <typename T, int D>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bsa_fwd_split(const T* __restrict__ Q, const T* __restrict__ K,
                                                     const T* __restrict__ V, int64_t S, int64_t H,
                                                     const int64_t* __restrict__ rp, const int64_t* __restrict__ ci,
                                                     int64_t Mt, float scale_log2, T* __restrict__ O,
                                                     float* __restrict__ rmax, float* __restrict__ rden) {
  typedef Tile<T, D> TL;
  constexpr int NU = TL::NU, WAVE = TL::NBUF * 2 * TL::BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * WAVE];
  __shared__ float stat[4][3][32];
  int64_t head, m;
  int sub;
  if (!item_of(Mt, H, head, m, sub)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int64_t hs = head * S * D, q = m * BS + 32 * sub + l32;  // < S since m < Mt
  typename TL::Own qf;
  TL::load_own(Q + hs + q * D, h, true, qf);
  f32x16 o[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) o[u] = f32x16{};
  constexpr float RESCALE = 8.f;  // lazy rescaling as in the full-grid kernels
  float mtrue = -INFINITY, mref = -INFINITY, lrun = 0.f;

  const int64_t start = rp[m];
  const int nblk = (int)(rp[m + 1] - start);
  const tsp::dma::i32x4 krs = tsp::dma::make_rsrc(K + hs, (uint32_t)(S * TL::ROWB));
  const tsp::dma::i32x4 vrs = tsp::dma::make_rsrc(V + hs, (uint32_t)(S * TL::ROWB));
  List ahead(ci + start, nblk, lane), here(ci + start, nblk, lane);
  auto key_of = [&](List& l, int i) { return (int64_t)l.get(i, lane) * BS + 32 * w; };
  auto st = make_stream<T, D, 0>(
      [&](int i, int which, uint32_t dst) { TL::fetch(which ? vrs : krs, key_of(ahead, i), dst, lane); },
      tsp::dma::lds_addr(lds) + w * WAVE, nblk);
  st.start();
  for (int i = 0; i < nblk; ++i) {
    const int64_t key0 = key_of(here, i);
    f32x16 sc = TL::scores(lds_ptr(st.first(i)), qf, h, l32);
    st.free_first(i);
    if (key0 + 32 > S) {
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (key0 + 8 * (v >> 2) + 4 * h + (v & 3) >= S) sc[v] = -INFINITY;
    }
    float mraw = sc[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) mraw = fmaxf(mraw, sc[v]);
    mraw = fmaxf(mraw, __shfl_xor(mraw, 32, 64));
    mtrue = fmaxf(mtrue, mraw * scale_log2);
    if (__builtin_amdgcn_ballot_w64(mtrue > mref + RESCALE) != 0) {
      const bool move = mtrue > mref + RESCALE;
      const float alpha = move ? (mref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mref - mtrue)) : 1.f;
      mref = move ? mtrue : mref;
      lrun *= alpha;
#pragma unroll
      for (int u = 0; u < NU; ++u) o[u] *= alpha;
    }
    const float nmx = mref == -INFINITY ? 0.f : -mref;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      sc[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[v], scale_log2, nmx));
      lrun += sc[v];  // this lane half's part
    }
    TL::add(lds_ptr(st.template second<true>(i)), sc, o, h, l32);
    st.free_second(i);
  }
  lrun += __shfl_xor(lrun, 32, 64);
  // the wavefronts' results, relative to the row's maximum
  if (h == 0) {
    stat[w][0][l32] = mtrue;
    stat[w][1][l32] = mref;
    stat[w][2][l32] = lrun;
  }
  tsp::dma::barrier();
  float M = -INFINITY, l = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) M = fmaxf(M, stat[k][0][l32]);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float r = stat[k][1][l32];
    l += stat[k][2][l32] * (r == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(r - M));
  }
  const bool empty = nblk == 0;
  const float den = l > 1e-12f ? l : 1e-12f;
  float r[NU][4];
  sum_waves<NU>((float*)lds, o, (mref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mref - M)) * (empty ? 0.f : 1.f / den),
                r, w, lane);
  TL::store(O + hs + q * D, r, w, h);
  if (rmax && w == 0 && h == 0) {
    rmax[head * Mt * BS + q] = empty ? 0.f : M * LN2;
    rden[head * Mt * BS + q] = empty ? 1e-12f : den;
  }
}

// dQ, and the query statistics for the dK / dV pass: plane 0 r = log2e *
// row_max + log2 row_denom, plane 1 D = rowsum(dO * O).
template <typename T, int D>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bsa_bwd_dq_split(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, const T* __restrict__ O,
    const T* __restrict__ dO, int64_t S, int64_t H, const int64_t* __restrict__ rp, const int64_t* __restrict__ ci,
    int64_t Mt, float scale_log2, float scale, const float* __restrict__ rmax, const float* __restrict__ rden,
    float* __restrict__ qstat, T* __restrict__ dQ) {
  typedef Tile<T, D> TL;
  constexpr int NU = TL::NU, WAVE = TL::NBUF * 2 * TL::BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * WAVE];
  int64_t head, m;
  int sub;
  if (!item_of(Mt, H, head, m, sub)) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int64_t hs = head * S * D, q = m * BS + 32 * sub + l32;
  typename TL::Own qf, dof;
  TL::load_own(Q + hs + q * D, h, true, qf);
  TL::load_own(dO + hs + q * D, h, true, dof);
  float Dq;
  {
    typename TL::Own of;
    TL::load_own(O + hs + q * D, h, true, of);
    Dq = TL::dot(dof, of);
  }
  Dq += __shfl_xor(Dq, 32, 64);
  const float rq = rmax[head * Mt * BS + q] * LOG2E + __builtin_amdgcn_logf(rden[head * Mt * BS + q]);
  if (w == 0 && h == 0) {
    qstat[head * S + q] = rq;
    qstat[H * S + head * S + q] = Dq;
  }
  f32x16 acc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) acc[u] = f32x16{};

  const int64_t start = rp[m];
  const int nblk = (int)(rp[m + 1] - start);
  const tsp::dma::i32x4 krs = tsp::dma::make_rsrc(K + hs, (uint32_t)(S * TL::ROWB));
  const tsp::dma::i32x4 vrs = tsp::dma::make_rsrc(V + hs, (uint32_t)(S * TL::ROWB));
  List ahead(ci + start, nblk, lane), here(ci + start, nblk, lane);
  auto key_of = [&](List& l, int i) { return (int64_t)l.get(i, lane) * BS + 32 * w; };
  auto st = make_stream<T, D, 0>(
      [&](int i, int which, uint32_t dst) { TL::fetch(which ? krs : vrs, key_of(ahead, i), dst, lane); },
      tsp::dma::lds_addr(lds) + w * WAVE, nblk);
  st.start();
  for (int i = 0; i < nblk; ++i) {
    const int64_t key0 = key_of(here, i);
    f32x16 dp = TL::scores(lds_ptr(st.first(i)), dof, h, l32);
    st.free_first(i);
    const uint8_t* kt = lds_ptr(st.template second<true>(i));
    const f32x16 sc = TL::scores(kt, qf, h, l32);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float p = key0 + 8 * (v >> 2) + 4 * h + (v & 3) >= S
                          ? 0.f
                          : __builtin_amdgcn_exp2f(__builtin_fmaf(sc[v], scale_log2, -rq));
      dp[v] = p * (dp[v] - Dq);
    }
    TL::add(kt, dp, acc, h, l32);
    st.free_second(i);
  }
  float r[NU][4];
  sum_waves<NU>((float*)lds, acc, scale, r, w, lane);
  TL::store(dQ + hs + q * D, r, w, h);
}

// dK and dV of 32 keys of a plan item's block column over its block rows;
// a segment of a split column writes fp32 partials for the reduce.
template <typename T, int D>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bsa_bwd_dkdv_split(
    const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V, const T* __restrict__ dO, int64_t S,
    int64_t H, const int64_t* __restrict__ crow, const int32_t* __restrict__ items, int n_items, int n_partials, int64_t Mt,
    float scale_log2, float scale, const float* __restrict__ qstat, T* __restrict__ dK, T* __restrict__ dV,
    float* __restrict__ partial) {
  typedef Tile<T, D> TL;
  constexpr int NU = TL::NU, WAVE = TL::NBUF * (2 * TL::BYTES + 1024);
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * WAVE];
  // (item, head, part), heaviest items first; the parts of one share an XCD
  const int64_t pair = (blockIdx.x >> 5) * 8 + (blockIdx.x & 7), it = pair / H, head = pair % H;
  const int sub = blockIdx.x >> 3 & 3;
  if (it >= n_items) return;
  const int col = items[4 * it], p0 = items[4 * it + 1], pslot = items[4 * it + 3];
  const int nblk = items[4 * it + 2] - p0;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h = lane >> 5, l32 = lane & 31;
  const int64_t hs = head * S * D, HS = H * S, key = (int64_t)col * BS + 32 * sub + l32;
  typename TL::Own kf, vf;
  TL::load_own(K + hs + key * D, h, key < S, kf);
  TL::load_own(V + hs + key * D, h, key < S, vf);
  f32x16 dk[NU], dv[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) dk[u] = dv[u] = f32x16{};
  const tsp::dma::i32x4 qrs = tsp::dma::make_rsrc(Q + hs, (uint32_t)(S * TL::ROWB));
  const tsp::dma::i32x4 ors = tsp::dma::make_rsrc(dO + hs, (uint32_t)(S * TL::ROWB));
  List ahead(crow + p0, nblk, lane), here(crow + p0, nblk, lane);
  auto st = make_stream<T, D, 1>(
      [&](int i, int which, uint32_t dst) {
        // rows past the whole blocks have no queries and no statistics: their
        // tiles are read past the buffers' ends, as zeros, and any 16 bytes of
        // this head stand in for the statistics
        const int64_t row = ahead.get(i, lane), q0 = row < Mt ? row * BS + 32 * w : S;
        TL::fetch(which ? qrs : ors, q0, dst, lane);
        // with dO: lanes 0-7 r, the rest D (from lane 16 on repeated)
        if (which == 0) {
          const float* stat = qstat + (lane & 8 ? HS : 0) + head * S + q0 + 4 * (lane & 7);
          tsp::dma::global16(row < Mt ? (const void*)stat : (const void*)(Q + hs), dst + TL::BYTES);
        }
      },
      tsp::dma::lds_addr(lds) + w * WAVE, nblk);
  st.start();
  for (int i = 0; i < nblk; ++i) {
    const bool there = here.get(i, lane) < Mt;
    const uint8_t* ot = lds_ptr(st.first(i));
    f32x16 dp = TL::scores(ot, vf, h, l32);
    const uint8_t* qt = lds_ptr(st.template second<false>(i));
    f32x16 sc = TL::scores(qt, kf, h, l32);
    const float* stats = (const float*)(ot + TL::BYTES);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const f32x4 r4 = *(const f32x4*)(stats + 8 * a + 4 * h);
      const f32x4 d4 = *(const f32x4*)(stats + 32 + 8 * a + 4 * h);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int v = 4 * a + c;
        const float p = there ? __builtin_amdgcn_exp2f(__builtin_fmaf(sc[v], scale_log2, -r4[c])) : 0.f;
        sc[v] = p;
        dp[v] = there ? p * (dp[v] - d4[c]) : 0.f;
      }
    }
    TL::add(ot, sc, dv, h, l32);
    st.free_first(i);
    TL::add(qt, dp, dk, h, l32);
    st.free_second(i);
  }
  float rk[NU][4], rv[NU][4];
  sum_waves<NU>((float*)lds, dk, scale, rk, w, lane);
  sum_waves<NU>((float*)lds, dv, 1.f, rv, w, lane);
  if (pslot < 0) {
    if (key < S) {
      TL::store(dK + hs + key * D, rk, w, h);
      TL::store(dV + hs + key * D, rv, w, h);
    }
  } else {
    float* pk = partial + (((int64_t)head * n_partials + pslot) * 2) * (BS * D) + (32 * sub + l32) * D;
    TL::store(pk, rk, w, h);
    TL::store(pk + BS * D, rv, w, h);
  }
}

template <typename T, int D>
int fwd(const void* Q, const void* K, const void* V, int64_t H, int64_t S, const int64_t* rp, const int64_t* ci,
        int64_t Mt, double scale, void* O, void* rmax, void* rden, hipStream_t st) {
  hipLaunchKernelGGL((bsa_fwd_split<T, D>), dim3((unsigned)tsp::head_grid(4 * Mt, H)), dim3(256), 0, st,
                     (const T*)Q, (const T*)K, (const T*)V, S, H, rp, ci, Mt, (float)(scale * 1.4426950408889634), (T*)O,
                     (float*)rmax, (float*)rden);
  return tsp::check_launch("bsa_fwd_split launch");
}

template <typename T, int D>
int dq(const void* Q, const void* K, const void* V, const void* O, const void* dO, int64_t H, int64_t S,
       const int64_t* rp, const int64_t* ci, int64_t Mt, double scale, const void* rmax, const void* rden, float* qstat,
       void* dQ, hipStream_t st) {
  hipLaunchKernelGGL((bsa_bwd_dq_split<T, D>), dim3((unsigned)tsp::head_grid(4 * Mt, H)), dim3(256), 0, st, (const T*)Q,
                     (const T*)K, (const T*)V, (const T*)O, (const T*)dO, S, H, rp, ci, Mt,
                     (float)(scale * 1.4426950408889634), (float)scale, (const float*)rmax, (const float*)rden, qstat,
                     (T*)dQ);
  return tsp::check_launch("bsa_bwd_dq_split launch");
}

template <typename T, int D>
int dkdv(const void* Q, const void* K, const void* V, const void* dO, int64_t H, int64_t S, const int64_t* crow,
         int64_t Mt, double scale, const int32_t* items, int64_t n_items, int64_t n_partials, const float* qstat,
         void* dK, void* dV, float* partial, hipStream_t st) {
  hipLaunchKernelGGL((bsa_bwd_dkdv_split<T, D>), dim3((unsigned)(tsp::ceil_div(n_items * H, 8) * 32)), dim3(256), 0, st,
                     (const T*)Q, (const T*)K, (const T*)V, (const T*)dO, S, H, crow, items, (int)n_items,
                     (int)n_partials, Mt, (float)(scale * 1.4426950408889634), (float)scale, qstat, (T*)dK, (T*)dV,
                     partial);
  return tsp::check_launch("bsa_bwd_dkdv_split launch");
}

}  // namespace

// Workgroups that share a CU (registers and LDS of head_dim 64 allow two), and
// the times of a round of them against a round of the full-grid kernel's
// workgroups, one per CU, measured in fp32 (heads of 4096, window 4, 2 global
// blocks: us at 64 / 128):
//   forward     31 of 52    35 of 108
//   dQ          43 of 85    50 of 162
//   dK / dV     always      42 of 138
// At head_dim 64 in fp32 two workgroups share a CU where the full-grid dK / dV
// kernel's registers allowed one: 184 work items 61 of 74 us, 276 95 of 142,
// 368 112 of 140, 1104 311 of 345, 32 heads of 8192 894 of 918, and 78 of 76
// only just below one full round (230), so that kernel is gone.
// Rows of one block pay for the merge at the end and no more: 12 heads of 2048 at
// 128 (192 block rows, 3 rounds of 1) take 37 us forward where the full-grid
// kernel takes 31, dQ 54 of 45, dK / dV 60 of 50, and dK / dV at 64 257 of 221 on
// 32 heads of 8192. The lengths are not known here, and other masks gain: the
// same 12 heads forward, window 4 110 of 115 us, causal 203 of 278, one global
// block row and column 137 of 277.
// bf16 products are too short to pay for the fourfold loads once a second
// round starts: 72 block rows at 128 (288 workgroups) 20.4 against 18.6 us, 64
// (256) 20.6 against 28.3; at 64, 128 block rows (512 workgroups, two to a CU)
// 12.7 against 14.6, 160 19.8 against 14.2. One head of 8192 at 64 in fp32:
// forward 54 -> 21 us, dK / dV 74 -> 42.
static bool split_pays(int dtype, int64_t D, int64_t items, int64_t num64, int64_t den64, int64_t num128,
                       int64_t den128) {
  const int64_t per_cu = D == 64 ? 2 : 1, rounds = tsp::ceil_div(4 * items, 256 * per_cu);
  if (dtype != TSP_F32) return rounds <= 1;
  if (items > 512) return false;  // the full-grid kernels' rounds no longer end together
  const int64_t full = tsp::ceil_div(items, 256);
  return D == 64 ? rounds * num64 < full * den64 : rounds * num128 < full * den128;
}
bool tsp::attn_split_fwd_pays(int dtype, int64_t D, int64_t H, int64_t Mt) {
  return (D == 64 || D == 128) && split_pays(dtype, D, H * Mt, 31, 52, 35, 108);
}
bool tsp::attn_split_dq_pays(int dtype, int64_t D, int64_t H, int64_t Mt) {
  return (D == 64 || D == 128) && split_pays(dtype, D, H * Mt, 43, 85, 50, 162);
}
bool tsp::attn_split_dkdv_pays(int dtype, int64_t D, int64_t H, int64_t n_items) {
  const int64_t items = H * n_items;
  if (D != 64 && D != 128) return false;
  if (dtype == TSP_F32 && D == 64) return true;
  return split_pays(dtype, D, items, 1, 1, 42, 138);
}

int tsp::launch_attn_split_fwd(int dtype, int64_t D, const void* Q, const void* K, const void* V, int64_t H, int64_t S,
                               const int64_t* rp, const int64_t* ci, int64_t Mt, double scale, void* O, void* rmax,
                               void* rden, hipStream_t st) {
  auto go = [&](auto f) { return f(Q, K, V, H, S, rp, ci, Mt, scale, O, rmax, rden, st); };
  if (dtype == TSP_F32) return D == 64 ? go(fwd<float, 64>) : go(fwd<float, 128>);
  return D == 64 ? go(fwd<uint16_t, 64>) : go(fwd<uint16_t, 128>);
}

int tsp::launch_attn_split_dq(int dtype, int64_t D, const void* Q, const void* K, const void* V, const void* O,
                              const void* dO, int64_t H, int64_t S, const int64_t* rp, const int64_t* ci, int64_t Mt,
                              double scale, const void* rmax, const void* rden, float* qstat, void* dQ,
                              hipStream_t st) {
  auto go = [&](auto f) { return f(Q, K, V, O, dO, H, S, rp, ci, Mt, scale, rmax, rden, qstat, dQ, st); };
  if (dtype == TSP_F32) return D == 64 ? go(dq<float, 64>) : go(dq<float, 128>);
  return D == 64 ? go(dq<uint16_t, 64>) : go(dq<uint16_t, 128>);
}

int tsp::launch_attn_split_dkdv(int dtype, int64_t D, const void* Q, const void* K, const void* V, const void* dO,
                                int64_t H, int64_t S, const int64_t* crow, int64_t Mt, double scale,
                                const int32_t* items, int64_t n_items, int64_t n_partials, const float* qstat,
                                void* dK, void* dV, float* partial, hipStream_t st) {
  auto go = [&](auto f) {
    return f(Q, K, V, dO, H, S, crow, Mt, scale, items, n_items, n_partials, qstat, dK, dV, partial, st);
  };
  if (dtype == TSP_F32) return D == 64 ? go(dkdv<float, 64>) : go(dkdv<float, 128>);
  return D == 64 ? go(dkdv<uint16_t, 64>) : go(dkdv<uint16_t, 128>);
}
