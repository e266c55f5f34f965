// Device-wide prefix sums and a stable LSD radix sort of (key, value) pairs,
// hand-written for gfx950 (wave64). Used by the format constructors (COO ->
// CSR, the CSR transpose, duplicate summation) and the SpMV column-plan
// build.
//
// Scan: blocks of 256 threads x 16 consecutive elements; a three-phase
// reduce / scan-of-block-sums / apply, the block sums scanned recursively.
//
// Sort: digits of 8 or 9 bits over bits [begin_bit, end_bit): 9 where that
// takes a pass less, the key bits spread evenly over the passes. Tiles of 4096
// keys: 256 threads x 16 keys or 512 x 8, a thread per digit (in the scatter,
// round i of lane l in wavefront w is key (4096 / wavefronts) w + 64 i + l).
// Per pass, three launches:
//   rs_count    per-tile digit counts into a tile-major table
//               counts[tile][d] (one coalesced row per tile);
//   rs_offsets  the table turned in place into the counts of the tiles
//               before, and each digit's total: a workgroup per 8 digits, 128
//               threads walking the tiles of each (past 1024 tiles, the chunks
//               of tiles, between two more launches);
//   rs_scatter  the digit bases from the totals, and each key's rank among
//               equal digits of its tile: each wavefront owns a contiguous
//               part of the tile and keeps a running count per digit in LDS
//               across its rounds; lanes of a round with the same digit are
//               found by a ballot per bit; the tile is reordered by digit in
//               LDS and written as runs, so consecutive lanes write
//               consecutive addresses.
// Equal digits keep their input order within and across tiles, so every
// pass and the sort are stable. Passes alternate between the output and a
// temporary buffer so the last one lands in the output.
// A pass reads and writes every pair, so the passes bound it and, up to some
// millions of keys, the launches. 2.4 M (column, row and value) pairs on 18 bits:
// two passes of 36 us; with three of 8 bits and five launches each, 118 us in
// all. CSR transposes of 2^18 columns, before -> now: 1 M entries 106 -> 72 us,
// 16 M 590 -> 489, 128 M 5000 -> 3945; COO -> CSR of 1 M 138 -> 117.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace tsp {
namespace rsort {

constexpr int NT = 256;             // threads per block
constexpr int NW = NT / 64;         // wavefronts per block
constexpr int SCAN_IPT = 16;        // scan elements per thread
constexpr int SCAN_TILE = NT * SCAN_IPT;
constexpr int SORT_TILE = 4096;     // sort keys per workgroup

inline size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// ------------------------------------------------------------------ scan

// Exclusive scan of one value per thread over the WAVES wavefronts of a block;
// `total` receives the block's sum. Every thread must call it.
template <typename T, int WAVES = NW>
__device__ inline T block_exclusive_scan(T v, T& total) {
  __shared__ T wsum[WAVES];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  T x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  T before = 0, all = 0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) {
    const T s = wsum[i];
    if (i < w) before += s;
    all += s;
  }
  __syncthreads();  // wsum may be reused by a later call
  total = all;
  return before + x - v;
}

template <typename T>
__global__ __launch_bounds__(NT) void scan_reduce_kernel(const T* __restrict__ in, int64_t n, T* __restrict__ sums) {
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_IPT;
  T s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_IPT; ++i)
    if (base + i < n) s += in[base + i];
  T total;
  block_exclusive_scan(s, total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// out[i] = init + offs[block] + (sum of in[block start .. i), or .. i] when inclusive).
// in == out is allowed: each thread reads its elements before writing them.
template <typename T>
__global__ __launch_bounds__(NT) void scan_apply_kernel(const T* in, T* out, int64_t n, const T* __restrict__ offs,
                                                        int inclusive, T init) {
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_IPT;
  T v[SCAN_IPT];
  T s = 0;
#pragma unroll
  for (int i = 0; i < SCAN_IPT; ++i) {
    v[i] = base + i < n ? in[base + i] : T(0);
    s += v[i];
  }
  T total;
  T run = block_exclusive_scan(s, total) + init + (offs ? offs[blockIdx.x] : T(0));
#pragma unroll
  for (int i = 0; i < SCAN_IPT; ++i) {
    if (base + i < n) out[base + i] = inclusive ? run + v[i] : run;
    run += v[i];
  }
}

// Temporary bytes for scan() over n elements: the block sums of every level.
inline size_t scan_tmp_bytes(int64_t n, size_t elem) {
  size_t b = 0;
  int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  while (nb > 1) {
    b += 2 * align256((size_t)nb * elem);
    nb = (nb + SCAN_TILE - 1) / SCAN_TILE;
  }
  return b + 256;
}

// Prefix sums of in[0, n) into out (in place allowed), plus init.
template <typename T>
hipError_t scan(void* tmp, const T* in, T* out, int64_t n, bool inclusive, T init, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
  if (nb > INT32_MAX) return hipErrorInvalidValue;
  if (nb == 1) {
    hipLaunchKernelGGL(scan_apply_kernel<T>, dim3(1), dim3(NT), 0, st, in, out, n, (const T*)nullptr,
                       inclusive ? 1 : 0, init);
    return hipGetLastError();
  }
  T* sums = (T*)tmp;
  T* offs = (T*)((char*)tmp + align256((size_t)nb * sizeof(T)));
  void* next = (char*)tmp + 2 * align256((size_t)nb * sizeof(T));
  hipLaunchKernelGGL(scan_reduce_kernel<T>, dim3((unsigned)nb), dim3(NT), 0, st, in, n, sums);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  e = scan(next, (const T*)sums, offs, nb, false, T(0), st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(scan_apply_kernel<T>, dim3((unsigned)nb), dim3(NT), 0, st, in, out, n, (const T*)offs,
                     inclusive ? 1 : 0, init);
  return hipGetLastError();
}

// rocPRIM-style entry points: tmp == nullptr stores the temporary size.
template <typename T>
hipError_t inclusive_scan(void* tmp, size_t& tmp_bytes, const T* in, T* out, int64_t n, hipStream_t st = 0) {
  if (!tmp) {
    tmp_bytes = scan_tmp_bytes(n, sizeof(T));
    return hipSuccess;
  }
  return scan(tmp, in, out, n, true, T(0), st);
}
template <typename T>
hipError_t exclusive_scan(void* tmp, size_t& tmp_bytes, const T* in, T* out, T init, int64_t n,
                          hipStream_t st = 0) {
  if (!tmp) {
    tmp_bytes = scan_tmp_bytes(n, sizeof(T));
    return hipSuccess;
  }
  return scan(tmp, in, out, n, false, init, st);
}

// ------------------------------------------------------------------ sort

template <typename K>
__device__ inline uint32_t digit_of(K k, int shift, uint32_t mask) {
  return (uint32_t)(k >> shift) & mask;
}

// One thread per digit: 1 << B threads.
template <typename K, int B>
__global__ __launch_bounds__(1 << B) void rs_count_kernel(const K* __restrict__ keys, int64_t n, int shift,
                                                          uint32_t mask, uint32_t* __restrict__ counts) {
  constexpr int RADIX = 1 << B, W = RADIX / 64, IPT = SORT_TILE / RADIX;
  __shared__ uint32_t h[W][RADIX];
  const int tid = threadIdx.x, w = tid >> 6;
  for (int i = tid; i < W * RADIX; i += RADIX) (&h[0][0])[i] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * SORT_TILE;
  if (base + SORT_TILE <= n && ((uintptr_t)keys & 15) == 0) {
    // full tile: counting ignores order, so each thread takes IPT consecutive keys in 16-byte loads
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    constexpr int PER = 16 / (int)sizeof(K), NV = IPT / PER;
    const u32x4* p = (const u32x4*)(keys + base + (int64_t)tid * IPT);
    u32x4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = p[j];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const K* kk = (const K*)&v[j];
#pragma unroll
      for (int e = 0; e < PER; ++e) atomicAdd(&h[w][digit_of(kk[e], shift, mask)], 1u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < IPT; ++i) {
      const int64_t idx = base + i * RADIX + tid;
      if (idx < n) atomicAdd(&h[w][digit_of(keys[idx], shift, mask)], 1u);
    }
  }
  __syncthreads();
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < W; ++i) s += h[i][tid];
  counts[(int64_t)blockIdx.x * RADIX + tid] = s;
}

// counts[t][d] <- the counts of d in the tiles before t, in place, and
// totals[d]. Workgroup of 8 digits x 128 parts of the tiles (32 bytes of a
// table row per load): each thread sums its part, 16 loads in flight, the parts
// of a digit are scanned, and each thread walks its part again.
constexpr int OFF_D = 8, OFF_PARTS = 128;
__global__ __launch_bounds__(OFF_D * OFF_PARTS) inline void rs_offsets_kernel(uint32_t* __restrict__ counts,
                                                                              int64_t ntiles, int radix,
                                                                              uint32_t* __restrict__ totals) {
  __shared__ uint32_t part[OFF_PARTS][OFF_D];
  const int d = threadIdx.x % OFF_D, p = threadIdx.x / OFF_D;
  const int64_t per = (ntiles + OFF_PARTS - 1) / OFF_PARTS;
  const int64_t r0 = p * per < ntiles ? p * per : ntiles;
  const int64_t r1 = r0 + per < ntiles ? r0 + per : ntiles;
  uint32_t* col = counts + blockIdx.x * OFF_D + d;
  uint32_t s = 0;
  int64_t t = r0;
  for (; t + 16 <= r1; t += 16) {
    uint32_t v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = col[(t + j) * radix];
#pragma unroll
    for (int j = 0; j < 16; ++j) s += v[j];
  }
  for (; t < r1; ++t) s += col[t * radix];
  part[p][d] = s;
  __syncthreads();
  if (threadIdx.x < 64) {  // lane (d, e): parts 16 e .. 16 e + 15 of digit d
    const int e = threadIdx.x / OFF_D;
    constexpr int EACH = OFF_PARTS * OFF_D / 64;
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < EACH; ++i) acc += part[EACH * e + i][d];
    uint32_t x = acc;  // inclusive over the lanes of the digit
#pragma unroll
    for (int o = OFF_D; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if ((int)threadIdx.x >= o) x += y;
    }
    if (e == 64 / OFF_D - 1) totals[blockIdx.x * OFF_D + d] = x;
    uint32_t run = x - acc;
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const uint32_t v = part[EACH * e + i][d];
      part[EACH * e + i][d] = run;
      run += v;
    }
  }
  __syncthreads();
  uint32_t run = part[p][d];
  for (t = r0; t + 16 <= r1; t += 16) {
    uint32_t v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = col[(t + j) * radix];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      col[(t + j) * radix] = run;
      run += v[j];
    }
  }
  for (; t < r1; ++t) {
    const uint32_t v = col[t * radix];
    col[t * radix] = run;
    run += v;
  }
}

// Where a pass stores the value of output position i: a plain array, or in
// the last pass a caller's writer (e.g. fields to separate arrays).
template <typename V>
struct VStore {
  V* p;
  __device__ void operator()(int64_t i, const V& v) const { p[i] = v; }
};

template <typename K, typename V, int B, typename VW>
__global__ __launch_bounds__(1 << B) void rs_scatter_kernel(const K* __restrict__ kin, const V* __restrict__ vin,
                                                            K* __restrict__ kout, VW vout, int64_t n, int shift,
                                                            uint32_t mask, const uint32_t* __restrict__ offs,
                                                            const uint32_t* __restrict__ totals) {
  constexpr int RADIX = 1 << B, W = RADIX / 64, IPT = SORT_TILE / RADIX, TILE = SORT_TILE;
  constexpr int Q = TILE / W;                // keys per wavefront, contiguous
  __shared__ uint16_t hw[W][RADIX];          // per wavefront: running count of each digit, then its start
  __shared__ uint32_t gbase[RADIX];          // output start of digit d's keys from this tile
  __shared__ uint32_t lbase[RADIX];          // start of digit d in the tile reordered by digit
  __shared__ K sk[TILE];
  __shared__ V sv[TILE];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  for (int i = tid; i < W * RADIX / 2; i += RADIX) ((uint32_t*)&hw[0][0])[i] = 0;
  const uint32_t before_tile = offs[(int64_t)blockIdx.x * RADIX + tid], digit_total = totals[tid];
  __syncthreads();
  const int64_t wbase = (int64_t)blockIdx.x * TILE + (int64_t)w * Q;  // round i, lane l: key wbase + 64 i + l
  const uint64_t lt = (1ull << lane) - 1;
  K k[IPT];
  V val[IPT];
  uint32_t dg[IPT], rk[IPT];
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const int64_t idx = wbase + 64 * i + lane;
    if (idx < n) {
      k[i] = kin[idx];
      val[i] = vin[idx];
    } else {
      k[i] = K(0);
    }
  }
  // rank of each key among the equal digits before it in the wavefront's
  // keys: the wavefront's running count of the digit (LDS, read by every
  // lane of the group before its leader adds the group) plus the rank among
  // this round's lanes with the same digit (a ballot per bit)
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const bool valid = wbase + 64 * i + lane < n;
    dg[i] = digit_of(k[i], shift, mask);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const bool bit = (dg[i] >> b) & 1;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const uint32_t below = (uint32_t)__popcll(peers & lt);
    const uint32_t before = hw[w][dg[i]];
    rk[i] = before + below;
    if (valid && below == 0) hw[w][dg[i]] = (uint16_t)(before + __popcll(peers));
  }
  __syncthreads();
  // digit tid: starts of its wavefront groups in key order, and its tile total
  uint32_t run = 0;
#pragma unroll
  for (int v = 0; v < W; ++v) {
    const uint32_t c = hw[v][tid];
    hw[v][tid] = (uint16_t)run;
    run += c;
  }
  uint32_t total;
  lbase[tid] = block_exclusive_scan<uint32_t, W>(run, total);
  gbase[tid] = before_tile + block_exclusive_scan<uint32_t, W>(digit_total, total);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    if (wbase + 64 * i + lane < n) {
      const uint32_t p = lbase[dg[i]] + hw[w][dg[i]] + rk[i];
      if (p < (uint32_t)TILE) {  // always true; keeps a miscount from writing outside the tile
        sk[p] = k[i];
        sv[p] = val[i];
      }
    }
  }
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * TILE;
  const int cnt_tile = (int)(n - base < TILE ? n - base : TILE);
  for (int j = tid; j < cnt_tile; j += RADIX) {
    const K kk = sk[j];
    const uint32_t d = digit_of(kk, shift, mask);
    const int64_t pos = (int64_t)gbase[d] + (j - (int64_t)lbase[d]);
    if (pos >= 0 && pos < n) {  // always true; keeps a miscount from writing outside the output
      kout[pos] = kk;
      vout(pos, sv[j]);
    }
  }
}

// zero key bits: the input in order, through the writer
template <typename K, typename V, typename VW>
__global__ __launch_bounds__(NT) void rs_copy_kernel(const K* __restrict__ kin, const V* __restrict__ vin,
                                                     K* __restrict__ kout, VW vout, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * NT + threadIdx.x;
  if (i < n) {
    kout[i] = kin[i];
    vout(i, vin[i]);
  }
}

// A table of many tiles: the column sums of chunks of ch tiles, which
// rs_offsets turns into the counts of the chunks before, and each chunk's
// tiles in order from there.
template <bool APPLY>
__global__ __launch_bounds__(256) void rs_chunk_kernel(uint32_t* __restrict__ counts, int64_t ntiles, int64_t ch,
                                                       int radix, uint32_t* __restrict__ csum) {
  const int d = blockIdx.y * 256 + threadIdx.x;
  const int64_t t0 = (int64_t)blockIdx.x * ch, t1 = t0 + ch < ntiles ? t0 + ch : ntiles;
  uint32_t* col = counts + d;
  uint32_t* sum = csum + (int64_t)blockIdx.x * radix + d;
  uint32_t run = APPLY ? *sum : 0;
  int64_t t = t0;
  for (; t + 16 <= t1; t += 16) {
    uint32_t v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = col[(t + j) * radix];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      if (APPLY) col[(t + j) * radix] = run;
      run += v[j];
    }
  }
  for (; t < t1; ++t) {
    const uint32_t v = col[t * radix];
    if (APPLY) col[t * radix] = run;
    run += v;
  }
  if (!APPLY) *sum = run;
}

// Tiles per chunk (1: rs_offsets walks the tiles themselves, a launch instead
// of three: transposes of 1 M entries 72 against 80 us, 4 M 133 of 132; its few
// workgroups lose on a longer table: 16 M 519 against 489, 128 M 4462 of 3957).
// At most 1024 chunks.
inline int64_t chunk_tiles(int64_t ntiles) {
  return ntiles <= 1024 ? 1 : ntiles > 32 * 1024 ? (ntiles + 1023) / 1024 : 32;
}

template <int B, typename K, typename V, typename VW>
hipError_t sort_pass(const K* kin, const V* vin, K* kout, VW vout, int64_t n, int shift, int bits, uint32_t* counts,
                     uint32_t* csum, uint32_t* totals, hipStream_t st) {
  const int64_t ntiles = (n + SORT_TILE - 1) / SORT_TILE;
  const uint32_t mask = (1u << bits) - 1;
  hipLaunchKernelGGL((rs_count_kernel<K, B>), dim3((unsigned)ntiles), dim3(1 << B), 0, st, kin, n, shift, mask, counts);
  const int64_t ch = chunk_tiles(ntiles), nch = (ntiles + ch - 1) / ch;
  const dim3 cg((unsigned)nch, (1 << B) / 256);
  if (ch > 1)
    hipLaunchKernelGGL(rs_chunk_kernel<false>, cg, dim3(256), 0, st, counts, ntiles, ch, 1 << B, csum);
  hipLaunchKernelGGL(rs_offsets_kernel, dim3((1 << B) / OFF_D), dim3(OFF_D * OFF_PARTS), 0, st, ch > 1 ? csum : counts,
                     nch, 1 << B, totals);
  if (ch > 1) hipLaunchKernelGGL(rs_chunk_kernel<true>, cg, dim3(256), 0, st, counts, ntiles, ch, 1 << B, csum);
  hipLaunchKernelGGL((rs_scatter_kernel<K, V, B, VW>), dim3((unsigned)ntiles), dim3(1 << B), 0, st, kin, vin, kout, vout,
                     n, shift, mask, (const uint32_t*)counts, (const uint32_t*)totals);
  return hipGetLastError();
}

// Stable sort of (kin, vin)[0, n) by key bits [begin_bit, end_bit) into (kout, vout);
// the inputs are left unchanged. tmp == nullptr stores the temporary size.
// Keys must be unsigned; n < 2^32.
// radix_sort_pairs_to: the same, with the last pass's values stored by
// `last` (vout then only serves as scratch between passes).
template <typename K, typename V, typename LastW>
hipError_t radix_sort_pairs_to(void* tmp, size_t& tmp_bytes, const K* kin, K* kout, const V* vin, V* vout,
                               int64_t n, int begin_bit, int end_bit, LastW last, hipStream_t st = 0) {
  if (n < 0 || n > (int64_t)UINT32_MAX || begin_bit < 0 || end_bit > (int)(8 * sizeof(K)) || end_bit < begin_bit)
    return hipErrorInvalidValue;
  const int nbits = end_bit - begin_bit;
  const int p8 = (nbits + 7) / 8, p9 = (nbits + 8) / 9;
  // A pass less pays while the pairs stay in the 256 MB memory-side cache, and
  // where a tile of 256 threads has the CU to itself (20-byte pairs): sorts on
  // 18 bits in a transpose, us at 9 / 8 bits a digit: 12-byte pairs, 1 M 71 /
  // 87, 4 M 131 / 155, 8 M 290 / 277, 16 M 585 / 525 (runs of 8 keys per digit
  // and tile against 64); 20-byte pairs, 1 M 102 / 141, 16 M 877 / 1312.
  constexpr int PAIR = (int)(sizeof(K) + sizeof(V));
  const bool nine = p9 < p8 && (PAIR >= 20 || n <= (64 << 20) / PAIR);
  const int passes = nine ? p9 : p8, radix = nine ? 512 : 256;
  const int64_t ntiles = (n + SORT_TILE - 1) / SORT_TILE;
  const size_t kb = align256((size_t)n * sizeof(K)), vb = align256((size_t)n * sizeof(V));
  const size_t cb = align256((size_t)radix * (ntiles > 0 ? ntiles : 1) * sizeof(uint32_t));
  const int64_t ch = chunk_tiles(ntiles);
  const size_t sb = ch > 1 ? align256((size_t)radix * ((ntiles + ch - 1) / ch) * sizeof(uint32_t)) : 0;
  const size_t need = kb + vb + cb + sb + align256((size_t)radix * sizeof(uint32_t));
  if (!tmp) {
    tmp_bytes = need;
    return hipSuccess;
  }
  if (tmp_bytes < need) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  K* tk = (K*)tmp;
  V* tv = (V*)((char*)tmp + kb);
  uint32_t* counts = (uint32_t*)((char*)tmp + kb + vb);
  uint32_t* csum = (uint32_t*)((char*)tmp + kb + vb + cb);
  uint32_t* totals = (uint32_t*)((char*)tmp + kb + vb + cb + sb);
  if (passes == 0) {
    hipLaunchKernelGGL((rs_copy_kernel<K, V, LastW>), dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, st, kin, vin,
                       kout, last, n);
    return hipGetLastError();
  }
  const int each = (nbits + passes - 1) / passes;
  const K* sk = kin;
  const V* sv = vin;
  for (int p = 0; p < passes; ++p) {
    // the last pass writes the output: an odd count starts there, an even one in tmp
    const bool to_out = ((passes - 1 - p) & 1) == 0;
    K* dk = to_out ? kout : tk;
    V* dv = to_out ? vout : tv;
    const int shift = begin_bit + each * p;
    const int bits = end_bit - shift < each ? end_bit - shift : each;
    hipError_t e;
    if (p == passes - 1)
      e = nine ? sort_pass<9>(sk, sv, dk, last, n, shift, bits, counts, csum, totals, st)
               : sort_pass<8>(sk, sv, dk, last, n, shift, bits, counts, csum, totals, st);
    else
      e = nine ? sort_pass<9>(sk, sv, dk, VStore<V>{dv}, n, shift, bits, counts, csum, totals, st)
               : sort_pass<8>(sk, sv, dk, VStore<V>{dv}, n, shift, bits, counts, csum, totals, st);
    if (e != hipSuccess) return e;
    sk = dk;
    sv = dv;
  }
  return hipSuccess;
}

template <typename K, typename V>
hipError_t radix_sort_pairs(void* tmp, size_t& tmp_bytes, const K* kin, K* kout, const V* vin, V* vout, int64_t n,
                            int begin_bit, int end_bit, hipStream_t st = 0) {
  return radix_sort_pairs_to(tmp, tmp_bytes, kin, kout, vin, vout, n, begin_bit, end_bit, VStore<V>{vout}, st);
}

}  // namespace rsort
}  // namespace tsp
