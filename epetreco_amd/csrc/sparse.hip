// sparse.hip -- COO sort, COO->CSR->ECSR, and library-matrix utilities.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <vector>

#include "epet_block.hpp"
#include "epet_internal.hpp"
#include "epet_rows.hpp"

namespace epet {

// ------------------------------------------------------------------ radix sort
// Stable LSD radix sort of (key, value) pairs with 8-bit digits.  A key packs
// (row, col) with flipped sign bits, so unsigned order = lexicographic signed
// (row, col) order, the order of cooIdLess (cooSort.hpp:26-44).  Digits on
// which all keys agree are skipped.
constexpr int RS_BLOCK = 256;
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = RS_BLOCK * RS_ITEMS;
constexpr int RS_BINS = 256;

__device__ __forceinline__ uint64_t coo_key(int row, int col) {
  return ((uint64_t)((uint32_t)row ^ 0x80000000u) << 32) | (uint64_t)((uint32_t)col ^ 0x80000000u);
}

__global__ __launch_bounds__(256) void k_pack_keys(const int* __restrict__ row,
                                                   const int* __restrict__ col, long long n,
                                                   uint64_t* __restrict__ key) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  key[i] = coo_key(row[i], col[i]);
}

__global__ __launch_bounds__(256) void k_unpack_keys(const uint64_t* __restrict__ key,
                                                     long long n, int* __restrict__ row,
                                                     int* __restrict__ col) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t k = key[i];
  row[i] = (int)((uint32_t)(k >> 32) ^ 0x80000000u);
  col[i] = (int)((uint32_t)k ^ 0x80000000u);
}

// One read of the (row, col) pairs: bitwise AND and OR over all keys (digits
// where they agree are constant), and whether any key is below the one before
// it (out[2]).  Bound by the 8 bytes per pair it reads: a lane takes four pairs by
// two 16-byte loads, the key before them comes from the lane before (with two
// 4-byte reads of every pair, 40M pairs took 30 us more).  The atomics on one cache
// line are taken one by one, so few large workgroups reduce before theirs: 40M
// pairs 99 us, 113 with 2,048 workgroups of 256 threads, 411 with atomics per wavefront.
constexpr int SCAN_BLOCK = 1024;
typedef int coo_i4 __attribute__((ext_vector_type(4), aligned(4)));
__global__ __launch_bounds__(SCAN_BLOCK) void k_coo_scan(const int* __restrict__ row,
                                                  const int* __restrict__ col, long long n,
                                                  unsigned long long* __restrict__ out) {
  __shared__ unsigned long long s_a[SCAN_BLOCK / WAVE], s_o[SCAN_BLOCK / WAVE];
  __shared__ int s_f[SCAN_BLOCK / WAVE];
  uint64_t a = ~0ull, o = 0ull;
  bool below = false;
  const long long nq = n / 4;
  const int lane = lane_id();
  for (long long q0 = (long long)blockIdx.x * SCAN_BLOCK + wave_id() * WAVE; q0 < nq;
       q0 += (long long)gridDim.x * SCAN_BLOCK) {
    const bool in = q0 + lane < nq;
    const long long q = in ? q0 + lane : nq - 1;
    const coo_i4 r = *reinterpret_cast<const coo_i4*>(row + 4 * q);
    const coo_i4 c = *reinterpret_cast<const coo_i4*>(col + 4 * q);
    const long long before = q0 > 0 ? 4 * q0 - 1 : 0;
    const uint64_t first = coo_key(row[before], col[before]);
    uint64_t k[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      k[i] = coo_key(r[i], c[i]);
      a &= k[i];
      o |= k[i];
      if (i > 0) below |= k[i] < k[i - 1];
    }
    uint64_t prev = __shfl_up(k[3], 1, WAVE);
    if (lane == 0) prev = first;
    below |= in && k[0] < prev;
  }
  // the last 0 to 3 pairs
  if (blockIdx.x == 0 && threadIdx.x < (unsigned)(n - 4 * nq)) {
    const long long i = 4 * nq + threadIdx.x;
    const uint64_t k = coo_key(row[i], col[i]);
    a &= k;
    o |= k;
    if (i > 0) below |= k < coo_key(row[i - 1], col[i - 1]);
  }
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1) {
    a &= __shfl_xor(a, off, WAVE);
    o |= __shfl_xor(o, off, WAVE);
  }
  const bool any = __any(below);
  if (lane_id() == 0) {
    s_a[wave_id()] = a;
    s_o[wave_id()] = o;
    s_f[wave_id()] = any;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < SCAN_BLOCK / WAVE; w++) {
      a &= s_a[w];
      o |= s_o[w];
      s_f[0] |= s_f[w];
    }
    atomicAnd(&out[0], (unsigned long long)a);
    atomicOr(&out[1], (unsigned long long)o);
    if (s_f[0]) atomicOr(&out[2], 1ull);
  }
}

__global__ void k_init_scan(unsigned long long* out) {
  if (threadIdx.x == 0) { out[0] = ~0ull; out[1] = 0ull; out[2] = 0ull; }
}

__global__ __launch_bounds__(RS_BLOCK) void k_rs_hist(const uint64_t* __restrict__ key,
                                                      long long n, int shift, int ntiles,
                                                      int* __restrict__ hist) {
  __shared__ int h[RS_BINS];
  h[threadIdx.x] = 0;
  __syncthreads();
  const long long base = (long long)blockIdx.x * RS_TILE;
#pragma unroll
  for (int j = 0; j < RS_ITEMS; j++) {
    const long long i = base + j * RS_BLOCK + threadIdx.x;
    if (i < n) atomicAdd(&h[(key[i] >> shift) & 0xFF], 1);
  }
  __syncthreads();
  hist[(long long)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(RS_BLOCK) void k_rs_scatter(const uint64_t* __restrict__ kin,
                                                         const float* __restrict__ vin,
                                                         long long n, int shift, int ntiles,
                                                         const int64_t* __restrict__ offs,
                                                         uint64_t* __restrict__ kout,
                                                         float* __restrict__ vout) {
  __shared__ int64_t s_base[RS_BINS];
  __shared__ int s_run[RS_BINS];
  __shared__ int s_wcnt[RS_BLOCK / WAVE][RS_BINS];
  const int tid = threadIdx.x;
  s_base[tid] = offs[(long long)tid * ntiles + blockIdx.x];
  s_run[tid] = 0;
  const int w = wave_id(), lane = lane_id();
  const uint64_t lt = lane ? (~0ull >> (64 - lane)) : 0ull;
  const long long base = (long long)blockIdx.x * RS_TILE;
  for (int j = 0; j < RS_ITEMS; j++) {
#pragma unroll
    for (int q = 0; q < RS_BLOCK / WAVE; q++) s_wcnt[q][tid] = 0;
    __syncthreads();
    const long long i = base + j * RS_BLOCK + tid;
    const bool valid = i < n;
    uint64_t k = 0;
    float v = 0.0f;
    if (valid) { k = kin[i]; v = vin[i]; }
    const int d = (int)((k >> shift) & 0xFF);
    // lanes of this wavefront holding the same digit
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const bool bit = (d >> b) & 1;
      const uint64_t bal = __ballot(bit);
      peers &= bit ? bal : ~bal;
    }
    const int rank = __popcll(peers & lt);
    if (valid && rank == 0) s_wcnt[w][d] = __popcll(peers);
    __syncthreads();
    if (valid) {
      int before = 0;
      for (int q = 0; q < w; q++) before += s_wcnt[q][d];
      const int64_t pos = s_base[d] + s_run[d] + before + rank;
      kout[pos] = k;
      vout[pos] = v;
    }
    __syncthreads();
    int add = 0;
#pragma unroll
    for (int q = 0; q < RS_BLOCK / WAVE; q++) add += s_wcnt[q][tid];
    s_run[tid] += add;
    __syncthreads();
  }
}

// ------------------------------------------------------------------ CSR helpers
__global__ __launch_bounds__(256) void k_fill_i32(int* __restrict__ p, long long n, int v) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Entries per row id; row ids outside [0, m) are not counted (and flagged).
// A wavefront walks HIST_SPAN consecutive entries and counts runs of equal ids
// before it adds them: row ids come sorted or nearly so, and one atomic per
// entry serialises on the row's counter (40M entries of 2,001 sorted rows:
// 32.8 ms, with runs 0.1 ms, near the read of the ids).
constexpr int HIST_SPAN = 16 * WAVE;
constexpr int HIST_AHEAD = 8;   // loads of a wavefront in flight (40M sorted ids: 47 us, with one 61)
__global__ __launch_bounds__(256) void k_row_hist(const int* __restrict__ rowid, long long nnz,
                                                  int m, int* __restrict__ cnt,
                                                  int* __restrict__ bad) {
  const int lane = lane_id();
  auto add = [&](int r, int n) {
    if (r >= 0 && r < m) atomicAdd(&cnt[r], n);
    else atomicOr(bad, 1);
  };
  const long long nw = (long long)gridDim.x * (256 / WAVE);
  for (long long span = (long long)blockIdx.x * (256 / WAVE) + wave_id(); span * HIST_SPAN < nnz;
       span += nw) {
    const long long b = span * HIST_SPAN;
    const long long e = b + HIST_SPAN < nnz ? b + HIST_SPAN : nnz;
    int cur = 0, run = 0;   // wavefront-uniform: the run that reaches the end of the last 64
    for (long long at = b; at < e; at += HIST_AHEAD * WAVE) {
      int ahead[HIST_AHEAD];
#pragma unroll
      for (int j = 0; j < HIST_AHEAD; j++) {
        const long long i = at + j * WAVE + lane;
        ahead[j] = rowid[i < e ? i : e - 1];
      }
#pragma unroll
      for (int j = 0; j < HIST_AHEAD; j++) {
        const long long base = at + j * WAVE;
        if (base >= e) break;
        const bool in = base + lane < e;
        const int r = ahead[j];
        const int n = (int)(e - base < WAVE ? e - base : WAVE);
        if (run > 0 && __all(!in || r == cur)) {
          run += n;
          continue;
        }
        if (run > 0 && lane == 0) add(cur, run);
        // runs within these n entries; the last one is carried on
        const int prev = __shfl_up(r, 1, WAVE);
        const unsigned long long heads = __ballot(in && (lane == 0 || r != prev));
        const int last = 63 - __clzll((long long)heads);
        if (in && lane != last && ((heads >> lane) & 1)) {
          const unsigned long long after = heads & (~0ull << lane << 1);
          add(r, __ffsll((long long)after) - 1 - lane);
        }
        cur = __shfl(r, last, WAVE);
        run = n - last;
      }
    }
    if (run > 0 && lane == 0) add(cur, run);
  }
}

__global__ __launch_bounds__(256) void k_csr2ecsr(int* __restrict__ ecsr,
                                                  const int* __restrict__ yRowId, int nnzr,
                                                  const int* __restrict__ csr, int m) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nnzr) {
    const int y = yRowId[i];
    ecsr[i] = (y >= 0 && y <= m) ? csr[y] : -1;   // -1 marks an out-of-range row id
  }
  if (i == nnzr) ecsr[nnzr] = csr[m];
}

__global__ __launch_bounds__(256) void k_sel_counts(const int64_t* __restrict__ rowptr,
                                                    const int* __restrict__ rows, int nrows,
                                                    int m, int* __restrict__ cnt,
                                                    int* __restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nrows) return;
  const int r = rows[i];
  if (r < 0 || r >= m) { atomicOr(bad, 1); cnt[i] = 0; return; }
  cnt[i] = (int)(rowptr[r + 1] - rowptr[r]);
}

template <typename V>
__global__ __launch_bounds__(256) void k_sel_copy(const int64_t* __restrict__ rowptr,
                                                  const int* __restrict__ col,
                                                  const V* __restrict__ val,
                                                  const float* __restrict__ scale,
                                                  const int* __restrict__ rows, int m,
                                                  const int64_t* __restrict__ off,
                                                  int64_t* __restrict__ orow,
                                                  int* __restrict__ ocol, V* __restrict__ oval,
                                                  float* __restrict__ oscale) {
  const int i = blockIdx.x;
  const int r = rows[i];
  const int64_t o = off[i];
  if (threadIdx.x == 0) {
    orow[i] = o;
    if (oscale) oscale[i] = (r >= 0 && r < m) ? scale[r] : 0.0f;
  }
  if (r < 0 || r >= m) return;
  const int64_t b = rowptr[r], e = rowptr[r + 1];
  for (int64_t k = b + threadIdx.x; k < e; k += blockDim.x) {
    ocol[o + (k - b)] = col[k];
    oval[o + (k - b)] = val[k];
  }
}

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// per-row scale = max |a|; stored value = a / scale
__global__ __launch_bounds__(256) void k_convert_rows(const int64_t* __restrict__ rowptr,
                                                      const float* __restrict__ val, int vt,
                                                      uint16_t* __restrict__ out,
                                                      float* __restrict__ scale) {
  __shared__ float s_w[256 / WAVE];
  const int r = blockIdx.x;
  const int64_t b = rowptr[r], e = rowptr[r + 1];
  float mx = 0.0f;
  for (int64_t k = b + threadIdx.x; k < e; k += blockDim.x) mx = fmaxf(mx, fabsf(val[k]));
#pragma unroll
  for (int off = WAVE / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, WAVE));
  if (lane_id() == 0) s_w[wave_id()] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_w[0], s_w[1]), fmaxf(s_w[2], s_w[3]));
  const float sc = mx > 0.0f ? mx : 1.0f;
  if (threadIdx.x == 0) scale[r] = sc;
  for (int64_t k = b + threadIdx.x; k < e; k += blockDim.x) {
    const float q = val[k] / sc;
    out[k] = (vt == EPET_VAL_BF16) ? f32_to_bf16_rne(q) : __half_as_ushort(__float2half_rn(q));
  }
}

template <typename V>
__device__ __forceinline__ float load_val(const V* p, long long k);
template <>
__device__ __forceinline__ float load_val<float>(const float* p, long long k) { return p[k]; }

__global__ __launch_bounds__(256) void k_colsum_f64(const int64_t* __restrict__ rowptr,
                                                    const int* __restrict__ col,
                                                    const void* __restrict__ val, int vt,
                                                    const float* __restrict__ scale, int m,
                                                    double* __restrict__ s) {
  const int r = blockIdx.x;
  if (r >= m) return;
  const int64_t b = rowptr[r], e = rowptr[r + 1];
  const float sc = scale ? scale[r] : 1.0f;
  for (int64_t k = b + threadIdx.x; k < e; k += blockDim.x) {
    float a;
    if (vt == EPET_VAL_F32) a = ((const float*)val)[k];
    else if (vt == EPET_VAL_BF16)
      a = __uint_as_float((uint32_t)((const uint16_t*)val)[k] << 16) * sc;
    else a = __half2float(__ushort_as_half(((const uint16_t*)val)[k])) * sc;
    unsafeAtomicAdd(&s[col[k]], (double)a);
  }
}

__global__ __launch_bounds__(256) void k_fill_f64(double* __restrict__ p, long long n) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

__global__ void k_set_last_i64(int64_t* p, int64_t v) {
  if (threadIdx.x == 0) *p = v;
}

__global__ __launch_bounds__(256) void k_gather_i32(const int* __restrict__ src,
                                                    const int* __restrict__ idx, int n,
                                                    int* __restrict__ dst) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

// Structure check of caller arrays: bit 1 = invalid (row pointers not
// monotone / not spanning [0, nnz], column outside [0, n)); bit 2 = columns not
// strictly ascending within a row.
__global__ __launch_bounds__(256) void k_check_csr(int m, int n, long long nnz,
                                                   const int64_t* __restrict__ rowptr,
                                                   const int* __restrict__ col,
                                                   int* __restrict__ flags) {
  const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m) return;
  const int64_t b = rowptr[r], e = rowptr[r + 1];
  int f = 0;
  if (r == 0 && b != 0) f |= 1;
  if (r == m - 1 && e != nnz) f |= 1;
  if (e < b || b < 0 || e > nnz) f |= 1;
  else {
    int prev = -1;
    for (int64_t k = b; k < e; k++) {
      const int c = col[k];
      if (c < 0 || c >= n) { f |= 1; break; }
      if (c <= prev) f |= 2;
      prev = c;
    }
  }
  if (f) atomicOr(flags, f);
}

}  // namespace epet

using namespace epet;

namespace epet {
// ------------------------------------------------------------------ transpose
// Deterministic transpose without global atomics.  Columns are cut into tiles
// whose counters fit LDS and rows into blocks; workgroup (tile, block) counts
// its entries per column with LDS atomics, a prefix over the blocks of every
// column turns the counts into start positions, and a second walk of the rows
// in order places the entries, one row per step (columns are distinct within a
// row), each step closed by a barrier on LDS only.  Entries of a column come
// out in ascending row order.
//
// The row walk is a chain of LDS read, write and barrier; what bounds the whole
// is the scattered 4-byte writes of the transposed entries.  Counters in memory
// instead of LDS (a read and a write of one random line per entry and pass) took
// 39.0 ms for 100,000 rows of 916 entries over 140,608 columns, this 4.0 ms.
constexpr int TR_BLOCK = 1024;
constexpr int TR_AHEAD = 4;
constexpr int TR_LDS = 144 * 1024;   // counters of a workgroup, of 160 KB of LDS
constexpr int TR_GRID = 1024;        // workgroups aimed at: 4 per CU, one after the other

// positions of a tile's entries within a batch of TR_BLOCK rows, one row per
// thread (columns ascend within a row)
__device__ __forceinline__ void tr_bounds(const int64_t* rowptr, const int* col, long long r,
                                          long long r1, int c0, int c1, int64_t* s_lo, int* s_n) {
  int64_t lo = 0, hi = 0;
  if (r < r1) {
    const int64_t b = rowptr[r], e = rowptr[r + 1];
    auto first_at = [&](int64_t from, int c) {   // first entry of the row with column >= c
      int64_t l = from, h = e;
      while (l < h) {
        const int64_t mid = (l + h) >> 1;
        if (col[mid] < c) l = mid + 1; else h = mid;
      }
      return l;
    };
    lo = first_at(b, c0);
    hi = first_at(lo, c1);
  }
  s_lo[threadIdx.x] = lo;
  s_n[threadIdx.x] = (int)(hi - lo);
}

// cnt[blk n + c]: entries of column c in row block blk
__global__ __launch_bounds__(TR_BLOCK) void k_tr_count(int m, int n, int T, int tile,
                                                       int rows_per_block,
                                                       const int64_t* __restrict__ rowptr,
                                                       const int* __restrict__ col,
                                                       uint32_t* __restrict__ cnt) {
  extern __shared__ uint32_t tr_c[];
  __shared__ int64_t s_lo[TR_BLOCK];
  __shared__ int s_n[TR_BLOCK];
  const int t = blockIdx.x % T;
  const long long blk = blockIdx.x / T;
  const int c0 = t * tile, c1 = min(n, c0 + tile);
  for (int i = threadIdx.x; i < c1 - c0; i += TR_BLOCK) tr_c[i] = 0;
  const long long r0 = blk * rows_per_block, r1 = min((long long)m, r0 + rows_per_block);
  for (long long rb = r0; rb < r1; rb += TR_BLOCK) {
    __syncthreads();
    tr_bounds(rowptr, col, rb + threadIdx.x, r1, c0, c1, s_lo, s_n);
    __syncthreads();
    const int nr = (int)min((long long)TR_BLOCK, r1 - rb);
    for (int i = wave_id(); i < nr; i += TR_BLOCK / WAVE) {
      const int64_t lo = s_lo[i];
      const int len = s_n[i];
      for (int k = lane_id(); k < len; k += 4 * WAVE) {
        int c[4];   // four loads requested together
#pragma unroll
        for (int j = 0; j < 4; j++) c[j] = k + j * WAVE < len ? col[lo + k + j * WAVE] : -1;
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (c[j] >= 0) atomicAdd(&tr_c[c[j] - c0], 1u);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < c1 - c0; i += TR_BLOCK) cnt[blk * n + c0 + i] = tr_c[i];
}

// Column sums in FP64: workgroup (tile, row block) adds its entries into doubles in
// LDS and then each column once to memory.  s is zero before.  100,000 rows of 885
// entries, 52^3 columns: 1.17 ms with an atomic in memory per entry, 0.35 ms so.
constexpr int CS_TILE = 16384;   // doubles of a workgroup, 128 KB
template <typename VT>
__global__ __launch_bounds__(TR_BLOCK) void k_colsum_tiles(int m, int n, int T, int rows_per_block,
                                                           const int64_t* __restrict__ rowptr,
                                                           const int* __restrict__ col,
                                                           const typename VT::T* __restrict__ val,
                                                           const float* __restrict__ scale,
                                                           double* __restrict__ s) {
  extern __shared__ double cs_sum[];
  __shared__ int64_t s_lo[TR_BLOCK];
  __shared__ int s_n[TR_BLOCK];
  const int t = blockIdx.x % T;
  const long long blk = blockIdx.x / T;
  const int c0 = t * CS_TILE, c1 = min(n, c0 + CS_TILE);
  for (int i = threadIdx.x; i < c1 - c0; i += TR_BLOCK) cs_sum[i] = 0.0;
  const long long r0 = blk * rows_per_block, r1 = min((long long)m, r0 + rows_per_block);
  for (long long rb = r0; rb < r1; rb += TR_BLOCK) {
    __syncthreads();
    tr_bounds(rowptr, col, rb + threadIdx.x, r1, c0, c1, s_lo, s_n);
    __syncthreads();
    const int nr = (int)min((long long)TR_BLOCK, r1 - rb);
    for (int i = wave_id(); i < nr; i += TR_BLOCK / WAVE) {
      const int64_t lo = s_lo[i];
      const int len = s_n[i];
      const float sc = scale ? scale[rb + i] : 1.0f;
      for (int k = lane_id(); k < len; k += 4 * WAVE) {
        int c[4];   // four entries requested together
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const bool in = k + j * WAVE < len;
          c[j] = in ? col[lo + k + j * WAVE] : -1;
          v[j] = in ? VT::get_cached(val, lo + k + j * WAVE) : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (c[j] >= 0) unsafeAtomicAdd(&cs_sum[c[j] - c0], (double)(v[j] * sc));
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < c1 - c0; i += TR_BLOCK)
    if (cs_sum[i] != 0.0) unsafeAtomicAdd(&s[c0 + i], cs_sum[i]);
}

template <typename VT>
static int launch_colsum_tiles(epet_ctx* ctx, const epet_matrix* A, double* s) {
  const int T = (A->n + CS_TILE - 1) / CS_TILE;
  // four workgroups per CU in turn, and rows enough for each to make up for adding
  // its columns to memory
  const int want = std::max(1, 4 * ctx->num_cus / T);
  const int rpb = std::max(16, (A->m + want - 1) / want);
  const long long grid = (long long)((A->m + rpb - 1) / rpb) * T;
  const size_t lds = sizeof(double) * (size_t)std::min(A->n, CS_TILE);
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)k_colsum_tiles<VT>,
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              CS_TILE * (int)sizeof(double));
  k_colsum_tiles<VT><<<(unsigned)grid, TR_BLOCK, lds, ctx->stream>>>(
      A->m, A->n, T, rpb, A->rowptr, A->col, (const typename VT::T*)A->val, A->rowscale, s);
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

// cnt[blk n + c] -> entries of column c before block blk; total[c] = all of them
__global__ __launch_bounds__(256) void k_tr_prefix(int n, int B, uint32_t* __restrict__ cnt,
                                                   int* __restrict__ total) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  uint32_t run = 0;
  for (int b = 0; b < B; b++) {
    const uint32_t v = cnt[(long long)b * n + c];
    cnt[(long long)b * n + c] = run;
    run += v;
  }
  total[c] = (int)run;
}

// P: the type of a position in the transposed arrays (32 bits where the entry
// count allows, so that a tile holds twice the columns)
template <typename V, typename P>
__global__ __launch_bounds__(TR_BLOCK) void k_tr_fill(int m, int n, int T, int tile,
                                                      int rows_per_block,
                                                      const int64_t* __restrict__ rowptr,
                                                      const int* __restrict__ col,
                                                      const V* __restrict__ val,
                                                      const uint32_t* __restrict__ cnt,
                                                      const int64_t* __restrict__ tptr,
                                                      int* __restrict__ orow,
                                                      V* __restrict__ oval) {
  extern __shared__ unsigned char tr_raw[];
  P* cur = reinterpret_cast<P*>(tr_raw);
  __shared__ int64_t s_lo[TR_BLOCK];
  __shared__ int s_n[TR_BLOCK];
  const int t = blockIdx.x % T;
  const long long blk = blockIdx.x / T;
  const int c0 = t * tile, c1 = min(n, c0 + tile);
  for (int i = threadIdx.x; i < c1 - c0; i += TR_BLOCK)
    cur[i] = (P)(tptr[c0 + i] + cnt[blk * n + c0 + i]);
  const long long r0 = blk * rows_per_block, r1 = min((long long)m, r0 + rows_per_block);
  for (long long rb = r0; rb < r1; rb += TR_BLOCK) {
    __syncthreads();
    tr_bounds(rowptr, col, rb + threadIdx.x, r1, c0, c1, s_lo, s_n);
    __syncthreads();
    const int nr = (int)min((long long)TR_BLOCK, r1 - rb);
    // this thread's first entries of the next TR_AHEAD rows, requested while
    // the TR_AHEAD before them are placed (4.5 ms against 4.9 one row ahead, both
    // with 256 threads)
    int cn[TR_AHEAD];
    V vn[TR_AHEAD];
    auto request = [&](int i0) {
#pragma unroll
      for (int j = 0; j < TR_AHEAD; j++) {
        cn[j] = -1;
        if (i0 + j < nr && (int)threadIdx.x < s_n[i0 + j]) {
          cn[j] = col[s_lo[i0 + j] + threadIdx.x] - c0;
          vn[j] = val[s_lo[i0 + j] + threadIdx.x];
        }
      }
    };
    request(0);
    for (int i0 = 0; i0 < nr; i0 += TR_AHEAD) {
      int c[TR_AHEAD];
      V v[TR_AHEAD];
#pragma unroll
      for (int j = 0; j < TR_AHEAD; j++) {
        c[j] = cn[j];
        v[j] = vn[j];
      }
      request(i0 + TR_AHEAD);
#pragma unroll
      for (int j = 0; j < TR_AHEAD; j++) {
        if (i0 + j >= nr) break;
        const int r = (int)(rb + i0 + j);
        if (c[j] >= 0) {
          const P pos = cur[c[j]];
          cur[c[j]] = pos + 1;
          orow[pos] = r;
          oval[pos] = v[j];
        }
        const int len = s_n[i0 + j];
        for (int k = threadIdx.x + TR_BLOCK; k < len; k += TR_BLOCK) {
          const int c2 = col[s_lo[i0 + j] + k] - c0;
          const P pos = cur[c2];
          cur[c2] = pos + 1;
          orow[pos] = r;
          oval[pos] = val[s_lo[i0 + j] + k];
        }
        // the next row's cursors are those this row left: wait for LDS, not for
        // the writes to memory that __syncthreads would wait for too
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    }
  }
}

// The same in two steps for longer rows.  What bounds k_tr_fill is its writes, 4
// bytes here and there over the whole of the transposed arrays (4.5 GB leave L2 for
// 0.7 GB of entries).  So the entries go first to the bucket of their TR_BUCKET
// columns, whose room is that of its columns in the result: entries of one row and
// bucket lie together (3 at 52^3), rows of a block follow one another, and one
// counter per bucket serves a workgroup for whole rows.  A workgroup then sorts a
// bucket in LDS, with the columns' next positions in its lanes and the rank of an
// entry among the 64 of a wavefront by ballots, and writes it in whole lines.
// Entries (rows of them), k_tr_fill against both steps: 2.7M (133) 90 and 78 us; 8.9M
// (885) 382 and 237; 89M (885) 3.24 and 1.71 ms; 87M (2,884, 104^3) 5.09 and 2.04.
// Writing pairs from k_tr_fill and splitting them took 2.48 ms for the 89M, buckets
// of 32 columns placed straight in memory 2.32.
constexpr int TR_BUCKET = 8, TR_BITS = 3;
constexpr int TRP_BLOCK = 512;
constexpr size_t TR_PAIR_BYTES = (size_t)1 << 30;   // of pairs

template <typename V> struct alignas(8) TrPair {
  unsigned key;   // row * TR_BUCKET + column in the bucket
  V val;
};

// first position of (bucket, row block blk) in pairs and result
__device__ __forceinline__ long long tr_bucket_start(long long n, long long blk, int bucket,
                                                     const uint32_t* __restrict__ cnt,
                                                     const int64_t* __restrict__ tptr) {
  const long long c0 = (long long)bucket * TR_BUCKET, c1 = min(n, c0 + TR_BUCKET);
  long long p = tptr[c0];
  for (long long c = c0; c < c1; c++) p += cnt[blk * n + c];
  return p;
}

template <typename V>
__global__ __launch_bounds__(TRP_BLOCK) void k_tr_bucket(int m, int n, int T, int tile,
                                                         int rows_per_block,
                                                         const int64_t* __restrict__ rowptr,
                                                         const int* __restrict__ col,
                                                         const V* __restrict__ val,
                                                         const uint32_t* __restrict__ cnt,
                                                         const int64_t* __restrict__ tptr,
                                                         TrPair<V>* __restrict__ out) {
  extern __shared__ unsigned tr_cur[];          // next position of the tile's buckets
  __shared__ int64_t s_lo[TRP_BLOCK];
  __shared__ int s_n[TRP_BLOCK];
  const int t = blockIdx.x % T;
  const long long blk = blockIdx.x / T;
  const int c0 = t * tile, c1 = min(n, c0 + tile);   // tile: whole buckets
  const int b0 = c0 / TR_BUCKET, nb = (c1 - c0 + TR_BUCKET - 1) / TR_BUCKET;
  for (int i = threadIdx.x; i < nb; i += TRP_BLOCK)
    tr_cur[i] = (unsigned)tr_bucket_start(n, blk, b0 + i, cnt, tptr);
  const int lane = lane_id();
  const long long r0 = blk * rows_per_block, r1 = min((long long)m, r0 + rows_per_block);
  // one entry per thread: runs of one bucket take their places together
  auto place = [&](bool in, int c, V v, int r) {
    const int b = in ? (c >> TR_BITS) - b0 : -1;
    const int left = __shfl_up(b, 1, WAVE);
    const bool head = in && (lane == 0 || left != b);
    const unsigned long long heads = __ballot(head), live = __ballot(in);
    if (live == 0) return;
    // the run's head, its length, and the own place in it (lanes in use come first)
    const unsigned long long below = heads & (~0ull >> (63 - lane));
    const int h = 63 - __clzll((long long)(below | 1ull));
    const unsigned long long above = lane == 63 ? 0ull : heads >> (lane + 1);
    unsigned base = 0;
    if (head) {
      const int next = above ? lane + __ffsll((long long)above) : __popcll(live);
      base = atomicAdd(&tr_cur[b], (unsigned)(next - lane));
    }
    base = __shfl(base, h, WAVE);
    if (in) out[(long long)base + (lane - h)] = TrPair<V>{(unsigned)r * TR_BUCKET + (c & (TR_BUCKET - 1)), v};
  };
  for (long long rb = r0; rb < r1; rb += TRP_BLOCK) {
    __syncthreads();
    tr_bounds(rowptr, col, rb + threadIdx.x, r1, c0, c1, s_lo, s_n);
    __syncthreads();
    const int nr = (int)min((long long)TRP_BLOCK, r1 - rb);
    int cn[TR_AHEAD];
    V vn[TR_AHEAD];
    auto request = [&](int i0) {
#pragma unroll
      for (int j = 0; j < TR_AHEAD; j++) {
        cn[j] = -1;
        if (i0 + j < nr && (int)threadIdx.x < s_n[i0 + j]) {
          cn[j] = col[s_lo[i0 + j] + threadIdx.x];
          vn[j] = val[s_lo[i0 + j] + threadIdx.x];
        }
      }
    };
    request(0);
    for (int i0 = 0; i0 < nr; i0 += TR_AHEAD) {
      int c[TR_AHEAD];
      V v[TR_AHEAD];
#pragma unroll
      for (int j = 0; j < TR_AHEAD; j++) {
        c[j] = cn[j];
        v[j] = vn[j];
      }
      request(i0 + TR_AHEAD);
#pragma unroll
      for (int j = 0; j < TR_AHEAD; j++) {
        if (i0 + j >= nr) break;
        const int r = (int)(rb + i0 + j), len = s_n[i0 + j];
        place(c[j] >= 0, c[j], v[j], r);
        for (int k = threadIdx.x + TRP_BLOCK; k - (int)threadIdx.x < len; k += TRP_BLOCK) {
          const bool in = k < len;
          place(in, in ? col[s_lo[i0 + j] + k] : -1, in ? val[s_lo[i0 + j] + k] : V(0), r);
        }
        // the next row's places come after this row's: wait for LDS alone
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    }
  }
}

// Workgroup = bucket, each wavefront a part of the row blocks: entries in order to
// their places, in LDS where the bucket fits (then the result is written in whole
// lines), else in memory.
constexpr int TR_WAVES = 4;
constexpr int TR_ROOM = 6144;    // entries of a bucket in LDS
template <typename V>
__global__ __launch_bounds__(TR_WAVES * WAVE) void k_tr_place(int n, int B,
                                                              const uint32_t* __restrict__ cnt,
                                                              const int64_t* __restrict__ tptr,
                                                              const TrPair<V>* __restrict__ in,
                                                              int* __restrict__ orow,
                                                              V* __restrict__ oval) {
  __shared__ int s_row[TR_ROOM];
  __shared__ V s_val[TR_ROOM];
  const int lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const long long c0 = (long long)blockIdx.x * TR_BUCKET;
  const long long first = tptr[c0], size = tptr[min((long long)n, c0 + TR_BUCKET)] - first;
  const bool fits = size <= TR_ROOM;
  const long long blk0 = (long long)B * w / TR_WAVES, blk1 = (long long)B * (w + 1) / TR_WAVES;
  const long long c = c0 + (lane & (TR_BUCKET - 1));
  // this lane's column: its next position in the bucket
  long long next = 0, a = 0, z = 0;
  if (c < n) {
    const long long p = tptr[c];
    a = blk0 < B ? cnt[blk0 * n + c] : tptr[c + 1] - p;
    z = blk1 < B ? cnt[blk1 * n + c] : tptr[c + 1] - p;
    next = p - first + a;
  }
  // the part's entries: from all columns' entries before it to those before its end
#pragma unroll
  for (int off = TR_BUCKET / 2; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, WAVE);
    z += __shfl_xor(z, off, WAVE);
  }
  const long long e0 = first + a, e1 = first + z;
  TrPair<V> q = e0 + lane < e1 ? in[e0 + lane] : TrPair<V>{0u, V(0)};
  for (long long k = e0; k < e1; k += WAVE) {
    const TrPair<V> p = q;
    const bool live = k + lane < e1;
    const long long kn = min(k + WAVE + lane, e1 - 1);
    q = in[kn];                               // the next 64, requested before these are placed
    const unsigned cl = p.key & (TR_BUCKET - 1);
    unsigned long long same = __ballot(live), own = same;
#pragma unroll
    for (int b = 0; b < TR_BITS; b++) {
      const unsigned long long bit = __ballot((cl >> b) & 1u);
      same &= (cl >> b) & 1u ? bit : ~bit;
      own &= (lane >> b) & 1 ? bit : ~bit;
    }
    const long long at = __shfl(next, (int)cl, WAVE) + __popcll(same & ((1ull << lane) - 1ull));
    if (live) {
      const int r = (int)(p.key >> TR_BITS);
      if (fits) {
        s_row[at] = r;
        s_val[at] = p.val;
      } else {
        orow[first + at] = r;
        oval[first + at] = p.val;
      }
    }
    next += __popcll(own);
  }
  __syncthreads();
  if (fits)
    for (int i = threadIdx.x; i < (int)size; i += TR_WAVES * WAVE) {
      orow[first + i] = s_row[i];
      oval[first + i] = s_val[i];
    }
}

// Places the entries by buckets; *done = false where that does not apply: rows too
// short to occupy a workgroup (57 entries: no gain), keys beyond 32 bits, counters
// beyond LDS, pairs of more than TR_PAIR_BYTES, or no memory for them.
template <typename V>
static int tr_by_buckets(epet_ctx* ctx, const epet_matrix* A, int rpb, int B, const uint32_t* cnt,
                         const int64_t* tptr, int* orow, void* oval, bool* done) {
  *done = false;
  const int nbuckets = (int)(((long long)A->n + TR_BUCKET - 1) / TR_BUCKET);
  if (A->nnz < 128ll * A->m || A->m >= (1 << (32 - TR_BITS))) return EPET_OK;
  const int per_wg = 48 * 1024 / (int)sizeof(unsigned);
  // two workgroups per CU (one to eight made no difference)
  const int fit = (nbuckets + per_wg - 1) / per_wg;
  int T = std::max(fit, std::min(16, std::max(1, 512 / B)));
  if (fit > 16) return EPET_OK;
  const int tile = (nbuckets + T - 1) / T * TR_BUCKET;
  T = (A->n + tile - 1) / tile;
  hipStream_t st = ctx->stream;
  // A block that is kept for the next matrix once freed (0.7 GB from the pool of
  // temporaries, beyond what that kept, took 35 ms longer a reconstruction).
  const size_t bytes = sizeof(TrPair<V>) * (size_t)A->nnz;
  if (bytes > TR_PAIR_BYTES) return EPET_OK;
  struct Block {
    void* p = nullptr;
    ~Block() { (void)dev_free(p); }            // waits for the device
  } block;
  if (dev_malloc(&block.p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return EPET_OK;
  }
  TrPair<V>* pairs = (TrPair<V>*)block.p;
  k_tr_bucket<V><<<(unsigned)(B * T), TRP_BLOCK, sizeof(unsigned) * (size_t)(tile / TR_BUCKET), st>>>(
      A->m, A->n, T, tile, rpb, A->rowptr, A->col, (const V*)A->val, cnt, tptr, pairs);
  k_tr_place<V><<<(unsigned)nbuckets, TR_WAVES * WAVE, 0, st>>>(A->n, B, cnt, tptr, pairs, orow,
                                                                (V*)oval);
  EPET_HIP(hipGetLastError());
  *done = true;
  return EPET_OK;
}

template <typename V, typename P>
static void launch_tr_fill(hipStream_t st, int grid, int m, int n, int T, int tile, int rpb,
                           const int64_t* rowptr, const int* col, const void* val,
                           const uint32_t* cnt, const int64_t* tptr, int* orow, void* oval) {
  const size_t lds = sizeof(P) * (size_t)std::min(n, tile);
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)k_tr_fill<V, P>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, TR_LDS);
  k_tr_fill<V, P><<<grid, TR_BLOCK, lds, st>>>(m, n, T, tile, rpb, rowptr, col, (const V*)val, cnt,
                                               tptr, orow, (V*)oval);
}
}  // namespace epet

epet_matrix::~epet_matrix() {
  if (bp_toff) (void)dev_free(bp_toff);
  if (bp_partial) (void)dev_free(bp_partial);
  if (xb_toff) (void)dev_free(xb_toff);
  if (xb_partial) (void)dev_free(xb_partial);
  if (lds_off) (void)dev_free(lds_off);
  if (lds_val) (void)dev_free(lds_val);
  if (lds_col16) (void)dev_free(lds_col16);
  if (lds_plan) (void)dev_free(lds_plan);
  if (lds_partial) (void)dev_free(lds_partial);
  epet::blk_release(this);
  epet::brk_release(this);
  if (tr) epet_matrix_destroy(tr);
}

namespace epet {
void xb_prepare(epet_ctx* ctx, epet_matrix* At);
int matrix_alloc(epet_matrix** out, int m, int n, long long nnz, int value_type) {
  epet_matrix* A = new epet_matrix();
  A->m = m;
  A->n = n;
  A->nnz = nnz;
  A->value_type = value_type;
  const size_t vb = value_type == EPET_VAL_F32 ? 4 : 2;
  bool ok = dev_malloc((void**)&A->rowptr, sizeof(int64_t) * ((size_t)m + 1)) == hipSuccess &&
            dev_malloc((void**)&A->col, sizeof(int) * (size_t)std::max(1ll, nnz)) == hipSuccess &&
            dev_malloc((void**)&A->val, vb * (size_t)std::max(1ll, nnz)) == hipSuccess;
  if (ok && value_type != EPET_VAL_F32)
    ok = dev_malloc((void**)&A->rowscale, sizeof(float) * (size_t)std::max(1, m)) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    if (A->rowptr) (void)dev_free(A->rowptr);
    if (A->col) (void)dev_free(A->col);
    if (A->val) (void)dev_free(A->val);
    delete A;
    EPET_FAIL(EPET_ERR_ALLOC, "matrix allocation (" + std::to_string(nnz) + " entries) failed");
  }
  (void)hipGetDevice(&A->device);
  *out = A;
  return EPET_OK;
}
}  // namespace epet

extern "C" {

int epet_cooSort(epet_ctx* ctx, float* val, int* row, int* col, long long N) {
  EPET_CHECK(ctx && (N == 0 || (val && row && col)), EPET_ERR_ARG, "null argument");
  EPET_CHECK(N >= 0, EPET_ERR_ARG, "negative length");
  if (N <= 1) return EPET_OK;
  const long long ntiles = (N + RS_TILE - 1) / RS_TILE;
  EPET_CHECK(ntiles * RS_BINS < (1ll << 31), EPET_ERR_UNSUPPORTED, "cooSort input too long");
  uint64_t *k0 = nullptr, *k1 = nullptr;
  float* v1 = nullptr;
  int* hist = nullptr;
  int64_t* offs = nullptr;
  unsigned long long* scan = nullptr;
  hipStream_t st = ctx->stream;
  StreamTemps tmp(st);
  EPET_HIP(tmp.alloc(&scan, sizeof(unsigned long long) * 3));
  k_init_scan<<<1, 64, 0, st>>>(scan);
  k_coo_scan<<<grid_for((N + 3) / 4, SCAN_BLOCK, 2ll * ctx->num_cus), SCAN_BLOCK, 0, st>>>(row, col, N, scan);
  EPET_HIP(hipGetLastError());
  unsigned long long ao[3];
  EPET_TRY(read_pinned(ctx, ao, scan, sizeof(ao)));
  // in order already (a generated matrix comes row by row, voxels ascending):
  // the stable sort leaves every entry where it is
  if (!ao[2]) return EPET_OK;
  EPET_HIP(tmp.alloc(&k0, sizeof(uint64_t) * N));
  EPET_HIP(tmp.alloc(&k1, sizeof(uint64_t) * N));
  EPET_HIP(tmp.alloc(&v1, sizeof(float) * N));
  EPET_HIP(tmp.alloc(&hist, sizeof(int) * ntiles * RS_BINS));
  EPET_HIP(tmp.alloc(&offs, sizeof(int64_t) * (ntiles * RS_BINS + 1)));
  const unsigned g = grid_for(N, 256, 1ll << 31);
  k_pack_keys<<<g, 256, 0, st>>>(row, col, N, k0);
  EPET_HIP(hipGetLastError());
  const uint64_t vary = ao[0] ^ ao[1];
  uint64_t* kin = k0;
  uint64_t* kout = k1;
  float* vin = val;
  float* vout = v1;
  int rc = EPET_OK;
  for (int shift = 0; shift < 64 && rc == EPET_OK; shift += 8) {
    if (((vary >> shift) & 0xFF) == 0) continue;
    k_rs_hist<<<(unsigned)ntiles, RS_BLOCK, 0, st>>>(kin, N, shift, (int)ntiles, hist);
    EPET_HIP(hipGetLastError());
    rc = exclusive_scan_i32_to_i64(ctx, hist, offs, ntiles * RS_BINS, nullptr);
    k_rs_scatter<<<(unsigned)ntiles, RS_BLOCK, 0, st>>>(kin, vin, N, shift, (int)ntiles, offs,
                                                        kout, vout);
    EPET_HIP(hipGetLastError());
    std::swap(kin, kout);
    std::swap(vin, vout);
  }
  if (vin != val) EPET_HIP(hipMemcpyAsync(val, vin, sizeof(float) * N, hipMemcpyDeviceToDevice, st));
  k_unpack_keys<<<g, 256, 0, st>>>(kin, N, row, col);
  EPET_HIP(hipGetLastError());
  return rc;
}

int epet_convertCoo2Csr(epet_ctx* ctx, int* csrRowPtr, const int* cooRowId, long long nnz, int m) {
  EPET_CHECK(ctx && csrRowPtr && (nnz == 0 || cooRowId), EPET_ERR_ARG, "null argument");
  EPET_CHECK(m >= 0 && nnz >= 0 && nnz < (1ll << 31), EPET_ERR_ARG, "bad sizes");
  hipStream_t st = ctx->stream;
  StreamTemps tmp(st);
  int* bad = nullptr;
  EPET_HIP(tmp.alloc(&bad, sizeof(int)));
  k_fill_i32<<<1, 64, 0, st>>>(bad, 1, 0);
  k_fill_i32<<<grid_for(m + 1, 256, 1ll << 31), 256, 0, st>>>(csrRowPtr, m + 1, 0);
  if (nnz > 0)
    k_row_hist<<<grid_for((nnz + HIST_SPAN - 1) / HIST_SPAN, 256 / WAVE, 16ll * ctx->num_cus), 256, 0,
                 st>>>(cooRowId, nnz, m, csrRowPtr, bad);
  EPET_HIP(hipGetLastError());
  EPET_TRY(exclusive_scan_i32(ctx, csrRowPtr, csrRowPtr, (long long)m + 1, nullptr));
  int hbad = 0;
  EPET_TRY(read_pinned(ctx, &hbad, bad, sizeof(int)));
  EPET_CHECK(!hbad, EPET_ERR_ARG, "COO row id outside [0, m)");
  return EPET_OK;
}

int epet_convertCsr2Ecsr(epet_ctx* ctx, int* ecsr, const int* yRowId, int nnzr, const int* csr,
                         int m) {
  EPET_CHECK(ctx && ecsr && csr && (nnzr == 0 || yRowId), EPET_ERR_ARG, "null argument");
  EPET_CHECK(nnzr >= 0 && m >= 0, EPET_ERR_ARG, "bad sizes");
  k_csr2ecsr<<<grid_for((long long)nnzr + 1, 256, 1ll << 31), 256, 0, ctx->stream>>>(ecsr, yRowId,
                                                                                  nnzr, csr, m);
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

int epet_matrix_info(const epet_matrix* A, int* m, int* n, long long* nnz, int* value_type) {
  EPET_CHECK(A, EPET_ERR_ARG, "null matrix");
  if (m) *m = A->m;
  if (n) *n = A->n;
  if (nnz) *nnz = A->nnz;
  if (value_type) *value_type = A->value_type;
  return EPET_OK;
}

int epet_matrix_arrays(const epet_matrix* A, int64_t** rowptr, int** col, void** val,
                       float** rowscale) {
  EPET_CHECK(A, EPET_ERR_ARG, "null matrix");
  if (rowptr) *rowptr = A->rowptr;
  if (col) *col = A->col;
  if (val) *val = A->val;
  if (rowscale) *rowscale = A->rowscale;
  const_cast<epet_matrix*>(A)->exposed.store(true);
  return EPET_OK;
}

int epet_matrix_read(epet_ctx* ctx, const epet_matrix* A, int64_t* rowptr, int* col, void* val,
                     float* rowscale) {
  EPET_CHECK(ctx && A, EPET_ERR_ARG, "null argument");
  hipStream_t st = ctx->stream;
  const size_t vb = A->value_type == EPET_VAL_F32 ? 4 : 2;
  if (rowptr)
    EPET_HIP(hipMemcpyAsync(rowptr, A->rowptr, sizeof(int64_t) * ((size_t)A->m + 1),
                            hipMemcpyDeviceToDevice, st));
  if (col && A->nnz)
    EPET_HIP(hipMemcpyAsync(col, A->col, sizeof(int) * A->nnz, hipMemcpyDeviceToDevice, st));
  if (val && A->nnz) EPET_HIP(hipMemcpyAsync(val, A->val, vb * A->nnz, hipMemcpyDeviceToDevice, st));
  if (rowscale && A->rowscale && A->m)
    EPET_HIP(hipMemcpyAsync(rowscale, A->rowscale, sizeof(float) * A->m, hipMemcpyDeviceToDevice, st));
  return EPET_OK;
}

int epet_matrix_destroy(epet_matrix* A) {
  if (!A) return EPET_OK;
  (void)hipDeviceSynchronize();
  if (A->owns) {
    if (A->rowptr) (void)dev_free(A->rowptr);
    if (A->col) (void)dev_free(A->col);
    if (A->val) (void)dev_free(A->val);
    if (A->rowscale) (void)dev_free(A->rowscale);
    if (A->row_ids) (void)dev_free(A->row_ids);
  }
  delete A;
  return EPET_OK;
}

int epet_matrix_create(epet_ctx* ctx, int m, int n, long long nnz, const int64_t* rowptr,
                       const int* col, const float* val, epet_matrix** out) {
  EPET_CHECK(ctx && out && rowptr && (nnz == 0 || (col && val)), EPET_ERR_ARG, "null argument");
  EPET_CHECK(m >= 0 && n >= 0 && nnz >= 0, EPET_ERR_ARG, "bad sizes");
  hipStream_t st = ctx->stream;
  int hflags = 0;
  if (m > 0) {
    StreamTemps tmp(st);
    int* flags = nullptr;
    EPET_HIP(tmp.alloc(&flags, sizeof(int)));
    k_fill_i32<<<1, 64, 0, st>>>(flags, 1, 0);
    k_check_csr<<<grid_for(m, 256, 1ll << 31), 256, 0, st>>>(m, n, nnz, rowptr, col, flags);
    EPET_HIP(hipGetLastError());
    EPET_TRY(read_pinned(ctx, &hflags, flags, sizeof(int)));
    EPET_CHECK(!(hflags & 1), EPET_ERR_ARG,
               "invalid CSR arrays (row pointers or column ids out of range)");
  }
  epet_matrix* A = nullptr;
  EPET_TRY(matrix_alloc(&A, m, n, nnz, EPET_VAL_F32));
  MatrixGuard keep(A);
  // the tiled back projection needs ascending columns within rows
  if (hflags & 2) { A->bp_failed = true; A->cols_strict = false; }
  EPET_HIP(hipMemcpyAsync(A->rowptr, rowptr, sizeof(int64_t) * ((size_t)m + 1),
                          hipMemcpyDeviceToDevice, st));
  if (nnz) {
    EPET_HIP(hipMemcpyAsync(A->col, col, sizeof(int) * nnz, hipMemcpyDeviceToDevice, st));
    EPET_HIP(hipMemcpyAsync(A->val, val, sizeof(float) * nnz, hipMemcpyDeviceToDevice, st));
  }
  EPET_HIP(hipStreamSynchronize(st));
  *out = keep.release();
  return EPET_OK;
}

int epet_matrix_select_rows(epet_ctx* ctx, const epet_matrix* A, const int* rows, int nrows,
                            epet_matrix** out) {
  EPET_CHECK(ctx && A && out && (nrows == 0 || rows), EPET_ERR_ARG, "null argument");
  EPET_CHECK(nrows >= 0, EPET_ERR_ARG, "negative row count");
  hipStream_t st = ctx->stream;
  StreamTemps tmp(st);
  int* cnt = nullptr;
  int64_t* off = nullptr;
  int* bad = nullptr;
  EPET_HIP(tmp.alloc(&cnt, sizeof(int) * std::max(1, nrows)));
  EPET_HIP(tmp.alloc(&off, sizeof(int64_t) * ((size_t)nrows + 1)));
  EPET_HIP(tmp.alloc(&bad, sizeof(int)));
  k_fill_i32<<<1, 64, 0, st>>>(bad, 1, 0);
  if (nrows)
    k_sel_counts<<<grid_for(nrows, 256, 1ll << 31), 256, 0, st>>>(A->rowptr, rows, nrows, A->m,
                                                                  cnt, bad);
  EPET_HIP(hipGetLastError());
  int hbad = 0;
  EPET_TRY(read_pinned(ctx, &hbad, bad, sizeof(int)));
  EPET_CHECK(!hbad, EPET_ERR_ARG, "row index out of range");
  long long nnz = 0;
  EPET_TRY(exclusive_scan_i32_to_i64(ctx, cnt, off, nrows, &nnz));
  epet_matrix* B = nullptr;
  EPET_TRY(matrix_alloc(&B, nrows, A->n, nnz, A->value_type));
  MatrixGuard keep(B);
  if (nrows) {
    if (A->value_type == EPET_VAL_F32)
      k_sel_copy<float><<<nrows, 256, 0, st>>>(A->rowptr, A->col, (const float*)A->val,
                                               A->rowscale, rows, A->m, off, B->rowptr, B->col,
                                               (float*)B->val, B->rowscale);
    else
      k_sel_copy<uint16_t><<<nrows, 256, 0, st>>>(A->rowptr, A->col, (const uint16_t*)A->val,
                                                  A->rowscale, rows, A->m, off, B->rowptr,
                                                  B->col, (uint16_t*)B->val, B->rowscale);
    EPET_HIP(hipGetLastError());
  }
  if (A->row_ids) {
    if (dev_malloc((void**)&B->row_ids, sizeof(int) * (size_t)std::max(1, nrows)) != hipSuccess) {
      (void)hipGetLastError();
      B->row_ids = nullptr;
    } else if (nrows) {
      k_gather_i32<<<grid_for(nrows, 256, 1ll << 31), 256, 0, st>>>(A->row_ids, rows, nrows,
                                                                    B->row_ids);
      EPET_HIP(hipGetLastError());
    }
    if (B->row_ids) B->mg = A->mg;
  }
  // last row pointer = nnz
  {
    int64_t h = nnz;
    EPET_HIP(hipMemcpyAsync(B->rowptr + nrows, &h, sizeof(int64_t), hipMemcpyHostToDevice, st));
    EPET_HIP(hipStreamSynchronize(st));
  }
  *out = keep.release();
  return EPET_OK;
}

int epet_matrix_convert(epet_ctx* ctx, const epet_matrix* A, int vt, epet_matrix** out) {
  EPET_CHECK(ctx && A && out, EPET_ERR_ARG, "null argument");
  EPET_CHECK(A->value_type == EPET_VAL_F32, EPET_ERR_STATE, "conversion source must be FP32");
  EPET_CHECK(vt == EPET_VAL_BF16 || vt == EPET_VAL_F16 || vt == EPET_VAL_F32, EPET_ERR_ARG,
             "unknown value type");
  hipStream_t st = ctx->stream;
  epet_matrix* B = nullptr;
  EPET_TRY(matrix_alloc(&B, A->m, A->n, A->nnz, vt));
  MatrixGuard keep(B);
  EPET_HIP(hipMemcpyAsync(B->rowptr, A->rowptr, sizeof(int64_t) * ((size_t)A->m + 1),
                          hipMemcpyDeviceToDevice, st));
  if (A->nnz) EPET_HIP(hipMemcpyAsync(B->col, A->col, sizeof(int) * A->nnz, hipMemcpyDeviceToDevice, st));
  if (vt == EPET_VAL_F32) {
    if (A->nnz)
      EPET_HIP(hipMemcpyAsync(B->val, A->val, sizeof(float) * A->nnz, hipMemcpyDeviceToDevice, st));
  } else if (A->m) {
    k_convert_rows<<<A->m, 256, 0, st>>>(A->rowptr, (const float*)A->val, vt,
                                         (uint16_t*)B->val, B->rowscale);
    EPET_HIP(hipGetLastError());
  }
  if (A->row_ids && dev_malloc((void**)&B->row_ids, sizeof(int) * (size_t)std::max(1, A->m)) ==
                        hipSuccess) {
    if (A->m)
      EPET_HIP(hipMemcpyAsync(B->row_ids, A->row_ids, sizeof(int) * A->m, hipMemcpyDeviceToDevice,
                              st));
    B->mg = A->mg;
  } else {
    (void)hipGetLastError();
  }
  EPET_HIP(hipStreamSynchronize(st));
  *out = keep.release();
  return EPET_OK;
}

int epet_matrix_colsum_f64(epet_ctx* ctx, const epet_matrix* A, double* s) {
  EPET_CHECK(ctx && A && s, EPET_ERR_ARG, "null argument");
  hipStream_t st = ctx->stream;
  k_fill_f64<<<grid_for(A->n, 256, 1ll << 31), 256, 0, st>>>(s, A->n);
  // sums in LDS where a column has entries enough to make up for adding it to memory
  // once per row block (3 a column: 14.0 us against 9.9; 13: 120 against 202; 125: 18
  // against 50)
  if (A->m > 0 && A->n > 0 && A->cols_strict && A->nnz >= 8ll * A->n) {
    switch (A->value_type) {
      case EPET_VAL_F32: return launch_colsum_tiles<ValF32>(ctx, A, s);
      case EPET_VAL_BF16: return launch_colsum_tiles<ValBF16>(ctx, A, s);
      default: return launch_colsum_tiles<ValF16>(ctx, A, s);
    }
  }
  if (A->m)
    k_colsum_f64<<<A->m, 256, 0, st>>>(A->rowptr, A->col, A->val, A->value_type, A->rowscale,
                                       A->m, s);
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

int epet_matrix_transpose(epet_ctx* ctx, epet_matrix* A) {
  EPET_CHECK(ctx && A, EPET_ERR_ARG, "null argument");
  if (A->tr) return EPET_OK;
  EPET_CHECK(A->cols_strict, EPET_ERR_STATE,
             "transpose needs strictly ascending columns within every row");
  hipStream_t st = ctx->stream;
  // counters of a tile: 32-bit positions up to 2^32 entries, 64-bit above
  const bool wide = A->nnz > 0xFFFFFFFFll;
  const int tile = TR_LDS / (wide ? 8 : 4);
  const int nt = std::max(1, (A->n + tile - 1) / tile);
  const int want = std::max(1, TR_GRID / nt);
  const int rpb = std::max(16, (A->m + want - 1) / want);
  const int B = (A->m + rpb - 1) / rpb;
  const long long ncnt = (long long)A->n * B;
  StreamTemps tmp(st);
  uint32_t* cnt = nullptr;
  int* total = nullptr;
  EPET_HIP(tmp.alloc(&cnt, sizeof(uint32_t) * std::max(1ll, ncnt)));
  EPET_HIP(tmp.alloc(&total, sizeof(int) * std::max(1, A->n)));
  const bool any = A->m > 0 && A->n > 0;
  if (any) {
    const size_t lds = sizeof(uint32_t) * (size_t)std::min(A->n, tile);
    if (lds > 64 * 1024)
      (void)hipFuncSetAttribute((const void*)k_tr_count,
                                hipFuncAttributeMaxDynamicSharedMemorySize, TR_LDS);
    k_tr_count<<<B * nt, TR_BLOCK, lds, st>>>(A->m, A->n, nt, tile, rpb, A->rowptr, A->col, cnt);
  }
  if (A->n) k_tr_prefix<<<grid_for(A->n, 256, 1ll << 31), 256, 0, st>>>(A->n, B, cnt, total);
  EPET_HIP(hipGetLastError());
  epet_matrix* T = nullptr;
  EPET_TRY(matrix_alloc(&T, A->n, A->m, A->nnz, A->value_type));
  MatrixGuard keep(T);
  if (T->rowscale) { (void)dev_free(T->rowscale); T->rowscale = nullptr; }
  long long tot = 0;
  EPET_TRY(exclusive_scan_i32_to_i64(ctx, total, T->rowptr, A->n, &tot));
  EPET_CHECK(tot == A->nnz, EPET_ERR_STATE, "transpose count mismatch");
  k_set_last_i64<<<1, 64, 0, st>>>(T->rowptr + A->n, (int64_t)A->nnz);
  if (any) {
    const int g = B * nt;
    bool done = false;
    // (pairs of at most TR_PAIR_BYTES: positions of 32 bits)
    if (A->value_type == EPET_VAL_F32)
      EPET_TRY((tr_by_buckets<float>(ctx, A, rpb, B, cnt, T->rowptr, T->col, T->val, &done)));
    else
      EPET_TRY((tr_by_buckets<uint16_t>(ctx, A, rpb, B, cnt, T->rowptr, T->col, T->val, &done)));
    if (!done && A->value_type == EPET_VAL_F32) {
      if (wide)
        launch_tr_fill<float, uint64_t>(st, g, A->m, A->n, nt, tile, rpb, A->rowptr, A->col, A->val,
                                        cnt, T->rowptr, T->col, T->val);
      else
        launch_tr_fill<float, uint32_t>(st, g, A->m, A->n, nt, tile, rpb, A->rowptr, A->col, A->val,
                                        cnt, T->rowptr, T->col, T->val);
    } else if (!done) {
      if (wide)
        launch_tr_fill<uint16_t, uint64_t>(st, g, A->m, A->n, nt, tile, rpb, A->rowptr, A->col,
                                           A->val, cnt, T->rowptr, T->col, T->val);
      else
        launch_tr_fill<uint16_t, uint32_t>(st, g, A->m, A->n, nt, tile, rpb, A->rowptr, A->col,
                                           A->val, cnt, T->rowptr, T->col, T->val);
    }
  }
  EPET_HIP(hipGetLastError());
  EPET_HIP(hipStreamSynchronize(st));
  T->bp_failed = true;
  xb_prepare(ctx, T);   // optional: without a plan the plain row kernel runs
  A->tr = keep.release();
  return EPET_OK;
}

}  // extern "C"
