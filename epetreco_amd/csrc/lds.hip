// lds.hip -- LDS-tiled row products y = A x (and, over a transposed copy, the
// back projection).
//
// The gathered vector x (n entries) is cut into tiles of LDS_TILE entries.  A
// workgroup of 1024 threads copies one tile into LDS and sums, for its rows, the
// entries whose column lies in that tile, with x read from LDS.  The row's
// partial for tile t goes to partial[t m + r]; a reduction sums the partials of
// every row in tile order (deterministic) and applies the row scale, alpha/beta
// or the MLEM ratio.  With a single tile the product is written at once.
//
// The kernels read a tile-major copy of the matrix built once per matrix: the
// entries of (tile t, row r) lie contiguously at lds_off[t m + r], rows of one
// tile back to back, columns stored tile-local in 16 bits, every segment padded
// to whole chunks of 8 entries.  So an FP32 entry costs 6 bytes, HBM sees the
// entry stream once, x once per workgroup, and 12 bytes of offset and partial per
// (row, tile).
//
// What bounds it is that stream, and keeping it in flight.  A wavefront therefore
// runs through its rows' chunks as one stream, 64 chunks (a block) at a time
// whatever the rows' lengths, three blocks requested ahead; a lane's chunk belongs
// to one row, and the lanes' sums are added up by row with a segmented scan.
// Before, R rows at a time had 64/R lanes each and one chunk per lane in flight:
// lanes idle at every row's end, and a wait per pass.  The rows are dealt out so
// that every wavefront has the same number of chunks (k_lds_plan).
// Forward / back projection, FP32, 52^3 voxels, before -> now:
//   1,100,000 rows, 979M entries   1163 -> 1055 / 1199 -> 1027 us (5.6 TB/s)
//   100,000 rows, 88M entries       141 ->  107 /  212 ->  106 us
//   11,250 rows, 4.6M entries        19 ->   11 us forward
// (a large tensor is read at 6.2 TB/s on the same card.)
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "epet_block.hpp"
#include "epet_internal.hpp"
#include "epet_rows.hpp"

namespace epet {

void launch_row_plan(hipStream_t st, int m, int T, int TS, const int64_t* rowptr, const int* col,
                     uint32_t* toff);

constexpr int LDS_BLOCK = 1024;
constexpr int LDS_WAVES = LDS_BLOCK / WAVE;
// blocks in flight per wavefront: 1 / 2 / 3 / 4 / 6 took 1131 / 1126 / 1126 / 1138 /
// 1139 us forward and 1247 / 1167 / 1155 / 1172 / 1175 us back at 979M entries
constexpr int LDS_DEPTH = 3;
// Workgroups: as many per CU as give every wavefront LDS_MIN_BLOCKS blocks, at most
// LDS_PER_CU.  More even out the card's unequal speeds, but each copies its 128 KB
// tile before its first product, and one workgroup's LDS fills a CU.  At 979M
// entries 8 / 16 / 32 / 64 per CU took 1122 / 1076 / 1055 / 1117 us forward; at
// 88M, 4 / 8 / 12 / 16 blocks at least took 137 / 113 / 109 / 107 us.
constexpr int LDS_MIN_BLOCKS = 16, LDS_PER_CU = 32;
// A row's own cost in chunks: rows with next to no entries in a tile still take
// their turn in a window of 64.  At 88M entries (the fifth tile nearly empty) 0 /
// 0.25 / 0.5 / 1 / 2 / 4 took 235 / 136 / 117 / 111 / 110 / 119 us forward.
constexpr int LDS_ROW_COST = 2;

// The values of a chunk of LDS_CHUNK entries of the tile-major copy (one or two
// 16-byte loads; its eight 16-bit columns are a third).
template <typename VT> struct LdsChunkRaw {
  uint4 a;
  __device__ __forceinline__ void load(const uint16_t* __restrict__ val, long long k) {
    a = *reinterpret_cast<const uint4*>(val + k);
  }
  __device__ __forceinline__ void get(float v[8]) const {
    const unsigned w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if constexpr (std::is_same<VT, ValBF16>::value) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
      } else {
        v[2 * i] = __half2float(__ushort_as_half((uint16_t)(w[i] & 0xFFFFu)));
        v[2 * i + 1] = __half2float(__ushort_as_half((uint16_t)(w[i] >> 16)));
      }
    }
  }
};
template <> struct LdsChunkRaw<ValF32> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* __restrict__ val, long long k) {
    a = *reinterpret_cast<const float4*>(val + k);
    b = *reinterpret_cast<const float4*>(val + k + 4);
  }
  __device__ __forceinline__ void get(float v[8]) const {
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
};

// Where a row's sum goes: its tile's partial, or with one tile the result.
struct LdsStore {
  int direct;
  const float* rowscale;
  float alpha, beta;
  __device__ __forceinline__ void store(float* __restrict__ out, int t, int m, long long r,
                                        float s) const {
    if (!direct) {
      out[(long long)t * m + r] = s;
      return;
    }
    const float v = alpha * (rowscale ? rowscale[r] : 1.0f) * s;
    out[r] = beta == 0.0f ? v : v + beta * out[r];
  }
};

// Lane l's value of the lane d below it in the same row of 16 (0 shifted in).
template <int D>
__device__ __forceinline__ float dpp_shr(float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x110 + D, 0xF, 0xF, true));
}

// Sums over the lanes of each segment up to and including the own lane: `before`
// is the number of lanes below the own one that belong to its segment.
__device__ __forceinline__ float segment_scan(float v, int before, int lane) {
  const int in16 = lane & 15, b16 = std::min(before, in16);
  float t;
  t = dpp_shr<1>(v);
  v += b16 >= 1 ? t : 0.0f;
  t = dpp_shr<2>(v);
  v += b16 >= 2 ? t : 0.0f;
  t = dpp_shr<4>(v);
  v += b16 >= 4 ? t : 0.0f;
  t = dpp_shr<8>(v);
  v += b16 >= 8 ? t : 0.0f;
  // carries across the rows of 16: each row's last lane into the next row
#pragma unroll
  for (int row = 1; row < 4; row++) {
    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16 * row - 1));
    if ((lane >> 4) == row && before > in16) v += c;
  }
  return v;
}

template <typename VT>
struct LdsBlock {
  uint4 c;
  LdsChunkRaw<VT> v;
};

// D blocks of 64 chunks in flight per wavefront; BWD = 1 marks the back
// projection over a transposed copy (a separate instantiation, so that profiles
// tell the two products apart).  out: the partials, or with T = 1 the result.
template <typename VT, int D, int BWD>
__global__ __launch_bounds__(LDS_BLOCK) void k_rows_lds(int m, int n, const int4* __restrict__ plan,
                                                        const int64_t* __restrict__ off,
                                                        const uint16_t* __restrict__ col,
                                                        const typename VT::T* __restrict__ val,
                                                        const float* __restrict__ x,
                                                        float* __restrict__ out, LdsStore ep,
                                                        ColMap mp) {
  extern __shared__ float xs[];
  const int lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  // this wavefront's rows [wa, wb) of tile t and their chunks [q, qe)
  const int4 unit = plan[(long long)blockIdx.x * LDS_WAVES + w];
  const int t = unit.z;
  if (t < 0) return;   // the whole workgroup
  const long long wa = unit.x, wb = unit.y;
  const long long tb = (long long)t * LDS_TILE;
  const int cnt = (int)std::min<long long>(LDS_TILE, (long long)n - tb);
  const int64_t* offt = off + (long long)t * m;
  long long q = offt[wa] / LDS_CHUNK;
  const long long qe = offt[wb] / LDS_CHUNK, qlast = std::max(0ll, qe - 1);
  auto load = [&](long long qb) {
    LdsBlock<VT> b;
    const long long k = std::min(qb + lane, qlast) * LDS_CHUNK;   // past the end: not used
    b.c = *reinterpret_cast<const uint4*>(col + k);
    b.v.load(val, k);
    return b;
  };
  LdsBlock<VT> buf[D];
#pragma unroll
  for (int j = 0; j < D; j++) buf[j] = load(q + (long long)j * WAVE);
  // lane l owns row wr + l of the window: its chunks [s, e)
  long long wr = wa;
  auto bound = [&](long long r) { return offt[std::min(r, wb)] / LDS_CHUNK; };
  long long s = bound(wr + lane), e = bound(wr + lane + 1);
  long long ns = bound(wr + WAVE + lane), ne = bound(wr + WAVE + lane + 1);
  if (mp.nx == 0) {
    // tile copy: 16-byte loads when the tile start is 16-byte aligned
    const int c4 = ((reinterpret_cast<uintptr_t>(x + tb) & 15) == 0) ? (cnt >> 2) : 0;
    const float4* x4 = reinterpret_cast<const float4*>(x + tb);
    constexpr int N4 = LDS_TILE / 4 / LDS_BLOCK;
    if (c4 == N4 * LDS_BLOCK) {   // a whole tile: all its loads at once
      float4 r[N4];
#pragma unroll
      for (int i = 0; i < N4; i++) r[i] = x4[threadIdx.x + i * LDS_BLOCK];
#pragma unroll
      for (int i = 0; i < N4; i++) reinterpret_cast<float4*>(xs)[threadIdx.x + i * LDS_BLOCK] = r[i];
    } else {
#pragma unroll 4
      for (int i = threadIdx.x; i < c4; i += LDS_BLOCK) reinterpret_cast<float4*>(xs)[i] = x4[i];
    }
    for (int i = (c4 << 2) + threadIdx.x; i < cnt; i += LDS_BLOCK) xs[i] = x[tb + i];
  } else {
    // renumbered columns: tile entry i is column colmap_inv(tb + i) of x
    for (int i = threadIdx.x; i < cnt; i += LDS_BLOCK) xs[i] = x[colmap_inv(tb + i, mp)];
  }
  __syncthreads();
  if (wa >= wb) return;
  const unsigned last = (unsigned)(cnt - 1);
  float acc = 0.0f;
  for (;;) {
#pragma unroll
    for (int j = 0; j < D; j++) {
      const unsigned cw[4] = {buf[j].c.x, buf[j].c.y, buf[j].c.z, buf[j].c.w};
      float v[LDS_CHUNK];
      buf[j].v.get(v);
      float a = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        // the clamp keeps LDS reads in range whatever the data
        const unsigned lo = std::min(cw[i] & (i == 0 ? 0x7FFFu : 0xFFFFu), last);
        const unsigned hi = std::min(cw[i] >> 16, last);
        a += v[2 * i] * xs[lo];
        a += v[2 * i + 1] * xs[hi];
      }
      // lanes of the own segment below the own lane
      const unsigned long long heads = __ballot((cw[0] & 0x8000u) != 0);
      const unsigned long long below = heads & (~0ull >> (63 - lane));
      a = segment_scan(a, below ? lane - (63 - __clzll((long long)below)) : lane, lane);
      buf[j] = load(q + (long long)D * WAVE);
      const long long qn = q + WAVE;
      for (;;) {
        // the part of the own row in this block ends at lane min(e, qn) - 1 - q
        const int at = (int)(std::min(e, qn) - 1 - q);
        const float p = __shfl(a, at & (WAVE - 1), WAVE);
        if (s < qn && e > q && s < e) acc += p;
        if (lane_value_i64(e, WAVE - 1) > qn) break;   // the window goes on in the next block
        const long long r = wr + lane;
        if (r < wb) ep.store(out, t, m, r, acc);
        wr += WAVE;
        if (wr >= wb) return;
        acc = 0.0f;
        s = ns;
        e = ne;
        ns = bound(wr + WAVE + lane);
        ne = bound(wr + WAVE + lane + 1);
      }
      q = qn;
    }
  }
}

// ------------------------------------------------------------------ tile-major copy
// Stable counting sort of every row's entries by the voxel's y index (one
// wavefront per row, per-wave bucket counters in LDS): rows ascending in
// (ix, iy, iz) become ascending in (iy, ix, iz), i.e. in the y-major column
// colmap_fwd(c).  Writes the renumbered columns and the values in that order.
template <typename T>
__global__ __launch_bounds__(256) void k_ysort_rows(int m, const int64_t* __restrict__ rowptr,
                                                    const int* __restrict__ col,
                                                    const T* __restrict__ val, ColMap mp,
                                                    int* __restrict__ colp, T* __restrict__ valp) {
  extern __shared__ int bucket[];                 // (256 / WAVE) x ny
  const int lane = lane_id();
  const int w = wave_id();
  int* cnt = bucket + w * mp.ny;
  const long long nw = (long long)gridDim.x * (256 / WAVE);
  for (long long r = (long long)blockIdx.x * (256 / WAVE) + w; r < m; r += nw) {
    const long long b = rowptr[r], e = rowptr[r + 1];
    for (int i = lane; i < mp.ny; i += WAVE) cnt[i] = 0;
    __builtin_amdgcn_wave_barrier();
    for (long long k = b + lane; k < e; k += WAVE) atomicAdd(&cnt[(col[k] / mp.nz) % mp.ny], 1);
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
      int run = 0;
      for (int i = 0; i < mp.ny; i++) {
        const int c = cnt[i];
        cnt[i] = run;
        run += c;
      }
    }
    __builtin_amdgcn_wave_barrier();
    for (long long base = b; base < e; base += WAVE) {
      const long long k = base + lane;
      bool act = k < e;
      const int c = act ? col[k] : 0;
      const int iy = act ? (c / mp.nz) % mp.ny : -1;
      // lanes grouped by y, each group placed after the earlier entries of its
      // bucket in lane (= entry) order
      unsigned long long left = __ballot(act);
      while (left) {
        const int lead = __ffsll((long long)left) - 1;
        const int key = __shfl(iy, lead);
        const unsigned long long mask = __ballot(act && iy == key);
        const int start = cnt[key];
        if (act && iy == key) {
          const int rank = __popcll(mask & ((1ull << lane) - 1ull));
          colp[b + start + rank] = (int)colmap_fwd(c, mp);
          valp[b + start + rank] = val[k];
          act = false;
        }
        __builtin_amdgcn_wave_barrier();
        if (lane == lead) cnt[key] = start + __popcll(mask);
        __builtin_amdgcn_wave_barrier();
        left &= ~mask;
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// padded segment lengths: every (tile, row) segment is a whole number of
// LDS_CHUNK-entry chunks, so a lane reads a chunk's columns and values with
// 16-byte loads
__global__ __launch_bounds__(256) void k_lds_counts(int m, int T, const uint32_t* __restrict__ toff,
                                                    int* __restrict__ cnt) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;   // i = t m + r
  if (i >= (long long)m * T) return;
  const int t = (int)(i / m);
  const long long r = i % m;
  const uint32_t* o = toff + r * (T + 1) + t;
  cnt[i] = ((int)(o[1] - o[0]) + LDS_CHUNK - 1) & ~(LDS_CHUNK - 1);
}

__global__ void k_lds_set_last(int64_t* __restrict__ off, long long i, long long v) {
  if (threadIdx.x == 0 && blockIdx.x == 0) off[i] = v;
}

// Copies values and tile-local columns of every (tile, row) segment, then zero
// entries (the segment's last column, value 0) up to the padded length.  Bit 15 of a
// segment's first column marks it.  16 lanes take a segment, each a chunk of 8
// entries, whose 48 bytes (FP32) it writes with 16-byte stores.  Waits bound it: a
// wavefront per segment, an entry per lane, took 452 us for 88M entries of 100,000 rows
// in 5 tiles, this 347: 3.5 TB/s read and written.
constexpr int LDSF_LANES = 16;
template <typename T>
__global__ __launch_bounds__(256) void k_lds_fill(int m, int T_, int mask,
                                                  const int64_t* __restrict__ rowptr,
                                                  const uint32_t* __restrict__ toff,
                                                  const int* __restrict__ col,
                                                  const T* __restrict__ val,
                                                  const int64_t* __restrict__ off,
                                                  uint16_t* __restrict__ col16,
                                                  T* __restrict__ val2) {
  static_assert(LDS_CHUNK == 8, "a lane writes eight entries");
  // entries may start at any element
  typedef int Cols __attribute__((ext_vector_type(4), aligned(4)));
  typedef T Vals __attribute__((ext_vector_type(8), aligned(sizeof(T))));
  typedef T Out __attribute__((ext_vector_type(8)));
  const int sub = threadIdx.x % LDSF_LANES;
  const long long nw = (long long)gridDim.x * (256 / LDSF_LANES);
  for (long long i = (long long)blockIdx.x * (256 / LDSF_LANES) + threadIdx.x / LDSF_LANES;
       i < (long long)m * T_; i += nw) {
    const int t = (int)(i / m);
    const long long r = i % m;
    const uint32_t* o = toff + r * (T_ + 1) + t;
    const long long src = rowptr[r] + o[0];
    const long long len = o[1] - o[0];
    const long long dst = off[i], plen = off[i + 1] - dst;
    for (long long k = sub * LDS_CHUNK; k < plen; k += LDSF_LANES * LDS_CHUNK) {
      unsigned c[8];
      Out v;
      if (k + LDS_CHUNK <= len) {
        const Cols c0 = *reinterpret_cast<const Cols*>(col + src + k);
        const Cols c1 = *reinterpret_cast<const Cols*>(col + src + k + 4);
        v = *reinterpret_cast<const Vals*>(val + src + k);
#pragma unroll
        for (int j = 0; j < 4; j++) {
          c[j] = (unsigned)(c0[j] & mask);
          c[4 + j] = (unsigned)(c1[j] & mask);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const bool in = k + j < len;
          c[j] = (unsigned)(col[src + (in ? k + j : len - 1)] & mask);
          v[j] = in ? val[src + k + j] : (T)0;
        }
      }
      if (k == 0) c[0] |= 0x8000u;
      *reinterpret_cast<uint4*>(col16 + dst + k) =
          make_uint4(c[0] | c[1] << 16, c[2] | c[3] << 16, c[4] | c[5] << 16, c[6] | c[7] << 16);
      *reinterpret_cast<Out*>(val2 + dst + k) = v;
    }
  }
}

// ------------------------------------------------------------------ work split
// Unit u = 16 wg + w: the rows (x, y) of tile z that wavefront w of workgroup wg
// sums.  Tile t has max(1, ceil(cost / target)) workgroups, cost = chunks +
// LDS_ROW_COST rows, and its cost is cut evenly over their wavefronts, each row
// going to the wavefront its first chunk falls to; z = -1 past the last tile's
// workgroups.
__global__ __launch_bounds__(256) void k_lds_plan(int m, int T, long long target, long long nunits,
                                                  const int64_t* __restrict__ off,
                                                  int4* __restrict__ plan) {
  const long long u = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= nunits) return;
  long long wg = u / LDS_WAVES;
  int t = 0;
  long long c0 = 0, chunks = 0, wgs = 0;
  for (; t < T; t++) {
    c0 = off[(long long)t * m] / LDS_CHUNK;
    chunks = off[(long long)(t + 1) * m] / LDS_CHUNK - c0 + (long long)LDS_ROW_COST * m;
    wgs = std::max(1ll, (chunks + target - 1) / target);
    if (wg < wgs) break;
    wg -= wgs;
  }
  if (t == T) {
    plan[u] = make_int4(0, 0, -1, 0);
    return;
  }
  const int64_t* offt = off + (long long)t * m;
  const long long k = wg * LDS_WAVES + u % LDS_WAVES, nk = wgs * LDS_WAVES;
  // first row whose first chunk is at or past share j of the tile
  auto row = [&](long long j) {
    if (j == 0) return 0;
    if (j == nk) return m;
    const long long c = c0 + (long long)((double)chunks * (double)j / (double)nk);
    int lo = 0, hi = m;
    while (lo < hi) {
      const int mid = lo + (hi - lo) / 2;
      if (offt[mid] / LDS_CHUNK + (long long)LDS_ROW_COST * mid < c) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  plan[u] = make_int4(row(k), row(k + 1), t, 0);
}

// ------------------------------------------------------------------ reductions
// y_r = alpha * scale_r * sum_t partial[t][r] + beta * y_r
__global__ __launch_bounds__(256) void k_lds_reduce(int m, int T, const float* __restrict__ partial,
                                                    const float* __restrict__ rowscale,
                                                    float alpha, float beta,
                                                    float* __restrict__ y) {
  const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= m) return;
  const float s = sum_ahead(partial + r, T, m);
  const float v = alpha * (rowscale ? rowscale[r] : 1.0f) * s;
  y[r] = beta == 0.0f ? v : v + beta * y[r];
}

// MLEM forward step from the partials: yhat_r = scale_r * sum_t partial[t][r],
// e_r = y_r / yhat_r (0 where yhat_r = 0; times the row scale when fold = 1),
// FP64 log-likelihood sum y log yhat - yhat, one atomic per workgroup: they are
// taken one by one, 12 ns each, so few workgroups of 1024 threads (1.1M rows of 5
// tiles: 56 us with 4096 workgroups of 256, 16 us with 512).
__global__ __launch_bounds__(LDS_BLOCK) void k_lds_ratio(int m, int T, const float* __restrict__ partial,
                                                   const float* __restrict__ rowscale,
                                                   const float* __restrict__ y,
                                                   float* __restrict__ e, int fold,
                                                   const int* __restrict__ itp,
                                                   double* __restrict__ loglik) {
  __shared__ double s_w[LDS_WAVES];
  double ll = 0.0;
  for (long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x; r < m;
       r += (long long)gridDim.x * blockDim.x) {
    const float yi = y[r];   // requested with the partials
    const float s = sum_ahead(partial + r, T, m);
    const float sc = rowscale ? rowscale[r] : 1.0f;
    const float yh = s * sc;
    const float ev = yh > 0.0f ? yi / yh : 0.0f;
    e[r] = fold ? ev * sc : ev;
    if (yh > 0.0f) ll += (double)yi * log((double)yh) - (double)yh;
  }
  ll = wave_sum(ll);
  if (lane_id() == 0) s_w[wave_id()] = ll;
  __syncthreads();
  if (threadIdx.x == 0 && loglik) {
    double tsum = 0.0;
    for (int w = 0; w < LDS_WAVES; w++) tsum += s_w[w];
    unsafeAtomicAdd(&loglik[*itp], tsum);
  }
}

// ------------------------------------------------------------------ dispatch
template <typename VT, int BWD>
static void launch_rows_lds(epet_ctx* ctx, const epet_matrix* A, const float* x, float* out,
                            const LdsStore& ep) {
  constexpr int D = LDS_DEPTH;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)k_rows_lds<VT, D, BWD>,
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              LDS_TILE * (int)sizeof(float));
    attr = true;
  }
  const size_t lds = sizeof(float) * (size_t)std::min(LDS_TILE, A->n);
  k_rows_lds<VT, D, BWD><<<(unsigned)A->lds_wgs, LDS_BLOCK, lds, ctx->stream>>>(
      A->m, A->n, A->lds_plan, A->lds_off, A->lds_col16,
      (const typename VT::T*)A->lds_val, x, out, ep, A->lds_map);
}

template <int BWD>
static void rows_lds(epet_ctx* ctx, const epet_matrix* A, const float* x, float* out,
                     const LdsStore& ep) {
  switch (A->value_type) {
    case EPET_VAL_F32: launch_rows_lds<ValF32, BWD>(ctx, A, x, out, ep); break;
    case EPET_VAL_BF16: launch_rows_lds<ValBF16, BWD>(ctx, A, x, out, ep); break;
    default: launch_rows_lds<ValF16, BWD>(ctx, A, x, out, ep); break;
  }
}

// Whether the LDS-tiled products apply (the context may turn them off): long
// rows, ascending columns.
static bool lds_wanted(const epet_ctx* ctx, const epet_matrix* A) {
  return ctx->opt.lds && A->m > 0 && A->cols_strict && (double)A->nnz / A->m >= 64.0;
}

static void lds_release(epet_matrix* A) {
  if (A->lds_off) (void)dev_free(A->lds_off);
  if (A->lds_val) (void)dev_free(A->lds_val);
  if (A->lds_col16) (void)dev_free(A->lds_col16);
  if (A->lds_partial) (void)dev_free(A->lds_partial);
  A->lds_off = nullptr;
  A->lds_val = nullptr;
  A->lds_col16 = nullptr;
  A->lds_partial = nullptr;
  if (A->lds_plan) (void)dev_free(A->lds_plan);
  A->lds_plan = nullptr;
  A->lds_T = A->lds_wgs = 0;
}

// Tile-major copy of A for column tiles of TV columns (a power of two up to
// 65536): *T_out tiles, offsets (T m + 1), values and tile-local 16-bit
// columns.  Allocates and synchronises.  On an allocation failure returns
// EPET_OK with *off == nullptr.
int build_tile_major(epet_ctx* ctx, const epet_matrix* A, int TV, ColMap mp, int* T_out,
                     long long* entries_out, int64_t** off_out, void** val_out, uint16_t** col_out) {
  *off_out = nullptr;
  *val_out = nullptr;
  *col_out = nullptr;
  hipStream_t st = ctx->stream;
  const int* scol = A->col;
  const void* sval = A->val;
  int* colp = nullptr;
  void* valp = nullptr;
  if (mp.nx > 0) {
    // renumbered columns: rows re-sorted into y-major column order first
    const size_t vb0 = A->value_type == EPET_VAL_F32 ? 4 : 2;
    if (dev_malloc((void**)&colp, sizeof(int) * (size_t)std::max(1ll, A->nnz)) != hipSuccess ||
        dev_malloc((void**)&valp, vb0 * (size_t)std::max(1ll, A->nnz)) != hipSuccess) {
      (void)hipGetLastError();
      if (colp) (void)dev_free(colp);
      return EPET_OK;
    }
    const unsigned g = (unsigned)std::max<long long>(
        1, std::min<long long>(((long long)A->m + 3) / 4, 16ll * ctx->num_cus));
    const size_t lds = sizeof(int) * (256 / WAVE) * (size_t)mp.ny;
    if (vb0 == 4)
      k_ysort_rows<float><<<g, 256, lds, st>>>(A->m, A->rowptr, A->col, (const float*)A->val, mp,
                                               colp, (float*)valp);
    else
      k_ysort_rows<uint16_t><<<g, 256, lds, st>>>(A->m, A->rowptr, A->col,
                                                  (const uint16_t*)A->val, mp, colp,
                                                  (uint16_t*)valp);
    const hipError_t le = hipGetLastError();
    if (le != hipSuccess) {
      (void)dev_free(colp);
      (void)dev_free(valp);
      EPET_FAIL(EPET_ERR_HIP, std::string("k_ysort_rows: ") + hipGetErrorString(le));
    }
    scol = colp;
    sval = valp;
  }
  const int T = (int)(((long long)A->n + TV - 1) / TV);
  const long long nseg = (long long)A->m * T;
  const size_t vb = A->value_type == EPET_VAL_F32 ? 4 : 2;
  uint32_t* toff = nullptr;
  int* cnt = nullptr;
  int64_t* off = nullptr;
  void* val = nullptr;
  uint16_t* col16 = nullptr;
  bool ok = T >= 1 &&
            dev_malloc((void**)&toff, sizeof(uint32_t) * (size_t)A->m * (T + 1)) == hipSuccess &&
            dev_malloc((void**)&cnt, sizeof(int) * (size_t)std::max(1ll, nseg)) == hipSuccess &&
            dev_malloc((void**)&off, sizeof(int64_t) * (size_t)(nseg + 1)) == hipSuccess;
  int rc = EPET_OK;
  long long tot = 0;
  if (ok) {
    launch_row_plan(st, A->m, T, TV, A->rowptr, scol, toff);
    k_lds_counts<<<grid_for(nseg, 256, 1ll << 31), 256, 0, st>>>(A->m, T, toff, cnt);
    rc = exclusive_scan_i32_to_i64(ctx, cnt, off, nseg, &tot);
    if (rc == EPET_OK && (tot < A->nnz || tot > A->nnz + (long long)(LDS_CHUNK - 1) * nseg))
      rc = fail(EPET_ERR_STATE, __FILE__, __LINE__, "tile-major copy: entry count mismatch");
    ok = rc == EPET_OK &&
         dev_malloc((void**)&val, vb * (size_t)std::max<long long>(LDS_CHUNK, tot)) == hipSuccess &&
         dev_malloc((void**)&col16, sizeof(uint16_t) * (size_t)std::max<long long>(LDS_CHUNK, tot)) == hipSuccess;
    if (rc == EPET_OK && !ok) (void)hipGetLastError();
    if (ok) {
      k_lds_set_last<<<1, 64, 0, st>>>(off, nseg, tot);
      const unsigned g = (unsigned)std::max<long long>(
          1, std::min<long long>((nseg * LDSF_LANES + 255) / 256, 16ll * ctx->num_cus));
      if (vb == 4)
        k_lds_fill<float><<<g, 256, 0, st>>>(A->m, T, TV - 1, A->rowptr, toff, scol,
                                             (const float*)sval, off, col16, (float*)val);
      else
        k_lds_fill<uint16_t><<<g, 256, 0, st>>>(A->m, T, TV - 1, A->rowptr, toff, scol,
                                                (const uint16_t*)sval, off, col16,
                                                (uint16_t*)val);
      if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
        rc = fail(EPET_ERR_HIP, __FILE__, __LINE__, "tile-major copy");
    }
  } else {
    (void)hipGetLastError();
  }
  if (toff) (void)dev_free(toff);
  if (cnt) (void)dev_free(cnt);
  if (colp) (void)dev_free(colp);
  if (valp) (void)dev_free(valp);
  if (!ok || rc != EPET_OK) {
    if (off) (void)dev_free(off);
    if (val) (void)dev_free(val);
    if (col16) (void)dev_free(col16);
    return rc;
  }
  *T_out = T;
  *entries_out = tot;
  *off_out = off;
  *val_out = val;
  *col_out = col16;
  return EPET_OK;
}

// y-major column order for the copy of a grid matrix when the context asks
// for it (EPET_LDS_MAP=1).  Off by default: rows then meet fewer tiles, but
// their segments become very uneven (most empty, a few long), which leaves the
// row groups of a wavefront idle; at 52^3 the forward product took 5.6 ms
// instead of 4.5 ms.
static ColMap voxel_map(const epet_ctx* ctx, const epet_matrix* A) {
  ColMap mp;
  if (!ctx->opt.lds_map || !ctx->have_geo) return mp;
  const int* gn = ctx->geo.gn;
  if ((long long)gn[0] * gn[1] * gn[2] != A->n || gn[1] > 4096) return mp;
  mp.nx = gn[0];
  mp.ny = gn[1];
  mp.nz = gn[2];
  return mp;
}

// Builds the tile-major copy and the partial buffer once (allocates and
// synchronises).  voxel_columns: the columns are
// image voxels (a forward projector), so they may be renumbered.  Leaves the
// matrix without them when an allocation fails; the other products then run.
int lds_prepare_map(epet_ctx* ctx, epet_matrix* A, bool voxel_columns) {
  if (A->lds_off || A->lds_failed || !lds_wanted(ctx, A)) return EPET_OK;
  int T = 0;
  const ColMap mp = voxel_columns ? voxel_map(ctx, A) : ColMap{};
  long long entries = 0;
  EPET_TRY(build_tile_major(ctx, A, LDS_TILE, mp, &T, &entries, &A->lds_off, &A->lds_val, &A->lds_col16));
  A->lds_map = mp;
  if (A->lds_off) {
    const long long cost = entries / LDS_CHUNK + (long long)LDS_ROW_COST * A->m * T;
    const long long per_cu =
        cost / ((long long)LDS_MIN_BLOCKS * WAVE * LDS_WAVES * ctx->num_cus) + 1;
    // whole rounds of the CUs, the tiles' own rounding up included
    const long long budget = std::min<long long>(LDS_PER_CU, per_cu) * ctx->num_cus;
    const long long target = 1 + cost / (budget > 2 * T ? budget - T : budget);
    const long long wgs = T + cost / target;
    if (wgs < (1ll << 31) &&
        dev_malloc((void**)&A->lds_plan, sizeof(int4) * LDS_WAVES * (size_t)wgs) == hipSuccess &&
        dev_malloc((void**)&A->lds_partial, sizeof(float) * (size_t)A->m * T) == hipSuccess) {
      k_lds_plan<<<grid_for(wgs * LDS_WAVES, 256, 1ll << 31), 256, 0, ctx->stream>>>(
          A->m, T, target, wgs * LDS_WAVES, A->lds_off, A->lds_plan);
      EPET_HIP(hipGetLastError());
      EPET_HIP(hipStreamSynchronize(ctx->stream));
      A->lds_T = T;
      A->lds_wgs = (int)wgs;
      return EPET_OK;
    }
  }
  (void)hipGetLastError();
  lds_release(A);
  A->lds_failed = true;
  return EPET_OK;
}

int lds_prepare(epet_ctx* ctx, epet_matrix* A) { return lds_prepare_map(ctx, A, false); }

bool lds_ready(const epet_ctx* ctx, const epet_matrix* A) {
  return A->lds_off != nullptr && lds_wanted(ctx, A);
}

// y = alpha * diag(scale) A x + beta y (scale: the row scale when use_scale;
// bwd: A is a transposed copy)
int lds_spmv(epet_ctx* ctx, const epet_matrix* A, const float* x, float alpha, float beta,
             float* y, bool use_scale, bool bwd) {
  const float* scale = use_scale ? A->rowscale : nullptr;
  const bool direct = A->lds_T == 1;
  const LdsStore ep{direct ? 1 : 0, scale, alpha, beta};
  float* out = direct ? y : A->lds_partial;
  if (bwd) rows_lds<1>(ctx, A, x, out, ep);
  else rows_lds<0>(ctx, A, x, out, ep);
  if (!direct)
    k_lds_reduce<<<grid_for(A->m, 256, 1ll << 31), 256, 0, ctx->stream>>>(
        A->m, A->lds_T, A->lds_partial, scale, alpha, beta, y);
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

// MLEM forward step (allocates nothing once prepared)
int lds_fwd_ratio(epet_ctx* ctx, const epet_matrix* A, const float* x, const float* y, float* e,
                  int fold, const int* itp, double* loglik) {
  rows_lds<0>(ctx, A, x, A->lds_partial, LdsStore{});
  k_lds_ratio<<<grid_for(A->m, LDS_BLOCK, 2ll * ctx->num_cus), LDS_BLOCK, 0, ctx->stream>>>(
      A->m, A->lds_T, A->lds_partial, A->rowscale, y, e, fold, itp, loglik);
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

}  // namespace epet
