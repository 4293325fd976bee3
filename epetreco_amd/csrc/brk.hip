// brk.hip -- multi-frame MLEM products on the matrix cores.
//
// F frames share one matrix M.  Rows that lie together in space meet the same
// columns: 32 channels of one neighbourhood of lines meet a third of the voxels
// in the union of their rows, 64 a quarter, and the same holds for neighbouring
// voxels and the channels through them.  So M is kept once more as bricks: 64
// rows (a row group) by 8 columns (an octet: a 2x2x2 brick of voxels, or 8
// neighbouring channels), of which about a sixth of the cells hold entries
// (52^3, 64 rays).  A step is two octets, the 32 x 16 operands of two matrix
// instructions (rows 0-31 and 32-63 of the group) that share the other operand:
//   mask[l]   lane l = 32 h + r, a halfword each for row r and row 32 + r: which
//             of the octet's 8 columns the row holds (low byte), words of the
//             half's entries before the row's (high byte)
//   head[h]   octet of half h; position of the step's first entry in the group;
//             words of the step's entries before half h of either rows
//   val       the entries, packed in (step, rows, half, row, column) order, a
//             row's 1 to 8 in an octet padded to whole words (pairs), a step's to
//             a multiple of 8
// Masks and heads of two steps make a record of 640 bytes, five cache lines that
// no other record shares (a load that meets a line still on its way waits for
// it), so an entry costs its value and 1.6 bytes of records.  A wavefront
// loads a step's entries as they lie (16 bytes a lane) and puts them in LDS, a
// lane reads its up to 8 entries from there, spreads them to their columns with
// byte permutes whose selectors come from a table of the 256 masks, and
// multiplies.
//
// Precision.  The matrix instruction multiplies bfloat16 exactly and adds in
// FP32, so both operands are split without loss: an FP32 number is the sum of
// three bfloat16 (8 of its 24 significant bits each, by truncation), a stored
// value of two (FP16) or one (BF16).  All part products are added, each exact, so
// the sums differ from FP32 fused multiply-adds only in the order of additions.
// By itself that would hold down to 2^-110 alone: a bfloat16 has no bits below
// 2^-133, an FP32 number has them down to 2^-149 (at 2^-120 the three parts miss 1e-4
// of it).  So k_brk_gather writes the vector times BRK_UP, and the sums are multiplied
// by 1 / BRK_UP (a factor in the main loop instead took 1 to 4% of the product).  The
// ratios that the forward product hands to the back projection are not scaled, as they
// may be large.  Matrices with stored values out of [BRK_VAL_MIN, BRK_VAL_MAX] stay
// with the other kernels.
// Measured against 64 bits (relative 2-norm of the images, 2 to 10 iterations of
// the four series in perf/cases.py): 1.9e-7 to 3.6e-7, with k_blk 2.9e-7 to 3.9e-7.
// The parts of the gathered vector are columns of the other operand: 8 frames x 3
// parts in one instruction of 32 columns, 16 frames in two, 32 in three, 64 in
// six.  They are made in registers, for both instructions of a step: kept split in
// memory the gathered vector took half as much again, and its cache lines are
// what a step waits for.
//
// Cells without an entry multiply the gathered vector by 0, which is not 0 for
// an infinity or NaN: frames that hold one are recomputed from the same bricks and
// the caller's vector entry by entry, and so are frames with numbers above BRK_BIG,
// whose scaled sums could leave the range, and with ratios below BRK_SMALL.  An
// infinite stored value would meet the zero parts of the vector: it is out of the
// range above.
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "epet_block.hpp"
#include "epet_internal.hpp"
#include "epet_plan.hpp"
#include "epet_rows.hpp"

namespace epet {

constexpr int BRK_SUB = 2;         // 32-row operands of a group
constexpr int BRK_ROWS = 32 * BRK_SUB;
constexpr int BRK_WAVES = 4;       // wavefronts (row groups) per workgroup
constexpr int BRK_PAD = 2;         // steps of a record; a group's steps are a multiple of it
constexpr int BRK_REC = 160;       // words of a record: 2 x 64 of masks, 2 x 2 x 4 of heads, 16 unused
constexpr int BRK_TAIL = 1024;     // readable entries past the last one (a step loads up to 1024)
constexpr int BRK_LL = 64;         // copies of the log-likelihood sums
// A step costs about the same however few entries it holds: 170 to 250 cycles of
// a CU measured (8 frames of FP16 values; 16 and 32), where k_blk took 2.3 to 2.9
// an entry.  MLEM iterations on bricks / k_blk / gather kernels in us, by the entries a
// step of both directions, FP32 values: 106 and 100, 4 frames 167 / 303 / 383; 85 and
// 130, 66 / 136 / 90; 67 and 84, 78 / 147 / 104; 50 and 65, 629 / 842 / 1434; 42 and 65,
// 69 / 104 / 81; 30 and 89, 401 / 346 / 714 (16 frames 408 / 510 / 607); 15 and 61,
// 1751 / 1499 / 2393 (32 frames 2500 / 5513 / 2349); BF16 values have won at all of
// them.  The line could lie at 40 to 50; it is where it was first drawn.
constexpr int BRK_MIN_ENTRIES = 80;

// scaled sums stay below 2^96 times a row's sum of magnitudes
constexpr float BRK_UP = 0x1p+24f, BRK_BIG = 0x1p+72f, BRK_SMALL = 0x1p-100f;
constexpr float BRK_VAL_MIN = 0x1p-100f, BRK_VAL_MAX = 0x1p+16f;

typedef __bf16 brk_bf8 __attribute__((ext_vector_type(8)));
typedef float brk_f16v __attribute__((ext_vector_type(16)));
typedef unsigned brk_u4 __attribute__((ext_vector_type(4)));
typedef float brk_f4 __attribute__((ext_vector_type(4)));

// matrix instructions of 32 columns per step for a padded frame count
__host__ __device__ constexpr int brk_nt(int Fp) { return Fp <= 8 ? 1 : Fp <= 16 ? 2 : Fp <= 32 ? 3 : 6; }
// parts of a stored value
static int brk_parts(int vt) { return vt == EPET_VAL_F32 ? 3 : vt == EPET_VAL_F16 ? 2 : 1; }

// The gathered vector of one padded frame count: [octet][2][Fp frames][4
// positions], so that a lane's two 16-byte loads lie next to its neighbours'.
struct BrkVec {
  int Fp = 0;
  float* x = nullptr;
  BrkVec* next = nullptr;
};

struct BrkCopy {
  int m = 0, mpos = 0, G = 0;       // rows, row positions (64 G), row groups
  int npos = 0, noct = 0;           // column positions (8 noct), octets
  int parts = 1;
  long long nsteps = 0, nent = 0;
  int* rowperm = nullptr;           // mpos: position -> row, -1 where none
  int* colinv = nullptr;            // npos: position -> column, -1 where none
  int64_t* gstep = nullptr;         // G + 1: first step of a group
  int64_t* gent = nullptr;          // G: first entry of a group
  unsigned* rec = nullptr;          // BRK_REC (nsteps / 2)
  uint16_t* val = nullptr;          // parts x (nent + BRK_TAIL)
  unsigned long long* flag = nullptr;   // frames of the gathered vector to do entry by entry
  double* ll = nullptr;             // BRK_LL x 64 log-likelihood sums (zero between iterations)
  float* partial = nullptr;         // splits x mpos x Fp
  long long partial_len = 0;
  BrkVec* vec = nullptr;
  // launch shape per padded frame count (log2 Fp - 3): splits, its time, frames tuned for
  int splits[4] = {1, 1, 1, 1}, tuned[4] = {0, 0, 0, 0};
  float ms[4] = {0, 0, 0, 0};
  ~BrkCopy() {
    for (void* p : {(void*)rowperm, (void*)colinv, (void*)gstep, (void*)gent, (void*)rec,
                    (void*)val, (void*)flag, (void*)ll, (void*)partial})
      if (p) (void)dev_free(p);
    while (vec) {
      BrkVec* v = vec;
      vec = v->next;
      if (v->x) (void)dev_free(v->x);
      delete v;
    }
  }
};

void brk_release(epet_matrix* A) {
  delete A->brk;
  A->brk = nullptr;
  A->brk_state.store(0);
}

static int brk_pad(int F) { return F <= 8 ? 8 : F <= 16 ? 16 : F <= 32 ? 32 : 64; }
static int brk_slot(int Fp) { return Fp == 8 ? 0 : Fp == 16 ? 1 : Fp == 32 ? 2 : 3; }

struct BrkArgs {
  int F, G, splits, mode;      // mode 0: MLEM ratio, 1: image, 2: partial sums
  int mpos;
  const int64_t* gstep;
  const int64_t* gent;
  const unsigned* rec;
  const uint16_t* val;
  long long vstride;           // between the parts of val
  const float* x;              // gathered vector
  float down;                  // 1 / its factor
  const float* xin;            // the vector it was gathered from, its columns by position
  const int* colinv;           // and a scale per column (or null); xin null: x is unscaled
  const float* xscale;
  const unsigned long long* flag;
  unsigned long long* clear;   // flag word of the other direction, cleared here (or null)
  const int* rowperm;
  float* out;                  // mode 1: rows x F, alpha scale_r sum + beta out
  float alpha, beta;
  float* oute;                 // mode 0: the other direction's gathered vector
  unsigned long long* oflag;   // mode 0: its flag word
  float* partial;
  const float* rowscale;
  int fold;
  const float* Y;
  const int* itp;
  double* ll;                  // BRK_LL copies (mode 0: added to; mode 1: summed into loglik)
  double* loglik;
};

// ------------------------------------------------------------------ splitting
// v truncated to bfloat16 (as FP32), and what that leaves; v is the sum of three
// such parts (8 significant bits each)
__device__ __forceinline__ float brk_hi(float v) {
  return __uint_as_float(__float_as_uint(v) & 0xFFFF0000u);
}
// the bfloat16 of a (low half) and b
__device__ __forceinline__ unsigned brk_pack(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float brk_bf(unsigned h) { return __uint_as_float(h << 16); }
// words of a record: mask of step st's lane l, head of its half h
__device__ __forceinline__ long long brk_mask_at(long long st, int l) {
  return (st >> 1) * BRK_REC + (st & 1) * 64 + l;
}
__device__ __forceinline__ long long brk_head_at(long long st, int h) {
  return (st >> 1) * BRK_REC + 128 + (st & 1) * 8 + h * 4;
}
// where position pos of frame f lies in the gathered vector
template <int FP>
__device__ __forceinline__ size_t brk_at(long long pos, int f) {
  return ((size_t)(pos >> 2) * FP + f) * 4 + (size_t)(pos & 3);
}
// Numbers that the split of a scaled and of an unscaled vector holds
__device__ __forceinline__ bool brk_fits_up(float v) { return fabsf(v) <= BRK_BIG; }
__device__ __forceinline__ bool brk_fits(float v) {
  return v == 0.0f || (fabsf(v) >= BRK_SMALL && fabsf(v) <= 3.402823466e38f);
}
// Flags the lanes' frames (lane l: frame base + l % FP, all lanes at once) by one
// atomic per wavefront and only where they are not flagged yet: atomics on one address
// take 12 ns each.
template <int FP>
__device__ __forceinline__ void brk_flag(unsigned long long* flag, bool set, int base) {
  unsigned long long m = __ballot(set);
  if (m == 0) return;
  if (FP <= 32) m |= m >> 32;
  if (FP <= 16) m |= m >> 16;
  if (FP <= 8) m |= m >> 8;
  if (FP < 64) m &= (1ull << (FP & 63)) - 1ull;
  m <<= base;
  if (lane_id() == 0 && (m & ~__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0)
    atomicOr(flag, m);
}

__device__ __forceinline__ void brk_store(const BrkArgs& a, long long at, float sum, float scale) {
  const float v = a.alpha * scale * sum;
  a.out[at] = a.beta == 0.0f ? v : v + a.beta * a.out[at];
}

// The gathered vector (times a scale per column, if any) times BRK_UP in position
// order: one thread per (four positions, frame).  Clears the other direction's flags
// and sets this one's.
template <int FP>
__global__ __launch_bounds__(256) void k_brk_gather(float* __restrict__ xs,
                                                    const float* __restrict__ X,
                                                    const float* __restrict__ scale,
                                                    const int* __restrict__ colinv, int nquad,
                                                    int F, unsigned long long* __restrict__ flag,
                                                    unsigned long long* __restrict__ clear) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && clear) *clear = 0;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int f = (int)(i % FP);
  const long long q = i / FP;
  bool out = false;
  if (q < nquad && f < F) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int c = colinv[q * 4 + j];
      v[j] = c >= 0 ? X[(long long)c * F + f] : 0.0f;
      if (scale && c >= 0) v[j] *= scale[c];
      out |= !brk_fits_up(v[j]);
      v[j] *= BRK_UP;
    }
    *reinterpret_cast<float4*>(xs + brk_at<FP>(q * 4, f)) = make_float4(v[0], v[1], v[2], v[3]);
  }
  brk_flag<FP>(flag, out, 0);
}

// ------------------------------------------------------------------ main kernel
// One wavefront per (row group, split of its steps), BRK_WAVES per workgroup;
// consecutive groups go to one XCD (workgroups are dealt to the 8 XCDs in turn),
// so that their octets of the gathered vector are read from its L2.
//
// A step's 64 rows share its loads of the gathered vector (2 KB at 32 frames),
// which come from L2 and are what bounds 32 frames of BF16 values: 30 cache lines
// a step and 11 TB/s of them, with the matrix cores busy a fifth of the time.  With
// 32 rows to a step and the vector kept split it took 1.00 ms (forward, 445,000
// rows of 899 entries), with 64 rows 0.77, with the parts made in registers 0.69,
// where k_blk took 2.0; the back projection 1.52, 0.80, 0.67 and 2.0 ms.  With
// two or three value parts and few frames it is the decoding's VALU work (75% busy).
// Loads run U to 2 U steps ahead; more wavefronts with fewer registers (4 per
// SIMD) spilled and took 1.5 times as long.
//
// Items are ordered by split first, so that the workgroups of one XCD work one
// part of the octets at a time (32-frame back projection: 1.52 -> 1.11 ms).
template <int NA, int FP>
__global__ __launch_bounds__(BRK_WAVES * WAVE) void k_brk(BrkArgs a) {
  constexpr int NT = brk_nt(FP);
  constexpr int NC = FP == 64 ? 2 : 1;              // accumulators of 32 columns
  constexpr int U = NA + NT <= 4 ? 2 : 1;           // steps per batch
  __shared__ uint4 selA[256];                       // columns 0-1, 2-3, 4-5, 6-7 from entries 0-3
  __shared__ uint2 selB[256];                       // columns 4-5, 6-7 from entries 4-7
  __shared__ brk_u4 s_val[BRK_WAVES][U * NA][2 * WAVE + 2];   // a step's entries (and words read past them)
  __shared__ double s_ll[64];
  {
    // byte selectors of each mask: column j takes entry popcount(mask below j)
    const unsigned m = threadIdx.x;
    unsigned lo[4], hi[4];
    int k = 0;
#pragma unroll
    for (int d = 0; d < 4; d++) {
      lo[d] = hi[d] = 0x0C0C0C0Cu;                  // 0x0C selects a zero byte
#pragma unroll
      for (int q = 0; q < 2; q++) {
        if ((m >> (2 * d + q)) & 1u) {
          const unsigned s = (unsigned)(2 * (k & 3)) * 0x0101u + 0x0100u;
          unsigned& to = k < 4 ? lo[d] : hi[d];
          to = (to & ~(0xFFFFu << (16 * q))) | (s << (16 * q));
          k++;
        }
      }
    }
    selA[m] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    selB[m] = make_uint2(hi[2], hi[3]);
  }
  if (threadIdx.x < 64) s_ll[threadIdx.x] = 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0 && a.clear) *a.clear = 0;
  if (a.mode != 0 && a.ll && blockIdx.x == 0 && (int)threadIdx.x < a.F) {
    // the forward product's log-likelihoods, in copy order
    double s = 0.0;
    for (int k = 0; k < BRK_LL; k++) {
      s += a.ll[k * 64 + threadIdx.x];
      a.ll[k * 64 + threadIdx.x] = 0.0;
    }
    if (a.loglik) a.loglik[(long long)(*a.itp) * a.F + threadIdx.x] += s;
  }
  __syncthreads();
  const int lane = lane_id(), h = lane >> 5, rl = lane & 31;
  const unsigned per = gridDim.x >> 3;
  const long long blk = (long long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const long long item = __builtin_amdgcn_readfirstlane((int)(blk * BRK_WAVES + wave_id()));
  double ll[NC] = {};
  if (item < (long long)a.G * a.splits) {
    const int g = (int)(item % a.G), sp = (int)(item / a.G);
    const long long s0 = a.gstep[g];
    const int nb = (int)((a.gstep[g + 1] - s0) / U);
    const int b0 = (int)((long long)nb * sp / a.splits);
    const int b1 = (int)((long long)nb * (sp + 1) / a.splits);
    // records, by 32-bit byte offsets from a uniform address
    const char* rp = reinterpret_cast<const char*>(a.rec + brk_mask_at(s0, 0));
    const unsigned ml = (unsigned)lane * 4;
    const unsigned hl = 512u + (unsigned)h * 16 + (U == 2 ? (unsigned)(lane & 1) * 32 : 0u);
    const char* vp = reinterpret_cast<const char*>(a.val + a.gent[g]);
    const char* xp = reinterpret_cast<const char*>(a.x);
    const unsigned xl = (unsigned)(FP >= 32 ? rl : rl % FP) * 16;
    const long long vs = 2 * a.vstride;

    struct Meta { brk_u4 hd; unsigned m[U]; };
    struct Data { brk_u4 v[U][NA]; brk_f4 x[U][NC][2]; unsigned m[U], at[U][BRK_SUB], pos[U]; };
    auto mask_at = [&](int st) {
      return __builtin_nontemporal_load(reinterpret_cast<const unsigned*>(
          rp + (size_t)(ml + (unsigned)(st >> 1) * (4u * BRK_REC) + (unsigned)(st & 1) * 256u)));
    };
    auto meta = [&](Meta& M, int b) {
      const int st = min(b, b1 - 1) * U;
      // one load for the heads of a batch: lane parity picks the step
      M.hd = __builtin_nontemporal_load(reinterpret_cast<const brk_u4*>(
          rp + (size_t)(hl + (unsigned)(st >> 1) * (4u * BRK_REC) + (unsigned)(st & 1) * 32u)));
#pragma unroll
      for (int u = 0; u < U; u++) M.m[u] = mask_at(st + u);
    };
    // word i of this lane's half's head of step u of a batch
    auto head = [&](const Meta& M, int u, int i) -> unsigned {
      if (U == 1) return M.hd[i];
      return u == 0 ? __builtin_amdgcn_mov_dpp(M.hd[i], 0xA0, 0xF, 0xF, true)    // lanes 0 0 2 2
                    : __builtin_amdgcn_mov_dpp(M.hd[i], 0xF5, 0xF, 0xF, true);   // lanes 1 1 3 3
    };
    // requests the steps of batch b (past the last one: no entries)
    auto data = [&](Data& D, const Meta& M, int b) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        D.m[u] = b < b1 ? M.m[u] & 0x00FF00FFu : 0u;
        const unsigned pos = head(M, u, 1), w = head(M, u, 3), t8 = w >> 16;
        D.at[u][0] = head(M, u, 2) + ((M.m[u] >> 8) & 0xFFu);
        D.at[u][1] = (w & 0xFFFFu) + (M.m[u] >> 24);
        D.pos[u] = pos | (t8 > 64u ? 1u : 0u);
        // lanes past the step's entries read its last ones again: a line that
        // the next step's loads want too would make those wait for it
        const unsigned at = 2 * pos + 16 * min((unsigned)lane, t8 - 1u);
        const unsigned xo = __umul24(head(M, u, 0), FP * 32) + xl;
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
          for (int q = 0; q < 2; q++)
            D.x[u][c][q] = *reinterpret_cast<const brk_f4*>(xp + (size_t)(xo + c * 512 + q * FP * 16));
#pragma unroll
        for (int k = 0; k < NA; k++)
          D.v[u][k] = __builtin_nontemporal_load(reinterpret_cast<const brk_u4*>(vp + k * vs + (size_t)at));
      }
    };
    brk_f16v acc[BRK_SUB][NC];
#pragma unroll
    for (int i = 0; i < BRK_SUB; i++)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][c][r] = 0.0f;
    brk_u4 (*sv)[2 * WAVE + 2] = s_val[wave_id()];
    // parts of an FP32 number: bits 31-16, 15-8 and 7-0, each with the exponent,
    // as differences of the number cut off at two places.  Up to 16 frames a
    // lane's column is one part (8 frames: 0, 1, 2 or none; 16: 0 or 1, then 2 or
    // none), by the places in its masks.
    constexpr unsigned HI = 0xFFFF0000u, MID = 0xFFFFFF00u;
    const int part = FP == 8 ? rl >> 3 : rl >> 4;
    const unsigned upto = part == 1 ? MID : ~0u;
    const unsigned from = part == 0 ? 0u : part == 1 ? HI : part == 2 ? MID : ~0u;
    const unsigned low = part == 0 ? MID : ~0u;                // 16 frames, t = 1
    auto cut = [](float v, unsigned mask) { return __uint_as_float(__float_as_uint(v) & mask); };
    auto work = [&](const Data& D) {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int k = 0; k < NA; k++) sv[u * NA + k][lane] = D.v[u][k];
#pragma unroll
      for (int u = 0; u < U; u++) {
        brk_u4 xt[NT];
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const float v0 = D.x[u][c][j >> 1][2 * (j & 1)], v1 = D.x[u][c][j >> 1][2 * (j & 1) + 1];
            if (FP <= 16) {
              xt[0][j] = brk_pack(cut(v0, upto) - cut(v0, from), cut(v1, upto) - cut(v1, from));
              if (FP == 16) xt[NT - 1][j] = brk_pack(v0 - cut(v0, low), v1 - cut(v1, low));
            } else {
              const float m0 = cut(v0, MID), m1 = cut(v1, MID);
              xt[(3 * c) % NT][j] = brk_pack(v0, v1);
              xt[(3 * c + 1) % NT][j] = brk_pack(m0 - cut(v0, HI), m1 - cut(v1, HI));
              xt[(3 * c + 2) % NT][j] = brk_pack(v0 - m0, v1 - m1);
            }
          }
        const unsigned pos = __builtin_amdgcn_readfirstlane(D.pos[u]);
        if (pos & 1u) {   // half full or more (rare): the entries past the 512 loaded ahead
#pragma unroll
          for (int k = 0; k < NA; k++)
            sv[u * NA + k][WAVE + lane] = *reinterpret_cast<const brk_u4*>(
                vp + k * vs + (size_t)(2 * (pos & ~7u) + 1024u + (unsigned)lane * 16));
        }
#pragma unroll
        for (int i = 0; i < BRK_SUB; i++) {
          const unsigned m = (D.m[u] >> (16 * i)) & 0xFFu;
          const uint4 sa = selA[m];
          const uint2 sb = selB[m];
#pragma unroll
          for (int k = 0; k < NA; k++) {
            // four words from a word (rows' entries start at words: from halfwords,
            // unaligned LDS reads took several times as long, and a fifth word
            // and four shifts a fifth of the loop)
            const unsigned* e = reinterpret_cast<const unsigned*>(sv[u * NA + k]) + D.at[u][i];
            const unsigned p0 = e[0], p1 = e[1], p2 = e[2], p3 = e[3];
            brk_u4 q;
            q.x = __builtin_amdgcn_perm(p1, p0, sa.x);
            q.y = __builtin_amdgcn_perm(p1, p0, sa.y);
            q.z = __builtin_amdgcn_perm(p1, p0, sa.z) | __builtin_amdgcn_perm(p3, p2, sb.x);
            q.w = __builtin_amdgcn_perm(p1, p0, sa.w) | __builtin_amdgcn_perm(p3, p2, sb.y);
            const brk_bf8 fa = __builtin_bit_cast(brk_bf8, q);
#pragma unroll
            for (int t = 0; t < NT; t++)
              acc[i][t / 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  fa, __builtin_bit_cast(brk_bf8, xt[t]), acc[i][t / 3], 0, 0, 0);
          }
        }
      }
    };
    if (b0 < b1) {
      // Loads return in order, so a batch's masks and heads are requested before
      // the entries of the batch before it: waiting for them then leaves those in
      // flight.  The loads stay where they are written: left to itself the
      // compiler moves each to its use, to hold fewer registers, and the
      // wavefront waits for every one.
      Meta M, N;
      Data A, B;
      meta(M, b0);
      meta(N, b0 + 1);
      data(A, M, b0);
      __builtin_amdgcn_sched_barrier(0);
      for (int b = b0; b < b1; b += 2) {
        meta(M, b + 2);
        __builtin_amdgcn_sched_barrier(0);
        data(B, N, b + 1);
        __builtin_amdgcn_sched_barrier(0);
        work(A);
        __builtin_amdgcn_sched_barrier(0);
        meta(N, b + 3);
        __builtin_amdgcn_sched_barrier(0);
        data(A, M, b + 2);
        __builtin_amdgcn_sched_barrier(0);
        work(B);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // lane (h, n) holds column n of rows 8 (r / 4) + 4 h + r % 4; the parts of a
    // frame that lie in several columns are added, so that every lane holds its
    // frame's sums
    if (FP <= 16) {
#pragma unroll
      for (int i = 0; i < BRK_SUB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          if (FP == 8) acc[i][0][r] += __shfl_xor(acc[i][0][r], 8, WAVE);
          acc[i][0][r] += __shfl_xor(acc[i][0][r], 16, WAVE);
        }
    }
    if (a.down != 1.0f) {
#pragma unroll
      for (int i = 0; i < BRK_SUB; i++)
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[i][c][r] *= a.down;
    }
    // frames with numbers that the split does not hold: entry by entry
    const unsigned long long bad = *a.flag & (a.F >= 64 ? ~0ull : (1ull << a.F) - 1ull);
    if (bad) {
      for (int f = 0; f < a.F; f++) {
        if (!((bad >> f) & 1ull)) continue;
        float sum[BRK_SUB] = {};
        for (int st = b0 * U; st < b1 * U; st++) {
          const brk_u4 hd = *reinterpret_cast<const brk_u4*>(a.rec + brk_head_at(s0 + st, h));
          const unsigned mk = mask_at(st);
#pragma unroll
          for (int i = 0; i < BRK_SUB; i++) {
            unsigned at = hd.y + 2 * ((i == 0 ? hd.z : hd.w & 0xFFFFu) + ((mk >> (16 * i + 8)) & 0xFFu));
            for (int j = 0; j < 8; j++) {
              if (!((mk >> (16 * i + j)) & 1u)) continue;
              float v = 0.0f;
              for (int k = NA - 1; k >= 0; k--)
                v += brk_bf(reinterpret_cast<const uint16_t*>(vp + k * vs)[at]);
              const long long pos = (long long)hd.x * 8 + j;
              float x;
              if (a.xin) {
                const int col = a.colinv[pos];
                x = a.xin[(long long)col * a.F + f];
                if (a.xscale) x *= a.xscale[col];
              } else {
                x = a.x[brk_at<FP>(pos, f)];
              }
              sum[i] += v * x;
              at++;
            }
          }
        }
#pragma unroll
        for (int i = 0; i < BRK_SUB; i++) {
          const float s = sum[i] + __shfl_xor(sum[i], 32, WAVE);   // row 32 i + rl of the group
#pragma unroll
          for (int c = 0; c < NC; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
              const float v = __shfl(s, 8 * (r >> 2) + 4 * h + (r & 3), WAVE);
              if (32 * c + rl % FP == f) acc[i][c][r] = v;
            }
        }
      }
    }
    // ---- epilogue
    const int f0 = FP >= 32 ? rl : rl % FP;         // this lane's frame (and f0 + 32)
    const int q = FP >= 32 ? 0 : rl / FP;           // which of the lanes that hold it
    constexpr int Q = FP >= 32 ? 1 : 32 / FP;
#pragma unroll
    for (int i = 0; i < BRK_SUB; i++) {
    const int p0 = g * BRK_ROWS + 32 * i;
    const int row = a.rowperm[p0 + rl];
    const float scale = a.rowscale && row >= 0 ? a.rowscale[row] : 1.0f;
    if (a.mode == 2) {
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (r % Q == q)
            a.partial[((long long)sp * a.mpos + p0 + 8 * (r >> 2) + 4 * h + (r & 3)) * FP + 32 * c +
                      f0] = acc[i][c][r];
    } else if (a.mode == 1) {
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int o = __shfl(row, 8 * (r >> 2) + 4 * h + (r & 3), WAVE);
          const int f = 32 * c + f0;
          const float sc = __shfl(scale, 8 * (r >> 2) + 4 * h + (r & 3), WAVE);
          if (r % Q == q && o >= 0 && f < a.F) brk_store(a, (long long)o * a.F + f, acc[i][c][r], sc);
        }
    } else {
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const int f = 32 * c + f0;
        bool out = false;
#pragma unroll
        for (int o8 = 0; o8 < 4; o8++) {            // octet o8 of the group, positions 4 h .. 4 h + 3
          float w[4];
#pragma unroll
          for (int r4 = 0; r4 < 4; r4++) {
            const int o = __shfl(row, 8 * o8 + 4 * h + r4, WAVE);
            const float sc = __shfl(scale, 8 * o8 + 4 * h + r4, WAVE);
            float ev = 0.0f;
            if (o >= 0 && f < a.F) {
              const float yh = acc[i][c][4 * o8 + r4] * sc;
              const float yi = a.Y[(long long)o * a.F + f];
              ev = yh > 0.0f ? yi / yh : 0.0f;
              if (yh > 0.0f && q == 0) ll[c] += (double)yi * log((double)yh) - (double)yh;
              if (a.fold) ev *= sc;
              out |= !brk_fits(ev);
            }
            w[r4] = ev;
          }
          if (q == 0)
            *reinterpret_cast<float4*>(a.oute + brk_at<FP>(p0 + 8 * o8 + 4 * h, f)) =
                make_float4(w[0], w[1], w[2], w[3]);
        }
        brk_flag<(FP < 32 ? FP : 32)>(a.oflag, out, 32 * c);
      }
    }
    }
  }
  if (a.mode == 0 && a.ll) {
    const int f0 = FP >= 32 ? (lane & 31) : (lane & 31) % FP;
#pragma unroll
    for (int c = 0; c < NC; c++)
      if (ll[c] != 0.0) atomicAdd(&s_ll[32 * c + f0], ll[c]);
    __syncthreads();
    if ((int)threadIdx.x < a.F)
      unsafeAtomicAdd(&a.ll[(blockIdx.x % BRK_LL) * 64 + threadIdx.x], s_ll[threadIdx.x]);
  }
}

// Sums of the splits, in split order: the ratio or the image of one (position,
// frame) per thread.
template <int FP>
__global__ __launch_bounds__(256) void k_brk_reduce(BrkArgs a) {
  __shared__ double s_ll[64];
  if (threadIdx.x < 64) s_ll[threadIdx.x] = 0.0;
  __syncthreads();
  const long long tot = (long long)a.mpos * FP;
  bool out = false;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < tot;
       i += (long long)gridDim.x * blockDim.x) {
    const long long p = i / FP;
    const int f = (int)(i % FP);
    if (f >= a.F) continue;
    const int o = a.rowperm[p];
    if (o < 0) continue;
    const float s = sum_ahead(a.partial + i, a.splits, (long long)a.mpos * FP);
    const float sc = a.rowscale ? a.rowscale[o] : 1.0f;
    if (a.mode == 1) {
      brk_store(a, (long long)o * a.F + f, s, sc);
      continue;
    }
    const float yh = s * sc;
    const float yi = a.Y[(long long)o * a.F + f];
    float ev = yh > 0.0f ? yi / yh : 0.0f;
    if (yh > 0.0f) atomicAdd(&s_ll[f], (double)yi * log((double)yh) - (double)yh);
    if (a.fold) ev *= sc;
    out |= !brk_fits(ev);
    a.oute[brk_at<FP>(p, f)] = ev;
  }
  if (a.mode == 0) brk_flag<FP>(a.oflag, out, 0);   // a thread stays on its frame
  if (a.mode == 0 && a.ll) {
    __syncthreads();
    if ((int)threadIdx.x < a.F)
      unsafeAtomicAdd(&a.ll[(blockIdx.x % BRK_LL) * 64 + threadIdx.x], s_ll[threadIdx.x]);
  }
}

// ------------------------------------------------------------------ build
constexpr int BRK_BUILD = 256;

// the octets that group g's rows meet, as bits in LDS
__device__ __forceinline__ void brk_bits(unsigned* bits, int nwords, int g,
                                         const int* __restrict__ rowperm,
                                         const int64_t* __restrict__ rowptr,
                                         const int* __restrict__ col,
                                         const int* __restrict__ cpos) {
  for (int i = threadIdx.x; i < nwords; i += BRK_BUILD) bits[i] = 0;
  __syncthreads();
  for (int r = wave_id(); r < BRK_ROWS; r += BRK_BUILD / WAVE) {
    const int row = rowperm[g * BRK_ROWS + r];
    if (row < 0) continue;
    const int64_t b = rowptr[row], e = rowptr[row + 1];
    for (int64_t k = b + lane_id(); k < e; k += WAVE) {
      const int o = cpos[col[k]] >> 3;
      atomicOr(&bits[o >> 5], 1u << (o & 31));
    }
  }
  __syncthreads();
}

// steps of every group
__global__ __launch_bounds__(BRK_BUILD) void k_brk_count(int nwords, const int* __restrict__ rowperm,
                                                         const int64_t* __restrict__ rowptr,
                                                         const int* __restrict__ col,
                                                         const int* __restrict__ cpos,
                                                         int* __restrict__ nstep) {
  extern __shared__ unsigned brk_lds[];
  __shared__ int s_wave[BRK_BUILD / WAVE];
  const int g = blockIdx.x;
  brk_bits(brk_lds, nwords, g, rowperm, rowptr, col, cpos);
  int c = 0;
  for (int i = threadIdx.x; i < nwords; i += BRK_BUILD) c += __popc(brk_lds[i]);
  int tot;
  (void)block_excl_sum<BRK_BUILD>(c, s_wave, &tot);
  if (threadIdx.x == 0) {
    const int steps = (tot + 1) / 2;
    nstep[g] = (steps + BRK_PAD - 1) / BRK_PAD * BRK_PAD;
  }
}

// bits and, per word, the octets before it: rank of an octet in the group
__device__ __forceinline__ void brk_ranks(unsigned* bits, int* before, int nwords, int* s_wave) {
  int run = 0;
  for (int base = 0; base < nwords; base += BRK_BUILD) {
    const int i = base + threadIdx.x;
    int tot;
    const int ex = block_excl_sum<BRK_BUILD>(i < nwords ? __popc(bits[i]) : 0, s_wave, &tot);
    if (i < nwords) before[i] = run + ex;
    run += tot;
  }
  __syncthreads();
}
__device__ __forceinline__ int brk_rank(const unsigned* bits, const int* before, int o) {
  return before[o >> 5] + __popc(bits[o >> 5] & ((1u << (o & 31)) - 1u));
}

// octets of the heads and masks of the entries (mask and head zero before)
__global__ __launch_bounds__(BRK_BUILD) void k_brk_masks(int nwords, const int* __restrict__ rowperm,
                                                         const int64_t* __restrict__ rowptr,
                                                         const int* __restrict__ col,
                                                         const int* __restrict__ cpos,
                                                         const int64_t* __restrict__ gstep,
                                                         unsigned* __restrict__ rec) {
  extern __shared__ unsigned brk_lds[];
  __shared__ int s_wave[BRK_BUILD / WAVE];
  int* before = reinterpret_cast<int*>(brk_lds + nwords);
  const int g = blockIdx.x;
  brk_bits(brk_lds, nwords, g, rowperm, rowptr, col, cpos);
  brk_ranks(brk_lds, before, nwords, s_wave);
  const long long s0 = gstep[g];
  for (int i = threadIdx.x; i < nwords; i += BRK_BUILD) {
    unsigned w = brk_lds[i];
    int q = before[i];
    while (w) {
      rec[brk_head_at(s0 + (q >> 1), q & 1)] = (unsigned)(i * 32 + __ffs(w) - 1);
      w &= w - 1;
      q++;
    }
  }
  for (int r = wave_id(); r < BRK_ROWS; r += BRK_BUILD / WAVE) {
    const int row = rowperm[g * BRK_ROWS + r];
    if (row < 0) continue;
    const int64_t b = rowptr[row], e = rowptr[row + 1];
    for (int64_t k = b + lane_id(); k < e; k += WAVE) {
      const int pos = cpos[col[k]];
      const int q = brk_rank(brk_lds, before, pos >> 3);
      atomicOr(&rec[brk_mask_at(s0 + (q >> 1), (q & 1) * 32 + (r & 31))],
               1u << ((pos & 7) + 16 * (r >> 5)));
    }
  }
}

// entries of the half before each lane (high bytes of the masks), of a step
// before its halves, positions of the steps' first entries in the group, and the
// group's entries with their padding
__global__ __launch_bounds__(BRK_BUILD) void k_brk_offsets(const int64_t* __restrict__ gstep,
                                                           unsigned* __restrict__ rec,
                                                           int* __restrict__ nent) {
  __shared__ int s_wave[BRK_BUILD / WAVE];
  const int g = blockIdx.x;
  const long long s0 = gstep[g];
  const int n = (int)(gstep[g + 1] - s0);
  const int lane = lane_id();
  for (int s = wave_id(); s < n; s += BRK_BUILD / WAVE) {
    const long long at = brk_mask_at(s0 + s, lane);
    unsigned m = rec[at] & 0x00FF00FFu;
    // words of both rows of the lane, a halfword each
    const unsigned own = (unsigned)(__popc(m & 0xFFFFu) + 1) / 2 |
                         (unsigned)(__popc(m >> 16) + 1) / 2 << 16;
    unsigned x = own;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
      const unsigned y = __shfl_up(x, off, 32);
      if ((lane & 31) >= off) x += y;
    }
    rec[at] = m | ((x - own) & 0x00FF00FFu) << 8;
    const unsigned a = __shfl(x, 31, WAVE), b = __shfl(x, 63, WAVE);
    if (lane == 0) {
      const unsigned n00 = a & 0xFFFFu, n01 = b & 0xFFFFu, n10 = a >> 16, n11 = b >> 16;
      const unsigned tot = n00 + n01 + n10 + n11;
      const unsigned t8 = (tot + 3u) / 4u << 16;   // 16-byte units, in the high half
      unsigned* hd = rec + brk_head_at(s0 + s, 0);   // two halves of four words
      hd[1] = 2 * ((tot + 3u) & ~3u);
      hd[2] = 0u;
      hd[6] = n00;
      hd[3] = (n00 + n01) | t8;
      hd[7] = (n00 + n01 + n10) | t8;
    }
  }
  __syncthreads();
  // positions of the steps' first entries
  int run = 0;
  for (int base = 0; base < n; base += BRK_BUILD) {
    const int i = base + threadIdx.x;
    unsigned* hd = rec + brk_head_at(s0 + min(i, n - 1), 0);
    const int c = i < n ? (int)hd[1] : 0;
    int tot;
    const int ex = block_excl_sum<BRK_BUILD>(c, s_wave, &tot);
    if (i < n) hd[1] = hd[5] = (unsigned)(run + ex);
    run += tot;
  }
  if (threadIdx.x == 0) nent[g] = run;
}

// the entries' parts
template <typename V>
__global__ __launch_bounds__(BRK_BUILD) void k_brk_values(int nwords, int vt, int parts,
                                                          const int* __restrict__ rowperm,
                                                          const int64_t* __restrict__ rowptr,
                                                          const int* __restrict__ col,
                                                          const V* __restrict__ mval,
                                                          const int* __restrict__ cpos,
                                                          const int64_t* __restrict__ gstep,
                                                          const int64_t* __restrict__ gent,
                                                          const unsigned* __restrict__ rec,
                                                          uint16_t* __restrict__ val,
                                                          long long vstride,
                                                          int* __restrict__ out_of_range) {
  extern __shared__ unsigned brk_lds[];
  __shared__ int s_wave[BRK_BUILD / WAVE];
  int* before = reinterpret_cast<int*>(brk_lds + nwords);
  const int g = blockIdx.x;
  brk_bits(brk_lds, nwords, g, rowperm, rowptr, col, cpos);
  brk_ranks(brk_lds, before, nwords, s_wave);
  const long long s0 = gstep[g], e0 = gent[g];
  for (int r = wave_id(); r < BRK_ROWS; r += BRK_BUILD / WAVE) {
    const int row = rowperm[g * BRK_ROWS + r];
    if (row < 0) continue;
    const int64_t b = rowptr[row], e = rowptr[row + 1];
    for (int64_t k = b + lane_id(); k < e; k += WAVE) {
      const int pos = cpos[col[k]];
      const int q = brk_rank(brk_lds, before, pos >> 3);
      const unsigned m = rec[brk_mask_at(s0 + (q >> 1), (q & 1) * 32 + (r & 31))] >> (16 * (r >> 5));
      const unsigned* hd = rec + brk_head_at(s0 + (q >> 1), q & 1);
      const long long at = e0 + hd[1] + 2 * ((r < 32 ? hd[2] : hd[3] & 0xFFFFu) + ((m >> 8) & 0xFFu)) +
                           __popc(m & 0xFFu & ((1u << (pos & 7)) - 1u));
      float v = vt == EPET_VAL_F32    ? (float)mval[k]
                : vt == EPET_VAL_BF16 ? brk_bf((unsigned)mval[k])
                                      : __half2float(__ushort_as_half((uint16_t)mval[k]));
      if (v != 0.0f && !(fabsf(v) >= BRK_VAL_MIN && fabsf(v) <= BRK_VAL_MAX)) *out_of_range = 1;
      if (vt == EPET_VAL_BF16) {
        val[at] = (uint16_t)mval[k];
      } else {
        for (int i = 0; i < parts; i++) {
          val[i * vstride + at] = (uint16_t)(__float_as_uint(v) >> 16);
          v -= brk_hi(v);
        }
      }
    }
  }
}

__global__ __launch_bounds__(256) void k_brk_zero(uint4* __restrict__ p, long long n16) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n16) p[i] = make_uint4(0u, 0u, 0u, 0u);
}
// bytes rounded up to 16 by the allocations
static void brk_zero(hipStream_t st, void* p, size_t bytes) {
  const long long n = (long long)((bytes + 15) / 16);
  if (n > 0) k_brk_zero<<<grid_for(n, 256, 1ll << 31), 256, 0, st>>>((uint4*)p, n);
}

// ------------------------------------------------------------------ orders (host)
std::vector<int> channel_order(const MatGeo& g, const std::vector<int>& ids);

static uint64_t brk_morton(uint32_t x, uint32_t y, uint32_t z) {
  uint64_t r = 0;
  for (int b = 0; b < 21; b++)
    r |= ((uint64_t)((x >> b) & 1u) << (3 * b + 2)) | ((uint64_t)((y >> b) & 1u) << (3 * b + 1)) |
         ((uint64_t)((z >> b) & 1u) << (3 * b));
  return r;
}

// Voxel positions: 2x2x2 bricks in Morton order, 8 positions each, -1 where a
// brick reaches past the grid.
static std::vector<int> brk_voxel_positions(const MatGeo& g) {
  const int bx = (g.nx + 1) / 2, by = (g.ny + 1) / 2, bz = (g.nz + 1) / 2;
  std::vector<std::pair<uint64_t, int>> key((size_t)bx * by * bz);
  for (int i = 0; i < (int)key.size(); i++)
    key[i] = {brk_morton(i / (by * bz), i / bz % by, i % bz), i};
  std::sort(key.begin(), key.end());
  std::vector<int> pos(key.size() * 8, -1);
  for (size_t k = 0; k < key.size(); k++) {
    const int i = key[k].second, x0 = 2 * (i / (by * bz)), y0 = 2 * (i / bz % by), z0 = 2 * (i % bz);
    for (int j = 0; j < 8; j++) {
      const int x = x0 + (j >> 2), y = y0 + ((j >> 1) & 1), z = z0 + (j & 1);
      if (x < g.nx && y < g.ny && z < g.nz) pos[k * 8 + j] = (x * g.ny + y) * g.nz + z;
    }
  }
  return pos;
}

// ------------------------------------------------------------------ build (host)
// Bricks of M with row positions `rows` and column positions `cols` (-1: none).
// EPET_OK with *out == nullptr when memory is short, or (*unfit) the sizes are
// beyond the kernel's, the values beyond the split's or the bricks too empty to pay.
static int brk_build(epet_ctx* ctx, const epet_matrix* M, const std::vector<int>& rows,
                     const std::vector<int>& cols, BrkCopy** out, bool* unfit) {
  *out = nullptr;
  hipStream_t st = ctx->stream;
  BrkCopy* B = new BrkCopy();
  struct Guard {
    BrkCopy* b;
    std::vector<void*> tmp;
    ~Guard() {
      for (void* p : tmp) (void)dev_free(p);
      delete b;
    }
  } own{B, {}};
  B->m = M->m;
  B->G = (int)((rows.size() + BRK_ROWS - 1) / BRK_ROWS);
  B->mpos = B->G * BRK_ROWS;
  // whole groups of positions: the forward product writes the ratios of a whole
  // row group into the other direction's gathered vector
  B->noct = (int)((cols.size() + BRK_ROWS - 1) / BRK_ROWS) * (BRK_ROWS / 8);
  B->npos = B->noct * 8;
  B->parts = brk_parts(M->value_type);
  const int nwords = (B->noct + 31) / 32;
  const size_t lds = 2 * sizeof(int) * (size_t)nwords;
  // octets of a row group in LDS (which bounds them below 2^24); entries
  // of a group and its steps' padding counted in 31 bits of bytes
  if (lds > 150 * 1024 || 4ll * BRK_ROWS * M->n >= (1ll << 31)) {
    *unfit = true;
    return EPET_OK;
  }
  std::vector<int> rp(B->mpos, -1), ci(B->npos, -1), cpos(std::max(1, M->n), 0);
  std::copy(rows.begin(), rows.end(), rp.begin());
  std::copy(cols.begin(), cols.end(), ci.begin());
  for (size_t i = 0; i < cols.size(); i++)
    if (cols[i] >= 0) cpos[cols[i]] = (int)i;
  bool ok = true;
  auto alloc = [&](auto** p, size_t bytes) {
    if (ok && dev_malloc((void**)p, (bytes + 15) & ~(size_t)15) != hipSuccess) {
      (void)hipGetLastError();
      ok = false;
    }
  };
  auto temp = [&](auto** p, size_t bytes) {
    alloc(p, bytes);
    if (*p) own.tmp.push_back(*p);
  };
  int *cpos_d = nullptr, *ns = nullptr, *ne = nullptr;
  alloc(&B->rowperm, sizeof(int) * rp.size());
  alloc(&B->colinv, sizeof(int) * ci.size());
  alloc(&B->gstep, sizeof(int64_t) * (B->G + 1));
  alloc(&B->gent, sizeof(int64_t) * B->G);
  alloc(&B->flag, 16);
  alloc(&B->ll, sizeof(double) * BRK_LL * 64);
  temp(&cpos_d, sizeof(int) * cpos.size());
  temp(&ns, sizeof(int) * B->G);
  temp(&ne, sizeof(int) * B->G);
  if (!ok) return EPET_OK;
  EPET_HIP(hipMemcpyAsync(B->rowperm, rp.data(), sizeof(int) * rp.size(), hipMemcpyHostToDevice, st));
  EPET_HIP(hipMemcpyAsync(B->colinv, ci.data(), sizeof(int) * ci.size(), hipMemcpyHostToDevice, st));
  EPET_HIP(hipMemcpyAsync(cpos_d, cpos.data(), sizeof(int) * cpos.size(), hipMemcpyHostToDevice, st));
  brk_zero(st, B->flag, 16);
  brk_zero(st, B->ll, sizeof(double) * BRK_LL * 64);
  for (const void* k : {(const void*)k_brk_count, (const void*)k_brk_masks,
                        (const void*)k_brk_values<float>, (const void*)k_brk_values<uint16_t>})
    (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
  k_brk_count<<<B->G, BRK_BUILD, lds, st>>>(nwords, B->rowperm, M->rowptr, M->col, cpos_d, ns);
  EPET_HIP(hipGetLastError());
  EPET_TRY(exclusive_scan_i32_to_i64(ctx, ns, B->gstep, B->G, &B->nsteps));
  if (M->nnz < BRK_MIN_ENTRIES * B->nsteps || B->nsteps == 0) {
    *unfit = true;
    return EPET_OK;
  }
  EPET_HIP(hipMemcpyAsync(B->gstep + B->G, &B->nsteps, sizeof(int64_t), hipMemcpyHostToDevice, st));
  const size_t rec_bytes = sizeof(unsigned) * BRK_REC * (B->nsteps / BRK_PAD);
  alloc(&B->rec, rec_bytes);
  if (!ok) {
    EPET_HIP(hipStreamSynchronize(st));
    return EPET_OK;
  }
  brk_zero(st, B->rec, rec_bytes);
  k_brk_masks<<<B->G, BRK_BUILD, lds, st>>>(nwords, B->rowperm, M->rowptr, M->col, cpos_d, B->gstep,
                                            B->rec);
  k_brk_offsets<<<B->G, BRK_BUILD, 0, st>>>(B->gstep, B->rec, ne);
  EPET_HIP(hipGetLastError());
  EPET_TRY(exclusive_scan_i32_to_i64(ctx, ne, B->gent, B->G, &B->nent));
  EPET_CHECK(B->nent >= M->nnz && B->nent <= 2 * M->nnz + 7 * B->nsteps, EPET_ERR_STATE,
             "bricks: entry count mismatch");
  const long long vstride = B->nent + BRK_TAIL;
  alloc(&B->val, sizeof(uint16_t) * B->parts * vstride);
  if (!ok) return EPET_OK;
  brk_zero(st, B->val, sizeof(uint16_t) * B->parts * vstride);
  brk_zero(st, ns, sizeof(int));
  if (M->value_type == EPET_VAL_F32)
    k_brk_values<float><<<B->G, BRK_BUILD, lds, st>>>(nwords, M->value_type, B->parts, B->rowperm,
                                                      M->rowptr, M->col, (const float*)M->val,
                                                      cpos_d, B->gstep, B->gent, B->rec,
                                                      B->val, vstride, ns);
  else
    k_brk_values<uint16_t><<<B->G, BRK_BUILD, lds, st>>>(nwords, M->value_type, B->parts,
                                                         B->rowperm, M->rowptr, M->col,
                                                         (const uint16_t*)M->val, cpos_d, B->gstep,
                                                         B->gent, B->rec, B->val, vstride, ns);
  EPET_HIP(hipGetLastError());
  int out_of_range = 0;
  EPET_TRY(read_pinned(ctx, &out_of_range, ns, sizeof(int)));
  if (out_of_range) {
    *unfit = true;
    return EPET_OK;
  }
  own.b = nullptr;
  *out = B;
  return EPET_OK;
}

// ------------------------------------------------------------------ launch
static BrkVec* brk_vec(const BrkCopy* B, int Fp) {
  for (BrkVec* v = B->vec; v; v = v->next)
    if (v->Fp == Fp) return v;
  return nullptr;
}

// gathered vector of B for Fp frames, zero where nothing is written
static int brk_vec_ensure(epet_ctx* ctx, BrkCopy* B, int Fp, bool* ok) {
  *ok = true;
  if (brk_vec(B, Fp)) return EPET_OK;
  const size_t bytes = sizeof(float) * (size_t)B->npos * Fp;
  float* x = nullptr;
  // 32-bit byte offsets in the kernel
  if (bytes >= (4ull << 30) || dev_malloc((void**)&x, bytes) != hipSuccess) {
    (void)hipGetLastError();
    *ok = false;
    return EPET_OK;
  }
  brk_zero(ctx->stream, x, bytes);
  BrkVec* v = new BrkVec();
  v->Fp = Fp;
  v->x = x;
  v->next = B->vec;
  B->vec = v;
  EPET_HIP(hipGetLastError());
  EPET_HIP(hipStreamSynchronize(ctx->stream));
  return EPET_OK;
}

// Room for `need` partial sums; a block that is there stays when there is no memory
// for a larger one.
static bool brk_partial_ensure(BrkCopy* B, long long need) {
  if (need <= B->partial_len) return true;
  float* p = nullptr;
  if (dev_malloc((void**)&p, sizeof(float) * (size_t)need) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (B->partial) (void)dev_free(B->partial);
  B->partial = p;
  B->partial_len = need;
  return true;
}
static long long brk_partials(const BrkCopy* B, int splits, int Fp) {
  return splits > 1 ? (long long)splits * B->mpos * Fp : 0;
}
// The partial sums of the launch shapes in use alone (what tuning asked for beyond
// them is given back; no memory for the smaller block leaves the larger).
static void brk_partial_fit(BrkCopy* B) {
  long long need = 0;
  for (int s = 0; s < 4; s++)
    if (B->tuned[s]) need = std::max(need, brk_partials(B, B->splits[s], 8 << s));
  if (need >= B->partial_len) return;
  float* p = nullptr;
  if (need > 0 && dev_malloc((void**)&p, sizeof(float) * (size_t)need) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  (void)dev_free(B->partial);
  B->partial = p;
  B->partial_len = need;
}

template <int NA, int FP>
static void brk_launch_t(epet_ctx* ctx, BrkArgs a) {
  const int mode = a.mode;
  if (a.splits > 1) a.mode = 2;
  const long long items = (long long)a.G * a.splits;
  const long long blocks = (items + BRK_WAVES - 1) / BRK_WAVES;
  const unsigned grid = (unsigned)((blocks + 7) / 8 * 8);
  k_brk<NA, FP><<<grid, BRK_WAVES * WAVE, 0, ctx->stream>>>(a);
  if (a.splits > 1) {
    a.mode = mode;
    k_brk_reduce<FP><<<grid_for((long long)a.mpos * FP, 256, 8ll * ctx->num_cus), 256, 0,
                       ctx->stream>>>(a);
  }
}

template <int NA>
static void brk_launch_p(epet_ctx* ctx, int Fp, const BrkArgs& a) {
  switch (Fp) {
    case 8: brk_launch_t<NA, 8>(ctx, a); break;
    case 16: brk_launch_t<NA, 16>(ctx, a); break;
    case 32: brk_launch_t<NA, 32>(ctx, a); break;
    default: brk_launch_t<NA, 64>(ctx, a); break;
  }
}

static int brk_launch(epet_ctx* ctx, const BrkCopy* B, int Fp, BrkArgs& a) {
  a.G = B->G;
  a.mpos = B->mpos;
  a.gstep = B->gstep;
  a.gent = B->gent;
  a.rec = B->rec;
  a.val = B->val;
  a.vstride = B->nent + BRK_TAIL;
  a.rowperm = B->rowperm;
  switch (B->parts) {
    case 1: brk_launch_p<1>(ctx, Fp, a); break;
    case 2: brk_launch_p<2>(ctx, Fp, a); break;
    default: brk_launch_p<3>(ctx, Fp, a); break;
  }
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

// One product of MLEM (o: the other direction's bricks): mode 0 the forward step,
// mode 1 the back projection.
static int brk_product(epet_ctx* ctx, const BrkCopy* B, const BrkCopy* o, int Fp, int splits,
                       int mode, const MfArgs& m, const float* rowscale) {
  EPET_CHECK(splits <= 1 || (B->partial && B->partial_len >= brk_partials(B, splits, Fp)),
             EPET_ERR_STATE, "bricks: partial buffer missing");
  EPET_CHECK(brk_vec(B, Fp) && brk_vec(o, Fp), EPET_ERR_STATE, "bricks: gathered vector missing");
  EPET_CHECK(mode != 0 || o->npos >= B->mpos, EPET_ERR_STATE,
             "bricks: the gathered vector is shorter than the row groups");
  BrkArgs a{};
  a.F = m.F;
  a.splits = splits;
  a.mode = mode;
  a.x = brk_vec(B, Fp)->x;
  a.flag = B->flag;
  a.partial = B->partial;
  a.itp = m.itp;
  a.alpha = 1.0f;
  a.down = mode == 0 ? 1.0f / BRK_UP : 1.0f;   // the image by k_brk_gather, the ratio as it is
  if (mode == 0) {
    a.xin = m.x;
    a.colinv = B->colinv;
    a.oute = brk_vec(o, Fp)->x;
    a.oflag = o->flag;
    a.rowscale = rowscale;
    a.fold = rowscale ? 1 : 0;
    a.Y = m.y;
    a.ll = m.loglik ? B->ll : nullptr;
  } else {
    a.clear = o->flag;
    a.out = m.c;
    a.ll = m.loglik ? o->ll : nullptr;
    a.loglik = m.loglik;
  }
  return brk_launch(ctx, B, Fp, a);
}

static int brk_gather(epet_ctx* ctx, const BrkCopy* B, int Fp, int F, float* xs, const float* x,
                      const float* scale, unsigned long long* flag, unsigned long long* clear) {
  const int nq = B->npos / 4;
  const unsigned g = grid_for((long long)nq * Fp, 256, 1ll << 31);
  switch (Fp) {
    case 8: k_brk_gather<8><<<g, 256, 0, ctx->stream>>>(xs, x, scale, B->colinv, nq, F, flag, clear); break;
    case 16: k_brk_gather<16><<<g, 256, 0, ctx->stream>>>(xs, x, scale, B->colinv, nq, F, flag, clear); break;
    case 32: k_brk_gather<32><<<g, 256, 0, ctx->stream>>>(xs, x, scale, B->colinv, nq, F, flag, clear); break;
    default: k_brk_gather<64><<<g, 256, 0, ctx->stream>>>(xs, x, scale, B->colinv, nq, F, flag, clear); break;
  }
  EPET_HIP(hipGetLastError());
  return EPET_OK;
}

static int brk_gather_x(epet_ctx* ctx, const BrkCopy* f, const BrkCopy* b, int Fp, const MfArgs& m) {
  return brk_gather(ctx, f, Fp, m.F, brk_vec(f, Fp)->x, m.x, nullptr, f->flag, b->flag);
}

// Builds the bricks of A and of its transposed copy once (allocates and
// synchronises), where the matrix knows its
// channels and grid (what makes neighbours of rows and columns).  Nothing is
// built when the bricks would be too empty or memory is short; short of memory it is
// tried again once clearly more is available.  Two threads may ask at once.
static std::mutex g_brk_build;
static bool brk_wanted(const epet_matrix* A, int F) {
  return A->tr && F >= 2 && F <= 64 && A->cols_strict && A->m > 0 && A->n > 0 && A->row_ids &&
         A->mg.n1y != 0 && (long long)A->mg.nx * A->mg.ny * A->mg.nz == A->n;
}
static int brk_build_both(epet_ctx* ctx, epet_matrix* A) {
  std::lock_guard<std::mutex> lock(g_brk_build);
  epet_matrix* At = A->tr;
  if (A->brk_state.load() != 0) return EPET_OK;
  const unsigned long long available = dev_available();
  if (!memory_worth_trying(available, A->brk_short.load())) return EPET_OK;
  if (available < bricks_at_least(A->nnz, brk_parts(A->value_type))) {
    A->brk_short.store(std::max(1ull, available));
    return EPET_OK;
  }
  bool unfit = false;
  int rc = EPET_OK;
  try {
    std::vector<int> ids(A->m);
    EPET_HIP(hipMemcpy(ids.data(), A->row_ids, sizeof(int) * A->m, hipMemcpyDeviceToHost));
    const std::vector<int> ch = channel_order(A->mg, ids);
    const std::vector<int> vx = brk_voxel_positions(A->mg);
    rc = brk_build(ctx, A, ch, vx, &A->brk, &unfit);
    if (rc == EPET_OK && A->brk) rc = brk_build(ctx, At, vx, ch, &At->brk, &unfit);
  } catch (const std::bad_alloc&) {
    // no host memory for the orders: the other kernels need none
  }
  const bool ok = rc == EPET_OK && A->brk && At->brk;
  if (!ok) {
    brk_release(A);
    brk_release(At);
  }
  A->brk_state.store(ok ? 1 : unfit ? -1 : 0);
  if (!ok && !unfit) A->brk_short.store(std::max(1ull, available));
  return rc;
}

int brk_prepare(epet_ctx* ctx, epet_matrix* A, int F) {
  if (!brk_wanted(A, F)) return EPET_OK;
  EPET_TRY(brk_build_both(ctx, A));
  if (A->brk_state.load() != 1) return EPET_OK;
  bool ok = true;
  EPET_TRY(brk_vec_ensure(ctx, A->brk, brk_pad(F), &ok));
  if (ok) EPET_TRY(brk_vec_ensure(ctx, A->tr->brk, brk_pad(F), &ok));
  return EPET_OK;
}

// Whether Y = A X is the faster one by the rows (k_spmm_n) than on bricks.  Bricks
// take 33 to 35 us of launches and working memory and 2 to 4 ps an entry, whatever
// the frames up to 16.  By the rows, a row is a wavefront's, F of its entries' frames
// at a time, so that few long rows wait for one load after the other (0.4 us each);
// else an entry and frame take 2 to 3 ps, 0.7 to 0.8 where the gathered vector stays
// near.  Rows / bricks in us, FP32: 9,001 rows, 0.49M entries, 16^3 voxels, 8 frames
// 6 / 34; 0.90M, 64 frames 46 / 39; 700 rows, 0.60M, 52^3, 4 frames 17 / 33, 16 frames
// 83 / 33; 4.4M, 2 frames 32 / 51, 4 frames 55 / 51; 18.5M, 2 frames 87 / 97, 3 frames
// 156 / 94; 48.8M, 2 frames 197 / 156.
// The back projection by the rows adds with float atomics, several times further from
// the exact sums (4e-7 against 1.1e-7, 50,000 rows of 899 entries), and stays on bricks.
static bool brk_rows_faster(const epet_matrix* A, int F) {
  const double e = 1e-6 * (double)A->nnz;
  int P = 2;
  while (P < F) P *= 2;
  const double serial = 0.4 / WAVE * P * (double)A->nnz / A->m;
  const double rows = 5.0 + std::max(serial, e * F * (A->n < 32768 ? 0.8 : 2.5));
  return rows < 35.0 + e * (1.5 + 0.7 * brk_parts(A->value_type));
}

// Y = alpha op(A) X + beta Y on bricks: *done = false where they do not apply.
// The bricks are built for a matrix with a transposed copy (a program that
// back-projects several frames again and again) once its products come to
// BRK_WORK entries x frames per row and column, unless they would take more than
// a quarter of the free memory or the stream is being captured.  The build takes
// 40 ns per row and column (5 to 8 ms for 50,000 to 139,000 rows and 52^3
// voxels), most of it ordering on the host: products of BRK_WORK pay it back in
// about 10 calls, and 8 rays on 52^3 (100 entries a row, 0.05 to 0.2 ms a
// product, bricks too empty in the end) would lose 2 ms on the first one.
// Working memory is the call's own, so calls on several streams do not meet.
// 4 images on 50,000 rows of 899 entries, FP32 values: 0.17 ms either way against
// 0.34 ms (k_spmm_n) and 1.02 ms (k_spmm_t, float atomics in memory).
constexpr long long BRK_WORK = 500;
int brk_spmm(epet_ctx* ctx, const epet_matrix* cA, int op, int F, float alpha, const float* X,
             float beta, float* Y, bool* done) {
  *done = false;
  epet_matrix* A = const_cast<epet_matrix*>(cA);
  // (bricks of a matrix whose arrays a caller holds may be out of date)
  if (!brk_wanted(A, F) || A->brk_state.load() < 0 || A->exposed.load()) return EPET_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(ctx->stream, &cap) != hipSuccess) {
    (void)hipGetLastError();
    return EPET_OK;
  }
  if (cap != hipStreamCaptureStatusNone) return EPET_OK;
  if (A->brk_state.load() == 0) {
    const long long work = A->nnz * F;
    if (A->brk_work.fetch_add(work) + work < BRK_WORK * ((long long)A->m + A->n)) return EPET_OK;
    // values with a quarter of padding, records, and as much again while building
    const double need = (double)A->nnz * 2.0 * (2.5 * brk_parts(A->value_type) + 4.0);
    if (need > 0.25 * (double)dev_available()) return EPET_OK;
    EPET_TRY(brk_build_both(ctx, A));
    if (A->brk_state.load() != 1) return EPET_OK;
  }
  if (op == EPET_OP_N && brk_rows_faster(A, F)) return EPET_OK;
  const BrkCopy* B = op == EPET_OP_N ? A->brk : A->tr->brk;
  const int Fp = brk_pad(F);
  // about 14,000 wavefronts (3.5 rounds of 16 per CU) measured best over the
  // series in perf/cases.py, no finer than two batches of steps each
  int splits = 1;
  while (splits < 64 && (long long)B->G * splits * 3 < 28000 && B->nsteps >= 8ll * B->G * splits)
    splits *= 2;
  const size_t xb = (sizeof(float) * (size_t)B->npos * Fp + 255) & ~(size_t)255;
  const size_t pb = splits > 1 ? sizeof(float) * (size_t)splits * B->mpos * Fp : 0;
  if (xb >= (4ull << 30)) return EPET_OK;   // 32-bit byte offsets in the kernel
  StreamTemps tmp(ctx->stream);
  unsigned char* w = nullptr;
  if (tmp.alloc(&w, 256 + xb + pb) != hipSuccess) {
    (void)hipGetLastError();
    return EPET_OK;
  }
  auto* flag = reinterpret_cast<unsigned long long*>(w);
  float* xs = reinterpret_cast<float*>(w + 256);
  brk_zero(ctx->stream, flag, 16);
  EPET_TRY(brk_gather(ctx, B, Fp, F, xs, X, op == EPET_OP_T ? A->rowscale : nullptr, flag, nullptr));
  BrkArgs a{};
  a.F = F;
  a.splits = splits;
  a.mode = 1;
  a.x = xs;
  a.down = 1.0f / BRK_UP;
  a.xin = X;
  a.colinv = B->colinv;
  a.xscale = op == EPET_OP_T ? A->rowscale : nullptr;
  a.flag = flag;
  a.partial = reinterpret_cast<float*>(w + 256 + xb);
  a.out = Y;
  a.alpha = alpha;
  a.beta = beta;
  a.rowscale = op == EPET_OP_N ? A->rowscale : nullptr;
  EPET_TRY(brk_launch(ctx, B, Fp, a));
  *done = true;
  return EPET_OK;
}

bool brk_built(const epet_matrix* A, int F) {
  return A->tr && F >= 2 && F <= 64 && A->brk_state.load() == 1 && brk_vec(A->brk, brk_pad(F)) &&
         brk_vec(A->tr->brk, brk_pad(F));
}

bool brk_ready(const epet_matrix* A, int F) {
  if (!brk_built(A, F)) return false;
  const int s = brk_slot(brk_pad(F));
  for (const BrkCopy* B : {A->brk, A->tr->brk})
    if (B->tuned[s] != F || B->partial_len < brk_partials(B, B->splits[s], brk_pad(F))) return false;
  return true;
}

// One multi-frame iteration's products (allocates nothing once prepared and tuned).
int brk_iteration(epet_ctx* ctx, const epet_matrix* A, const MfArgs& m) {
  const int Fp = brk_pad(m.F), s = brk_slot(Fp);
  const BrkCopy *f = A->brk, *b = A->tr->brk;
  EPET_TRY(brk_gather_x(ctx, f, b, Fp, m));
  EPET_TRY(brk_product(ctx, f, b, Fp, f->splits[s], 0, m, A->rowscale));
  EPET_TRY(brk_product(ctx, b, f, Fp, b->splits[s], 1, m, nullptr));
  return EPET_OK;
}

// Splits of a group's steps, per direction: enough wavefronts to fill the chip
// against partial sums to add, by time.  Tried are splits of two batches of steps
// and more whose partial sums take up to BRK_TRY_BYTES: 64 frames of 3.3M rows in 64
// parts, the limit by steps alone, would take 55 GB to find that one part is best.
// (A limit at 65,536 wavefronts instead left the back projection of 3.3M rows 16 parts
// for 32 to 64, and so longer FP32 sums: 2.4e-6 from 64 bits after 20 iterations of 32
// frames against 1.0e-6 to 1.5e-6.)
constexpr long long BRK_TRY_BYTES = 4ll << 30;
static int brk_most_splits(const BrkCopy* B, int Fp) {
  int most = 1;
  while (most < 64 && B->nsteps >= 8ll * B->G * most &&
         (long long)sizeof(float) * brk_partials(B, 2 * most, Fp) <= BRK_TRY_BYTES)
    most *= 2;
  return most;
}
int brk_tune(epet_ctx* ctx, epet_matrix* A, const MfArgs& m, int reps) {
  const int Fp = brk_pad(m.F), s = brk_slot(Fp);
  BrkCopy* dirs[2] = {A->brk, A->tr->brk};
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    if (e0) (void)hipEventDestroy(e0);
    return fail(EPET_ERR_HIP, __FILE__, __LINE__, "tuning events");
  }
  int rc = brk_gather_x(ctx, dirs[0], dirs[1], Fp, m);
  for (int d = 0; d < 2 && rc == EPET_OK; d++) {
    BrkCopy* B = dirs[d];
    float best = 1e30f;
    int most = brk_most_splits(B, Fp);
    while (most > 1 && !brk_partial_ensure(B, brk_partials(B, most, Fp))) most /= 2;
    for (int splits = 1; splits <= most && rc == EPET_OK; splits *= 2) {
      auto run = [&]() {
        MfArgs q = m;
        q.loglik = nullptr;
        return brk_product(ctx, B, dirs[1 - d], Fp, splits, d, q, d == 0 ? A->rowscale : nullptr);
      };
      rc = run();
      if (rc == EPET_OK && hipEventRecord(e0, ctx->stream) != hipSuccess)
        rc = fail(EPET_ERR_HIP, __FILE__, __LINE__, "tuning events");
      for (int r = 0; r < reps && rc == EPET_OK; r++) rc = run();
      float ms = 0.0f;
      if (rc == EPET_OK &&
          (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
           hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
        rc = fail(EPET_ERR_HIP, __FILE__, __LINE__, "tuning events");
      ms /= reps;
      if (rc == EPET_OK && ms < best) {
        best = ms;
        B->splits[s] = splits;
      }
    }
    B->ms[s] = best;
    B->tuned[s] = m.F;
    brk_partial_fit(B);
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

// {1, padded frames, parts of a stored value, rows per group, splits} of the
// forward product and {rows per group, splits} of the back projection, entries
// per step of both, and the tuned times; {0} when not in use
int brk_info(const epet_matrix* A, int F, int info[9], float ms[2]) {
  for (int i = 0; i < 9; i++) info[i] = 0;
  ms[0] = ms[1] = 0.0f;
  if (!brk_ready(A, F)) return EPET_OK;
  const int Fp = brk_pad(F), s = brk_slot(Fp);
  const BrkCopy *f = A->brk, *b = A->tr->brk;
  info[0] = 1;
  info[1] = Fp;
  info[2] = f->parts;
  info[3] = BRK_ROWS;
  info[4] = f->splits[s];
  info[5] = (int)(A->nnz / std::max(1ll, f->nsteps));
  info[6] = (int)(A->nnz / std::max(1ll, b->nsteps));
  info[7] = BRK_ROWS;
  info[8] = b->splits[s];
  ms[0] = f->ms[s];
  ms[1] = b->ms[s];
  return EPET_OK;
}

}  // namespace epet
