// bf16 / fp16 MFMA kernels (gfx950, wave64).  The arithmetic is laid out for d = e = W, W = 128 or 64.
// Three instantiations of every kernel and width: M_ALIGNED (chunk length a multiple of 64), M_RAGGED
// (one partial last block) and M_NARROW (rows of d, e < W features, multiples of 8, read
// zero-extended to W and written back at their own width; any chunk length).
//
// A sweep (`sweep_body` for W = 128, `ws_body` for W = 64) evaluates a causal (or anti-causal) decayed linear
// attention over a segment of 64-token blocks given the state entering it:
//
//   causal       out_a = sum_{b<=a} l^(a-b) (x_a . y_b) z_b + l^a      x_a St
//                St   <- l^64 St + sum_b l^(64-b) y_b^T z_b           (blocks ascending)
//   anti-causal  out_a = sum_{b>=a} l^(b-a) (x_a . y_b) z_b + l^(64-a) x_a St
//                St   <- l^64 St + sum_b l^b      y_b^T z_b           (blocks descending)
//
// (a, b: token index inside the block; St is W x W, rows = features of y,
// columns = features of z.)  The four outputs of the operator are instances:
//   O  : x=Q  y=K  z=V   causal       St = KV            lasp/lasp_fuse.py:104-124
//   dQ : x=dO y=V  z=K   causal       St = KV^T          lasp/lasp_fuse.py:237-260
//   dV : x=K  y=Q  z=dO  anti-causal  St = DKV           lasp/lasp_fuse.py:340-350
//   dK : x=V  y=dO z=Q   anti-causal  St = DKV^T         lasp/lasp_fuse.py:333-350
// `la_seg_state` computes a segment's own contribution to St (the pre-pass whose
// results the decayed scan stitches together).
//
// Work split inside a 512-thread workgroup (8 waves): four "math" waves own the state and the output (W = 128: wave w columns
// [32w, 32w+32), as four 32x32 fp32 MFMA accumulator tiles that never leave registers) and four "feed" waves see to the
// blocks to come, compute the 64x64 score tile (one 32x32 quadrant per wave; masked, rounded to 16 bits and shared through
// LDS) and store the outputs.  All products are arranged so that an accumulator tile can be fed back as an MFMA operand
// without a shuffle: v_mfma_f32_32x32x16_bf16 leaves C[8g+4hh+r][c] in register 4g+r of lane (c, hh) -- four consecutive
// rows per lane -- and the contraction index of the following product is permuted to match on both operands.
#include <type_traits>

#include "lasp_common.h"

namespace lasp {
namespace {

// native vector types (HIP's uint4 / uint2 structs copy through memcpy, which can pin
// a register array to scratch memory)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef uint16_t elem16_t;  // raw bits of one bf16 or fp16 element

constexpr int BLK = 64;     // tokens per block
constexpr float LOG2E = kLog2e;
constexpr float SKIP_LOG2 = kSkipLog2;  // decay weights below 2^-SKIP_LOG2 are treated as zero (see la_seg_state)
enum Mode { M_ALIGNED = 0, M_RAGGED = 1, M_NARROW = 2, M_ADDING = 3 };
// where a sweep takes the state entering its segment from (see ws_body)
enum Source { SRC_SCANNED = 0, SRC_WALK = 1, SRC_COMBINE = 2 };

// Element policies: the kernels move 16-bit elements as raw bits and only touch their value
// in three places -- widening one element, rounding two floats into a packed pair, and the
// MFMA itself.
struct ElemBF16 {
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
    float2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  }
  // `word` holds the element in its low (odd = false) or high (odd = true) half
  static __device__ __forceinline__ float widen(uint32_t word, bool odd) {
    return __uint_as_float(odd ? (word & 0xffff0000u) : (word << 16));
  }
  static __device__ __forceinline__ floatx16 mfma(u32x4 a, u32x4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
  }
};
struct ElemF16 {
  static __device__ __forceinline__ uint32_t pack(float lo, float hi) {
    float2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
  }
  static __device__ __forceinline__ float widen(uint32_t word, bool odd) {
    const f16x2_t h = __builtin_bit_cast(f16x2_t, word);
    return (float)(odd ? h.y : h.x);
  }
  static __device__ __forceinline__ floatx16 mfma(u32x4 a, u32x4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
  }
};

// A pointer that is the same for every lane, moved to scalar registers: loads through it then take
// the form scalar base + 32-bit lane offset + immediate, instead of a 64-bit address per lane that
// the loop optimiser would otherwise carry (and increment) in vector registers.  The result is
// typed as a global-memory pointer, which the round trip through integers would otherwise lose.
typedef const __attribute__((address_space(1))) char *gmem_ptr;
__device__ __forceinline__ gmem_ptr uniform_ptr(const char *p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (gmem_ptr)(((uint64_t)hi << 32) | lo);
}

// Left to itself the scheduler puts every LDS read right before the product that uses it, to save registers that these
// kernels have to spare; each product then waits for a whole LDS round trip.  Nothing is moved across this line, so the reads
// above it are in flight together.
__device__ __forceinline__ void reads_first() { __builtin_amdgcn_sched_barrier(0); }
__device__ __forceinline__ u32x4 lds16(const char *p) { return *reinterpret_cast<const u32x4 *>(p); }

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 *lds_v4i16;
// The transposing 8-byte read works in groups of 16 lanes: lane i of a group receives, as element j,
// element (i % 4) of what lane (4 j + i / 4) of the group addressed.  With lane s of a group addressing
// token T + s / 4, features f + 4 (s % 4) .. + 3, lane i ends up with feature f + i of tokens T .. T + 3.
__device__ __forceinline__ u32x2 lds_tr8(const char *p) {
  const v4i16 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(p));
  return __builtin_bit_cast(u32x2, r);
}

// element x (0..7) of a 16-byte group of 16-bit elements, widened to fp32
template <class E>
__device__ __forceinline__ float elem_f32(const u32x4 &q, int x) {
  const uint32_t w = (x >> 1) == 0 ? q.x : (x >> 1) == 1 ? q.y : (x >> 1) == 2 ? q.z : q.w;
  return E::widen(w, x & 1);
}
// a 16-byte group of 16-bit elements, each times w
template <class E>
__device__ __forceinline__ u32x4 scaled(const u32x4 &q, float w) {
  u32x4 o;
  o.x = E::pack(elem_f32<E>(q, 0) * w, elem_f32<E>(q, 1) * w);
  o.y = E::pack(elem_f32<E>(q, 2) * w, elem_f32<E>(q, 3) * w);
  o.z = E::pack(elem_f32<E>(q, 4) * w, elem_f32<E>(q, 5) * w);
  o.w = E::pack(elem_f32<E>(q, 6) * w, elem_f32<E>(q, 7) * w);
  return o;
}

// l^x for x >= 0
__device__ __forceinline__ float decay(float s_log2e, float x) {
  return __builtin_amdgcn_exp2f(-s_log2e * x);
}

// A block of token rows as a buffer that ends with them: a lane that addresses past the end -- a row that a partial block
// does not have, a piece beyond a narrow row's width, a block beyond the walk's end -- reads zeros and stores nothing, with no
// branch around the access.  (Branches would cost more than themselves: where the number of accesses in flight depends on
// the path, a wait for the oldest of them has to wait for all, the stores and the loads just issued among them.)
// Offsets are 32-bit and per lane; none is larger than 2 kOutside.
constexpr uint32_t kOutside = 0x40000000u;
typedef __amdgpu_buffer_rsrc_t rows_t;
__device__ __forceinline__ rows_t rows_of(const void *p, int bytes) {
  const gmem_ptr u = uniform_ptr(reinterpret_cast<const char *>(p));
  return __builtin_amdgcn_make_buffer_rsrc((void *)(const char *)u, 0, bytes, 0x00020000);
}
struct SegWork {
  int bh, seg;
  int64_t tok0;  // first token of the segment
  int nblk;      // 64-token blocks in it, the last one possibly partial
  int tail;      // tokens in its last block (1..64); below 64 only at the end of a ragged chunk
};
// `item` enumerates (b*h, segment) pairs
__device__ __forceinline__ SegWork seg_work(const Geom &g, int item) {
  SegWork r;
  r.bh = quotient(item, g.by_seg);
  r.seg = item - r.bh * g.n_seg;
  r.tok0 = (int64_t)r.seg * g.seg_len;
  int64_t t1 = r.tok0 + g.seg_len;
  if (t1 > g.n) t1 = g.n;
  const int tokens = (int)(t1 - r.tok0);
  r.nblk = (tokens + BLK - 1) / BLK;
  r.tail = tokens - (r.nblk - 1) * BLK;
  return r;
}

// blocks over which a head's decay falls to 2^-SKIP_LOG2, or `all` where it takes that many and more
__device__ __forceinline__ int reach_of(float slope, int all) {
  const float sl = slope * LOG2E;
  if (!(sl > 0.f)) return all;
  const float x = SKIP_LOG2 / (sl * (float)BLK);
  return x < (float)all ? (int)x + 1 : all;
}
// The same of a kernel that walks to its segment (SRC_WALK): segments of equal length for heads whose decay ends the walks soon, those of
// g.cut, shorter the longer the walk before them, for the others.
__device__ __forceinline__ SegWork walk_work(const Geom &g, int item, bool rev, int reach) {
  SegWork r;
  r.bh = quotient(item, g.by_seg);
  r.seg = item - r.bh * g.n_seg;
  const int total = (int)((g.n + BLK - 1) / BLK);
  int b0, b1;
  if (reach >= g.cut.from) {
    const int j = rev ? g.n_seg - 1 - r.seg : r.seg;  // segments visited before it
    const int from = g.cut.start(j), to = j + 1 < g.n_seg ? g.cut.start(j + 1) : total;
    b0 = rev ? total - to : from;
    b1 = rev ? total - from : to;
  } else {
    b0 = quotient(r.seg * total, g.by_seg);
    b1 = quotient((r.seg + 1) * total, g.by_seg);
  }
  r.tok0 = (int64_t)b0 * BLK;
  r.nblk = b1 - b0;
  r.tail = b1 == total ? (int)(g.n - (int64_t)(total - 1) * BLK) : BLK;
  return r;
}

// ------------------------------------------------------------------------------
// Every sweep kernel below is an instance of sweep_body (W = 128) or ws_body (W = 64, where neither d nor e is larger),
// <E, REV, TRANS, SRC, MODE>.
//
// MODE.  M_RAGGED: the chunk length is not a multiple of 64, so the last block of the last segment is
// partial (rows past its end read as zeros, stores are masked, and the decay factors of that one block use
// its true length).  M_NARROW: in addition X and Y rows hold `fa` features, Z and Out rows `fb`
// (multiples of 8, at most W), read zero-extended to W and written back at their own width; math
// waves of the 128-wide form whose columns all lie in the zero extension only take part in the barriers.  The slices of a wide
// head (d > 128) run in this mode too, their rows being g.dt features apart; M_ADDING: slices after the first, which add their
// O (dV) to what the slices before left there.  M_ALIGNED carries none of that bookkeeping; fa and fb are read from M_NARROW on.
//
// SRC says where the state entering the segment comes from.
// SRC_SCANNED: `states` holds it, left there by the decayed scan over the segments' own states.
// SRC_COMBINE: `states` holds the segments' OWN states as the pre-pass wrote them, and the
//   workgroup runs the scan's recurrence itself over the segments before (after) its own,
//   starting from the chunk's incoming state `carry_in` (d x e floats per (b, h), may be NULL):
//   St <- l^len_j St + own_j.  With few segments that is cheaper than a scan launch.
// SRC_WALK: no workspace at all: the state is rebuilt by first walking the blocks that precede the
//   segment (follow it, going backwards) and only updating the state: no X tile, no score, no
//   output.  The walk starts from `carry_in`, or from zero as many blocks back as the head's decay
//   reaches (weights below 2^-SKIP_LOG2 are dropped).  One launch then does a whole chunk; the
//   repeated walks make it a tool for short chunks.  In the 128-wide dQ sweep `carry_in` may be the states that
//   the forward's scan left (g.kept): it then starts from the one among them that entered the chunk.
// In the last two the workgroup of the segment visited last writes the state it ends with to
// `carry_out` (non-transposed roles only).
// ------------------------------------------------------------------------------
// The 64-wide sweep.  512 threads, two workgroups per CU, the work of a block split between two groups of waves (a workgroup
// whose waves all run fill -> products -> store one after the other spends most of a block waiting for its own LDS round trips):
//   waves 0-3 ("feed"): global loads, the LDS tiles of the NEXT block (waves 0, 1 fetch Y, waves 2, 3 Z, which they also write
//     scaled by the state update's decay), the masked score tile of the current block, the coalesced output stores;
//   waves 4-7 ("math"): state term, intra-block term, state update, output staging.  Wave 4 + w owns one 32 x 32 tile of the
//     output -- columns [32 (w & 1), + 32) of tokens [32 (w >> 1), + 32) -- and the 64 x 32 state columns it needs (both token
//     halves keep those: 8 products per block and wave, against a reduction through LDS).
// All tiles are token-major; what contracts over tokens is read transposed.  They are double-buffered (two sets of X, Y, Z and scaled
// Z, 73 728 B with the score tile), and a block takes two barriers:
//     feed: store O(t-1), score(t),   | math: state term(t), state update(t)
//           fill Y, Z(t+1),           |
//           issue loads Y, Z(t+2)     |
//   ---- barrier ----
//     feed: fill X(t+1),              | math: intra(t) from the score tile, stage O(t) into the X tile of block t
//           issue loads X(t+2)        |       (no longer read)
//   ---- barrier ----
// O(t-1) waits in the X tile of the set that the fill of X(t+1) overwrites after the first barrier; the set's other tiles
// were last read before the second barrier of block t-1.  Both groups run their own loop; each executes exactly
// 1 + 2 * nblk barriers.  At most 128 registers, so that two workgroups share a CU and fill each other's waits; bound by HBM on
// long chunks.  In us, with tiles transposed in registers on the way to LDS and as it is: backward sweep, b*h = 24, n = 2048:
// 14.0 and 12.8, b*h = 16, n = 16384: 54.2 and 51.8, b*h = 64, n = 4096: 54.8 and 52.5; one launch for b*h = 96, n = 512:
// 17.1 and 16.8 (forward 10.2 and 9.9).  The 128-wide form's pipeline, whose math waves scale Z themselves, twice here, took 56 to 59 for
// b*h = 64 where this one takes 52.5.
constexpr int WS_THREADS = 512;
struct WsLds {
  static constexpr int W = 64, ROW = 2 * W, TILE = BLK * ROW;
  static constexpr int X = 0, Y = TILE, Z = 2 * TILE, ZS = 3 * TILE, SET = 4 * TILE;  // one block's tiles; ZS: Z scaled
  static constexpr int SC = 2 * SET, SC_ROW = 2 * BLK;  // the score tile
  static constexpr int BYTES = SC + BLK * SC_ROW;       // 73 728 B: two workgroups per CU
  // Unit u (16 bytes) of row r lies at u ^ swizzle(r): the rows that a phase of a 16-byte read takes one unit of, and the four rows
  // x 64 bytes that half a wave reads transposed, fall on disjoint banks (two rows to a set of banks).
  static __device__ __forceinline__ int swizzle(int row) { return ((row & 2) << 1) | ((row >> 2) & 3); }
};
// workgroups of a sweep that share a CU, and with them the waves per SIMD the registers must leave room for
constexpr int ws_waves_per_simd(int w) { return w == 64 ? 4 : 1; }

template <class E, bool REV, bool TRANS, int SRC, int MODE>
__device__ __forceinline__ void
ws_body(const elem16_t *__restrict__ X, const elem16_t *__restrict__ Y, const elem16_t *__restrict__ Z,
        const float *__restrict__ S, const float *__restrict__ states, elem16_t *__restrict__ Out, const Geom &g,
        int fa, int fb, int item, char *smem, const float *__restrict__ carry_in,
        float *__restrict__ carry_out = nullptr) {
  constexpr bool RAGGED = MODE != M_ALIGNED, NARROW = MODE == M_NARROW;
  constexpr bool LEAVES_STATE = SRC != SRC_SCANNED;  // the sweep's final state is the chunk's outgoing one
  using L = WsLds;
  constexpr int W = L::W;
  constexpr int NT = W / 32;  // 32-row tiles of a wave's state columns
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = w8 & 3;                   // feed: score quadrant
  const int wcol = w & 1, ih = w >> 1;    // math: column block and token half
  const int c = lane & 31, hh = lane >> 5;

  const int bh = quotient(item, g.by_seg), head = bh - quotient(bh, g.by_h) * g.h;
  const int total_blk = (int)((g.n + BLK - 1) / BLK);  // blocks in the chunk
  float slope = 0.f;
  int reach = 0;
  if (SRC == SRC_WALK) {
    slope = S[head];
    reach = __builtin_amdgcn_readfirstlane(reach_of(slope, total_blk));
  }
  const SegWork sw = SRC == SRC_WALK ? walk_work(g, item, REV, reach) : seg_work(g, item);
  const int64_t row0 = (int64_t)sw.bh * g.n + sw.tok0;
  // elements from row to row of X and Y, and of Z and Out: q, k and their gradients have rows of g.dt features, of which
  // a slice of a wide head reads and writes fa (fb)
  const int xp = NARROW ? (TRANS ? g.e : g.dt) : W, zp = NARROW ? (TRANS ? g.dt : g.e) : W;
  const int nblk = sw.nblk;
  const int step = REV ? -1 : 1;
  const int blk0 = REV ? nblk - 1 : 0;

  // SRC_WALK: the state entering the segment is rebuilt by walking `runup` blocks outside it first (before it,
  // or after it going backwards), as far as the head's decay reaches, from the chunk's incoming state if the
  // walk gets to the chunk's end, else from zero.  Blocks are numbered relative to the segment; walk and sweep
  // form one run of runup + nblk blocks, first_blk, first_blk + step, ..., of which the first `runup` only
  // update the state (one barrier each, both groups).
  const int seg_blk0 = (int)(sw.tok0 / BLK);           // the segment's first block
  const int chunk_tail = (int)(g.n - (int64_t)(total_blk - 1) * BLK);
  // tokens in a block (numbered relative to the segment): a partial block is the chunk's last one
  auto len_of = [&](int blk) __attribute__((always_inline)) {
    if (!RAGGED) return BLK;
    return seg_blk0 + blk == total_blk - 1 ? chunk_tail : BLK;
  };
  int runup = 0;
  bool take_carry = false;
  if (SRC == SRC_WALK) {
    const int avail = REV ? total_blk - (seg_blk0 + nblk) : seg_blk0;
    runup = min(reach, avail);
    take_carry = carry_in != nullptr && runup == avail;
  }
  const int first_blk = blk0 - runup * step;
  const int run = runup + nblk;  // blocks in the whole run

  if (w8 < 4) {
    // ================================ feed waves ================================
    const int ftid = tid;  // 0..255
    const bool zfeed = w8 >= 2;  // a wave fetches Y or Z, not both
    // 16 bytes per thread and row: rows xr and xr + 32 of X, yr + 16 r of Y or Z
    const int unit = ftid & 7, xr = ftid >> 3, yr = (ftid & 127) >> 3;
    const int yp = zfeed ? zp : xp, yw = zfeed ? fb : fa;
    uint32_t x_off[2], y_off[4], o_off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x_off[i] = !NARROW || unit * 8 < fa ? (uint32_t)((xr + 32 * i) * xp * 2 + unit * 16) : kOutside;
      o_off[i] = !NARROW || unit * 8 < fb ? (uint32_t)((xr + 32 * i) * zp * 2 + unit * 16) : kOutside;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      y_off[r] = !NARROW || unit * 8 < yw ? (uint32_t)((yr + 16 * r) * yp * 2 + unit * 16) : kOutside;
    const int x_to = xr * L::ROW + ((unit ^ L::swizzle(xr)) << 4), y_to = yr * L::ROW + ((unit ^ L::swizzle(yr)) << 4);
    const elem16_t *Xg = X + row0 * xp, *Yg = zfeed ? Z + row0 * zp : Y + row0 * xp;
    elem16_t *Og = Out + row0 * zp;

    u32x4 nx[2], ny[4];  // the block in flight; ny: Y or Z
    // block k of the run as a buffer; none of its rows where it is not `wanted`
    auto rows = [&](const elem16_t *base, int k, int pitch, bool wanted) __attribute__((always_inline)) {
      const int blk = first_blk + k * step;
      return rows_of(base + (int64_t)blk * BLK * pitch, wanted ? len_of(blk) * pitch * 2 : 0);
    };
    // Always the same number of loads (see rows_of); walk blocks (k < runup) need no X tile
    auto issue_x = [&](int k) __attribute__((always_inline)) {
      const rows_t x = rows(Xg, k, xp, k < run && (SRC != SRC_WALK || k >= runup));
#pragma unroll
      for (int i = 0; i < 2; ++i) nx[i] = __builtin_amdgcn_raw_buffer_load_b128(x, (int)x_off[i], 0, 0);
    };
    auto issue_yz = [&](int k) __attribute__((always_inline)) {
      const rows_t y = rows(Yg, k, yp, k < run);
#pragma unroll
      for (int r = 0; r < 4; ++r) ny[r] = __builtin_amdgcn_raw_buffer_load_b128(y, (int)y_off[r], 0, 0);
    };
    // The slope comes as a lane's load in front of the first block's: as a scalar one, whose waits know no order, it would
    // have to arrive before the first of these loads could leave.
    int lane_head = head;
    asm volatile("" : "+v"(lane_head));
    const float slope = S[lane_head];
    issue_yz(0);
    issue_x(0);
    __builtin_amdgcn_sched_barrier(0);
    const float sl = slope * LOG2E;
    float kdec[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) kdec[r] = decay(sl, REV ? (float)(yr + 16 * r) : (float)(BLK - yr - 16 * r));
    // writes the block held in nx and ny into a tile set: X ...
    auto fill_x = [&](char *set, int k) __attribute__((always_inline)) {
      if (SRC != SRC_WALK || k >= runup) {  // a walk block is only multiplied into the state
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4 *>(set + L::X + x_to + 32 * i * L::ROW) = nx[i];
      }
    };
    // ... and Y, or Z as it is and scaled by the key decay
    auto fill_yz = [&](char *set, int k) __attribute__((always_inline)) {
      char *to = set + (zfeed ? L::Z : L::Y) + y_to;
#pragma unroll
      for (int r = 0; r < 4; ++r) *reinterpret_cast<u32x4 *>(to + 16 * r * L::ROW) = ny[r];
      if (!zfeed) return;
      const int len = len_of(first_blk + k * step);
      float kd[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) kd[r] = kdec[r];
      if (LEAVES_STATE && RAGGED && !REV && len != BLK) {
        // the chunk's partial last block, going forwards: its tokens sit `len - b` before the chunk end, which
        // matters here because the state it leaves is the outgoing one
#pragma unroll
        for (int r = 0; r < 4; ++r) kd[r] = decay(sl, (float)max(len - (yr + 16 * r), 0));
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) *reinterpret_cast<u32x4 *>(set + L::ZS + y_to + 16 * r * L::ROW) = scaled<E>(ny[r], kd[r]);
    };
    // the output tile staged in `set`'s X tile -> global rows of block k of the run
    auto store_out = [&](const char *set, int k, bool wanted) __attribute__((always_inline)) {
      const rows_t out = rows(Og, k, zp, wanted);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        __builtin_amdgcn_raw_buffer_store_b128(lds16(set + L::X + x_to + 32 * i * L::ROW), out, (int)o_off[i], 0,
                                               2 /* non-temporal */);
    };
    // this wave's quadrant of the transposed score tile: sc[4g+r] = y_b . x_a, b = 32qJ+8g+4hh+r, a = 32qI+c
    const int qI = w >> 1, qJ = w & 1;
    const bool q_active = REV ? !(qI == 1 && qJ == 0) : !(qI == 0 && qJ == 1);
    float mask[16];  // decay between the tokens of a score; negative: masked
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int a = 32 * qI + c, b = 32 * qJ + 8 * (r >> 2) + 4 * hh + (r & 3), dist = REV ? b - a : a - b;
      mask[r] = dist >= 0 ? decay(sl, (float)dist) : -1.f;
    }
    const int q_at = c * L::ROW + ((hh ^ L::swizzle(c)) << 4);
    const int sc_at = (32 * qI + c) * L::SC_ROW + ((4 * qJ ^ ((c >> 1) & 7)) << 4) + 8 * hh;
    auto score = [&](const char *set) __attribute__((always_inline)) {
      if (!q_active) return;
      floatx16 sc;
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[r] = 0.f;
      u32x4 yf[W / 16], xf[W / 16];
#pragma unroll
      for (int ks = 0; ks < W / 16; ++ks) {
        yf[ks] = lds16(set + L::Y + 32 * qJ * L::ROW + (q_at ^ (ks << 5)));
        xf[ks] = lds16(set + L::X + 32 * qI * L::ROW + (q_at ^ (ks << 5)));
      }
      reads_first();
#pragma unroll
      for (int ks = 0; ks < W / 16; ++ks) sc = E::mfma(yf[ks], xf[ks], sc);
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        float m[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) m[r] = mask[4 * gq + r] >= 0.f ? sc[4 * gq + r] * mask[4 * gq + r] : 0.f;
        u32x2 o;
        o.x = E::pack(m[0], m[1]);
        o.y = E::pack(m[2], m[3]);
        *reinterpret_cast<u32x2 *>(smem + L::SC + (sc_at ^ (gq << 4))) = o;
      }
    };

    fill_yz(smem, 0);
    issue_yz(1);
    fill_x(smem, 0);
    issue_x(1);
    __syncthreads();  // barrier 0: block 0 of the run visible
    int k = 0;
    for (; k < runup; ++k) {  // walk: the math waves multiply block k into the state meanwhile
      char *nxt = smem + ((k + 1) & 1) * L::SET;  // k + 1 < run: a sweep block follows the walk
      fill_yz(nxt, k + 1);
      issue_yz(k + 2);
      fill_x(nxt, k + 1);
      issue_x(k + 2);
      __syncthreads();  // walk barrier k
    }
    for (; k < run; ++k) {
      char *cur = smem + (k & 1) * L::SET, *nxt = smem + ((k + 1) & 1) * L::SET;
      // per block: 2 stores, 4 loads of Y or Z, 2 of X, in this order, so the waits of the fills leave what was issued
      // after their own loads in flight
      store_out(nxt, k - 1, k > runup);
      score(cur);
      if (k + 1 < run) fill_yz(nxt, k + 1);
      issue_yz(k + 2);
      __syncthreads();  // first barrier of a sweep block: score tile complete; X of `cur` and the output staged in `nxt` no longer read
      if (k + 1 < run) fill_x(nxt, k + 1);
      issue_x(k + 2);
      __syncthreads();  // second barrier: next block visible; output of this block staged
    }
    store_out(smem + ((run - 1) & 1) * L::SET, run - 1, true);
    return;
  }

  // ================================== math waves ==================================
  // (rows and columns of the state: see sweep_body)
  const int col = 32 * wcol + 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
  const float sl = S[head] * LOG2E;
  const float blockdec = decay(sl, (float)BLK);
  const int a_own = 32 * ih + c;  // the token whose output the lane holds
  const float qdec = decay(sl, REV ? (float)(BLK - a_own) : (float)a_own);
  floatx16 st[NT];
#pragma unroll
  for (int T = 0; T < NT; ++T)
#pragma unroll
    for (int r = 0; r < 16; ++r) st[T][r] = 0.f;
  // st <- f * st + M (`fresh`: st <- M, which leaves the loads in flight until a product needs them), M being the W x W fp32
  // tile whose element (row, col) is src[row * ld + col], or for a transposed role src[col * ld + row]; `bounded`: src holds
  // only fa x fb (transposed: fb x fa) elements
  auto add_state_ld = [&](const float *src, int ld, float f, bool bounded, bool fresh) __attribute__((always_inline)) {
    typedef const __attribute__((address_space(1))) float *gmem_f32;
    const uint32_t lane_off = (uint32_t)(TRANS ? col * ld + 8 * hh : 8 * hh * ld + col) * (uint32_t)sizeof(float);
    const bool col_ok = !bounded || col < fb;
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int band = 32 * T + 16 * (gq >> 1) + 4 * (gq & 1);
        const gmem_ptr bp = uniform_ptr(reinterpret_cast<const char *>(src + (TRANS ? band : (int64_t)band * ld)));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool ok = col_ok && (!bounded || band + 8 * hh + r < fa);
          const float own =
              ok ? *reinterpret_cast<gmem_f32>(bp + lane_off + (uint32_t)(TRANS ? r : r * ld) * sizeof(float)) : 0.f;
          st[T][4 * gq + r] = fresh ? own : fmaf(f, st[T][4 * gq + r], own);
        }
      }
  };
  // a state of the workspace (W x W, zero beyond fa x fb) / the chunk's incoming state (fa x fb, unpadded)
  auto add_state = [&](const float *src, float f, bool fresh = false) __attribute__((always_inline)) {
    add_state_ld(src, W, f, false, fresh);
  };
  auto add_carry = [&]() __attribute__((always_inline)) {
    add_state_ld(carry_in + (int64_t)sw.bh * g.dt * g.e, NARROW ? (TRANS ? fa : fb) : W, 0.f, NARROW, true);
  };
  if (SRC == SRC_WALK) {
    if (take_carry) add_carry();
  } else if (SRC == SRC_SCANNED) {
    if (states) {
      // the scanned state of this segment, or for a head the scan leaves out (state_dies_in_segment), whose
      // own states are still where the pre-pass put them, the own state of the segment visited before it
      // (the chunk's incoming state for the first one)
      // The workspace holds one state per segment of the pre-pass, of which this sweep segment spans
      // `sub` (1 unless the plan cut long segments finer for the pre-pass, or a backward sweeps several of the
      // forward's in a row): the state that enters it is the one entering its first piece in sweep order.
      const int sub = g.seg_len / g.pre_len;
      const int piece = REV ? min(sw.seg * sub + sub, g.pre_n) - 1 : sw.seg * sub;
      const float *src = states + ((int64_t)sw.bh * g.pre_n + piece) * (W * W);
      bool from_carry = false;
      if (state_dies_in_segment(S[head], g)) {
        const int nb = REV ? piece + 1 : piece - 1;
        if (nb < 0 || nb >= g.pre_n)
          from_carry = true;
        else
          src = states + ((int64_t)sw.bh * g.pre_n + nb) * (W * W);
      }
      // (for such a head the scan kernel has parked the chunk's incoming state in the slot of the piece it
      // visits last, so that nothing reads `carry_in`'s memory once the outgoing state may have replaced it)
      if (from_carry) src = states + ((int64_t)sw.bh * g.pre_n + (REV ? 0 : g.pre_n - 1)) * (W * W);
      if (!from_carry || carry_in != nullptr) add_state(src, 0.f, true);
    }
  } else {
    // `states` holds the segments' OWN states.  The scan's recurrence, St <- l^len_j St + own_j over the
    // segments visited before this one, is run here -- over as many of them as the head's decay reaches:
    // an own state further back arrives weighted below 2^-SKIP_LOG2 (everything between it and this
    // segment is a full-length segment) and is left out, and so is the chunk's incoming state unless the
    // walk starts at the chunk's end.  These waves have the time: the feed waves are fetching block 0.
    const int n_before = REV ? g.n_seg - 1 - sw.seg : sw.seg;
    int first = 0;
    if (sl > 0.f) {
      const float segs = SKIP_LOG2 / (sl * (float)g.seg_len);  // full segments over which a weight falls to 2^-SKIP_LOG2
      if (segs < (float)n_before) first = n_before - ((int)segs + 1);
    }
    first = __builtin_amdgcn_readfirstlane(first);
    if (first == 0 && carry_in) add_carry();
    if (states) {
      const float *base = states + (int64_t)sw.bh * g.n_seg * (W * W);
      const float full = decay(sl, (float)g.seg_len);
      const float last = decay(sl, (float)(g.n - (int64_t)(g.n_seg - 1) * g.seg_len));
      for (int i = first; i < n_before; ++i) {
        const int j = REV ? g.n_seg - 1 - i : i;
        add_state(base + (int64_t)j * (W * W), j == g.n_seg - 1 ? last : full);
      }
    }
  }
  const int s16 = lane & 15, q4 = s16 & 3, ch = (lane >> 4) & 1;
  const int t_row = 8 * hh + (s16 >> 2), t_swz = L::swizzle(t_row);
  const int y_at = t_row * L::ROW + (((2 * ch + (q4 & 1)) ^ t_swz) << 4) + ((q4 >> 1) << 3);
  const int z_at = t_row * L::ROW + (((4 * wcol + 2 * (q4 & 1) + ch) ^ t_swz) << 4) + ((q4 >> 1) << 3);
  const int x_at = a_own * L::ROW + ((hh ^ L::swizzle(c)) << 4);
  const int o_at = a_own * L::ROW + (((4 * wcol + 2 * hh) ^ L::swizzle(c)) << 4);
  const int sc_at = a_own * L::SC_ROW + ((hh ^ ((c >> 1) & 7)) << 4);
  // operand over tokens 16 u + 8 hh .. + 7 of a tile
  auto tokens = [&](const char *tile, int at, int u) __attribute__((always_inline)) {
    const u32x2 lo = lds_tr8(tile + at + 16 * u * L::ROW), hi = lds_tr8(tile + (at ^ 16) + (16 * u + 4) * L::ROW);
    u32x4 r;
    r.x = lo.x;
    r.y = lo.y;
    r.z = hi.x;
    r.w = hi.y;
    return r;
  };
  // St <- l^64 St + Y^T (scaled Z)
  auto update_state = [&](const char *set, float bd) __attribute__((always_inline)) {
    u32x4 yf[4][NT], zs[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      zs[u] = tokens(set + L::ZS, z_at, u);
#pragma unroll
      for (int T = 0; T < NT; ++T) yf[u][T] = tokens(set + L::Y, y_at ^ (T << 6), u);
    }
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r) st[T][r] *= bd;
    reads_first();
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int T = 0; T < NT; ++T) st[T] = E::mfma(yf[u][T], zs[u], st[T]);
  };
  __syncthreads();  // barrier 0
  for (int k = 0; k < runup; ++k) {  // walk
    const int len = len_of(first_blk + k * step);
    update_state(smem + (k & 1) * L::SET, RAGGED && len != BLK ? decay(sl, (float)len) : blockdec);
    __syncthreads();  // walk barrier k
  }
  for (int it = 0; it < nblk; ++it) {
    char *cur = smem + ((runup + it) & 1) * L::SET;
    // A partial block is the chunk's last one.  Going forwards nothing after it uses the state (but the outgoing
    // state where the sweep leaves it); going backwards it comes first and the entering state sits `len` (not 64)
    // tokens ahead.
    const int len = len_of(blk0 + it * step);
    float qd = qdec, bd = blockdec;
    if (RAGGED && REV && len != BLK) {
      qd = decay(sl, (float)max(len - a_own, 0));
      bd = decay(sl, (float)len);
    }
    if (LEAVES_STATE && RAGGED && !REV && len != BLK) bd = decay(sl, (float)len);
    // state term, transposed: acc[4g+r] = sum_f St[f][column] x_a[f], a = a_own
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    // all X fragments are requested before the first product
    u32x4 xf[W / 16];
#pragma unroll
    for (int ks = 0; ks < W / 16; ++ks) xf[ks] = lds16(cur + L::X + (x_at ^ (ks << 5)));
    reads_first();
#pragma unroll
    for (int ks = 0; ks < W / 16; ++ks) {
      const int T = ks >> 1, u = ks & 1;
      u32x4 a;
      a.x = E::pack(st[T][8 * u + 0], st[T][8 * u + 1]);
      a.y = E::pack(st[T][8 * u + 2], st[T][8 * u + 3]);
      a.z = E::pack(st[T][8 * u + 4], st[T][8 * u + 5]);
      a.w = E::pack(st[T][8 * u + 6], st[T][8 * u + 7]);
      acc = E::mfma(a, xf[ks], acc);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] *= qd;
    update_state(cur, bd);
    u32x4 zf[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) zf[u] = tokens(cur + L::Z, z_at, u);
    __syncthreads();  // barrier 2 it + 1: score tile complete
    // intra-block term: acc += Z^T[32 wcol.., tokens] * score[a][tokens]
    u32x4 sf[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) sf[u] = lds16(smem + L::SC + (sc_at ^ (u << 5)));
    reads_first();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool needed = REV ? (ih == 0 || u >= 2) : (ih == 1 || u < 2);
      if (needed) acc = E::mfma(zf[u], sf[u], acc);
    }
    // stage the output in the X tile of this block: the lane holds columns 32 wcol + 16 hh .. + 15
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      u32x4 o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = E::pack(acc[8 * p + 2 * i], acc[8 * p + 2 * i + 1]);
      *reinterpret_cast<u32x4 *>(cur + L::X + (o_at ^ (p << 4))) = o;
    }
    __syncthreads();  // barrier 2 it + 2
  }
  // the segment visited last leaves the chunk's outgoing state
  if (SRC != SRC_SCANNED && !TRANS && carry_out != nullptr && sw.seg == (REV ? 0 : g.n_seg - 1) && ih == 0) {
    float *cp = carry_out + (int64_t)sw.bh * g.dt * g.e, *tp = g.twin ? g.twin + (int64_t)sw.bh * g.dt * g.e : nullptr;
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * T + 16 * (r >> 3) + 8 * hh + 4 * ((r >> 2) & 1) + (r & 3);
        if (!NARROW || (row < fa && col < fb)) {
          cp[row * (NARROW ? fb : W) + col] = st[T][r];
          if (tp) tp[row * (NARROW ? fb : W) + col] = st[T][r];
        }
      }
  }
}

// LDS of the 128-wide sweep: three sets of token-major X, Y and Z tiles, and the score tile.
struct SweepLds {
  static constexpr int ROW = 256, TILE = BLK * ROW;
  static constexpr int X = 0, Y = TILE, Z = 2 * TILE, SET = 3 * TILE;
  static constexpr int SC = 3 * SET, SC_ROW = 2 * BLK;
  static constexpr int KDEC = SC + BLK * SC_ROW;  // decay between each token of a block and the state that the block leaves,
  static constexpr int KDEC_TAIL = KDEC + 4 * BLK;  // ... and of the chunk's partial last block
  static constexpr int BYTES = KDEC_TAIL + 4 * BLK;  // 156 160 B: one workgroup per CU
};
// unit u (16 bytes) of row r of such a tile lies at u ^ swizzle(r)
__device__ __forceinline__ int swizzle(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
__device__ __forceinline__ uint32_t lds_address(const char *p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p;
}
__device__ __forceinline__ u32x4 row_buffer(const void *p, int bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  u32x4 r;
  r.x = __builtin_amdgcn_readfirstlane((uint32_t)v);
  r.y = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  r.z = (uint32_t)__builtin_amdgcn_readfirstlane(bytes);
  r.w = 0x00020000u;
  return r;
}
// 16 bytes per lane from memory to LDS, lane after lane from `lds` on
__device__ __forceinline__ void load_to_lds(u32x4 rows, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(off), "s"(rows)
               : "memory", "m0");
}
// ... that the caches need not keep
__device__ __forceinline__ void load_to_lds_once(u32x4 rows, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds" ::"s"(lds), "v"(off), "s"(rows)
               : "memory", "m0");
}
// A barrier that the wave's LDS accesses have to be done for, but the N youngest (they are answered in order)
template <int N>
__device__ __forceinline__ void barrier_before() {
  asm volatile("s_waitcnt lgkmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// ------------------------------------------------------------------------------
// The 128-wide sweep.  512 threads, one workgroup per CU, two groups of waves:
//   waves 0-3 ("feed"): loads, which go from memory straight to LDS, two blocks ahead; the masked score tile; the output stores;
//   waves 4-7 ("math"): own the state and the output (wave 4 + w: 32 columns from 32 w on): state term, state update, the
//     scores' part of the output ("intra"), which follows while the next block is under way.
// A block takes two barriers:
//     feed: score(t) up to its products,  | math: upper half of the state update(t-1), intra(t-1), first half of the state
//           load Y, Z(t+2)                |       term(t), stage O(t-1) in the X tile of block t-1
//   ---- barrier m ----
//     feed: mask and write score(t),      | math: second half of the state term(t), lower half of the state update(t)
//           store O(t-1), load X(t+2)     |
//   ---- barrier b ----
// Every tile lies token-major, as in memory: what contracts over tokens is read transposed (ds_read_b64_tr_b16), the state update's
// decay goes to the 32 columns of Z that only one wave reads, and no wave moves a tile through its registers.
//
// What bounds a block.  The issue of the math waves' instructions, some 300 on the vector unit, 38 products and 70 LDS accesses
// in each; then the LDS, which moves some 330 KB a block, counted access by access.  So the vector work is dealt out
// between the products by hand (see `slot`), reads are asked for a phase ahead, and what a block's first reads would wait for is
// covered by products held back from the block before.  Neither stores nor loads to registers stand in the math waves: behind the feed waves' loads
// each of them waits its turn in the memory pipeline (and so does any register spilled to scratch).
//   Cycles a block, alone on a CU: 3100 (4130 with tiles that went through registers, transposed on the way, and the state update
// and both halves of the output between the same two barriers); LDS busy for 1410 of them (1860), 180 in conflicts (240).  Sweep
// kernels in us, that form and this one, one after the other on one card: b*h = 16, n = 65536: forward 194.3 and 195.7 (0.7 % lost),
// backward 481 and 437 (the forward moves its bytes at 5.6 TB/s either way; of the backward's 2.69 GB beyond L2 the
// memory-side cache serves a part); n = 16384 in 256 segments: 48 and 46, 136 and 113; b*h = 36,
// n = 5003: 34.8 and 32.4, 97 and 84.6; b*h = 24, n = 2048, 7 segments: 14.6 and 13.4, 30.4 and 27.7; two slices of d = 256, b*h = 8,
// n = 8192: 40 and 34, 97 and 82.
//   Rows of X and Y of at most 64 features (d = 128, e = 64 backwards) have two of four state tiles of zeros, which that form left out
// and this one multiplies: a branch there would cut the hand-made order.  Whole calls, forward and backward, b*h = 16, n = 65536:
// d = 128, e = 64 188 and 188, 451 and 391; 64 x 128 187 and 189, 435 and 378; b*h = 24, n = 2048, 128 x 64 27.7 and 25.9,
// 40.0 and 36.5.
// ------------------------------------------------------------------------------
template <class E, bool REV, bool TRANS, int SRC, int MODE>
__device__ __forceinline__ void
sweep_body(const elem16_t *__restrict__ X, const elem16_t *__restrict__ Y, const elem16_t *__restrict__ Z,
           const float *__restrict__ S, const float *__restrict__ states, elem16_t *__restrict__ Out, const Geom &g,
           int fa, int fb, int item, char *smem, const float *__restrict__ carry_in,
           float *__restrict__ carry_out = nullptr) {
  constexpr bool RAGGED = MODE != M_ALIGNED, NARROW = MODE >= M_NARROW;
  constexpr bool LEAVES_STATE = SRC != SRC_SCANNED;  // the sweep's final state is the chunk's outgoing one
  constexpr bool MAY_BE_KEPT = SRC == SRC_WALK && !REV && TRANS;  // dQ, see Geom::kept
  using L = SweepLds;
  constexpr int W = 128;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = w8 & 3;
  const int c = lane & 31, hh = lane >> 5;

  const int bh = quotient(item, g.by_seg), head = bh - quotient(bh, g.by_h) * g.h;
  const int total_blk = (int)((g.n + BLK - 1) / BLK);  // blocks in the chunk
  float slope = 0.f;
  int reach = 0;
  if (SRC == SRC_WALK) {
    slope = S[head];
    reach = __builtin_amdgcn_readfirstlane(reach_of(slope, total_blk));
  }
  const SegWork sw = SRC == SRC_WALK ? walk_work(g, item, REV, reach) : seg_work(g, item);
  const int64_t row0 = (int64_t)sw.bh * g.n + sw.tok0;
  // elements from row to row of X and Y, and of Z and Out: q, k and their gradients have rows of g.dt features, of which
  // a slice of a wide head reads and writes fa (fb)
  const int xp = NARROW ? (TRANS ? g.e : g.dt) : W, zp = NARROW ? (TRANS ? g.dt : g.e) : W;
  const int nblk = sw.nblk;
  const int step = REV ? -1 : 1;
  const int blk0 = REV ? nblk - 1 : 0;
  const int seg_blk0 = (int)(sw.tok0 / BLK);           // the segment's first block
  const int chunk_tail = (int)(g.n - (int64_t)(total_blk - 1) * BLK);
  // tokens in a block (numbered relative to the segment): a partial block is the chunk's last one
  auto len_of = [&](int blk) __attribute__((always_inline)) {
    if (!RAGGED) return BLK;
    return seg_blk0 + blk == total_blk - 1 ? chunk_tail : BLK;
  };
  // SRC_WALK: the state entering the segment is rebuilt by walking `runup` blocks outside it first (before it,
  // or after it going backwards), as far as the head's decay reaches, from the chunk's incoming state if the
  // walk gets to the chunk's end, else from zero.  Blocks are numbered relative to the segment; walk and sweep
  // form one run of runup + nblk blocks, first_blk, first_blk + step, ..., of which the first `runup` only
  // update the state.
  int runup = 0;
  bool take_carry = false;
  if (SRC == SRC_WALK) {
    const int avail = REV ? total_blk - (seg_blk0 + nblk) : seg_blk0;
    runup = min(reach, avail);
    take_carry = carry_in != nullptr && runup == avail;
  }
  const int first_blk = blk0 - runup * step;
  const int run = runup + nblk;  // blocks in the whole run

  if (w8 < 4) {
    // ================================ feed waves ================================
    // Wave w loads rows 16 w .. + 15 of every tile, four of them at a time: lane l's 16 bytes land at unit l % 16 of row l / 16.
    uint32_t x_off[4], z_off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 16 * w + 4 * i + (lane >> 4), unit = (lane & 15) ^ swizzle(row);
      x_off[i] = !NARROW || unit * 8 < fa ? (uint32_t)(row * xp * 2 + unit * 16) : kOutside;
      z_off[i] = !NARROW || unit * 8 < fb ? (uint32_t)(row * zp * 2 + unit * 16) : kOutside;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(smem) + 16 * w * L::ROW);
    const elem16_t *Xg = X + row0 * xp, *Yg = Y + row0 * xp, *Zg = Z + row0 * zp;
    auto fetch_tile = [&](const elem16_t *base, int blk, int pitch, const uint32_t (&off)[4], uint32_t lds)
                          __attribute__((always_inline)) {
      const u32x4 rows = row_buffer(base + (int64_t)blk * BLK * pitch, len_of(blk) * pitch * 2);
      if (SRC != SRC_WALK && !REV && blk < nblk - g.stay) {
#pragma unroll
        for (int i = 0; i < 4; ++i) load_to_lds_once(rows, off[i], lds + 4 * i * L::ROW);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) load_to_lds(rows, off[i], lds + 4 * i * L::ROW);
      }
    };
    // block k of the run into set `set`: four loads of X (none for a block that is only walked over), eight of Y and Z
    auto fetch_x = [&](int k, int set) __attribute__((always_inline)) {
      if (SRC != SRC_WALK || k >= runup) fetch_tile(Xg, first_blk + k * step, xp, x_off, lds0 + set * L::SET + L::X);
    };
    auto fetch_yz = [&](int k, int set) __attribute__((always_inline)) {
      const int blk = first_blk + k * step;
      fetch_tile(Yg, blk, xp, x_off, lds0 + set * L::SET + L::Y);
      fetch_tile(Zg, blk, zp, z_off, lds0 + set * L::SET + L::Z);
    };
    fetch_x(0, 0);
    fetch_yz(0, 0);
    if (run > 1) {
      fetch_x(1, 1);
      fetch_yz(1, 1);
    }
    const float *late = S + head;  // (asked for behind the first loads: it would have to arrive before they could leave)
    asm volatile("" : "+s"(late));
    const float sl = *late * LOG2E;
    if (tid < BLK) {
      *reinterpret_cast<float *>(smem + L::KDEC + 4 * tid) = decay(sl, REV ? (float)tid : (float)(BLK - tid));
      if (RAGGED) *reinterpret_cast<float *>(smem + L::KDEC_TAIL + 4 * tid) = decay(sl, REV ? (float)tid : (float)max(chunk_tail - tid, 0));
    }
    // this wave's quadrant of the transposed score tile: sc[4g+r] = y_b . x_a, b = 32qJ+8g+4hh+r, a = 32qI+c
    const int qI = w >> 1, qJ = w & 1;
    const bool q_active = REV ? !(qI == 1 && qJ == 0) : !(qI == 0 && qJ == 1);
    float mask[16];  // decay between the tokens of a score; negative: masked
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int a = 32 * qI + c, b = 32 * qJ + 8 * (r >> 2) + 4 * hh + (r & 3), dist = REV ? b - a : a - b;
      mask[r] = dist >= 0 ? decay(sl, (float)dist) : -1.f;
    }
    const int x_at = 32 * qI * L::ROW + c * L::ROW + ((hh ^ swizzle(c)) << 4);
    const int y_at = 32 * qJ * L::ROW + c * L::ROW + ((hh ^ swizzle(c)) << 4);
    const int sc_at = (32 * qI + c) * L::SC_ROW + ((4 * qJ ^ ((c >> 1) & 7)) << 4) + 8 * hh;
    floatx16 sc;
    auto write_scores = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        float m[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) m[r] = mask[4 * gq + r] >= 0.f ? sc[4 * gq + r] * mask[4 * gq + r] : 0.f;
        u32x2 o;
        o.x = E::pack(m[0], m[1]);
        o.y = E::pack(m[2], m[3]);
        *reinterpret_cast<u32x2 *>(smem + L::SC + (sc_at ^ (gq << 4))) = o;
      }
    };
    // the rows of output staged in a set's X tile, where this wave will load X: row by row to where the rows of Z lie
    elem16_t *Og = Out + row0 * zp;
    const char *const o_from = smem + L::X + 16 * w * L::ROW + lane * 16;
    u32x4 out[4];
    // Output is not read again here, and its stores say so, but the dV that the next slice of a wide head adds to: where the L2s hold it, it
    // stays there.  Backward, us, d = 256: b*h = 8, n = 8192 96.1 -> 89.1, b*h = 32, n = 3000 128.8 -> 120.9; beyond, b*h = 24, n = 12000 308 -> 313,
    // and in the forward, b*h = 4, n = 15761 60.1 -> 61.3, it would lose.
    constexpr int64_t L2_BYTES = (int64_t)32 << 20;
    const bool again = MODE == M_NARROW && REV && !TRANS && g.dt > W && (int64_t)(g.b * g.h) * g.n * g.e * 2 <= L2_BYTES;
    auto read_out = [&](int set) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) out[i] = lds16(o_from + set * L::SET + 4 * i * L::ROW);
    };
    auto store_out = [&](int k) __attribute__((always_inline)) {
      const int blk = first_blk + k * step;
      const rows_t rows = rows_of(Og + (int64_t)blk * BLK * zp, len_of(blk) * zp * 2);
      if (again) {
#pragma unroll
        for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_buffer_store_b128(out[i], rows, (int)z_off[i], 0, 0);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_buffer_store_b128(out[i], rows, (int)z_off[i], 0, 2 /* non-temporal */);
      }
    };
    // Everything that this wave has asked for but the loads of block 1 has arrived
    if (run == 1)
      wait_loads<0>();
    else if (SRC != SRC_WALK || runup <= 1)
      wait_loads<12>();
    else
      wait_loads<8>();
    __syncthreads();  // block 0 of the run visible
    int set = 0, spare = 2;  // of block k, and of the blocks before it and two after it
    int k = 0;
    for (; SRC == SRC_WALK && k < runup; ++k) {
      if (k + 2 < run) {
        fetch_x(k + 2, spare);
        fetch_yz(k + 2, spare);
      }
      if (k + 2 >= run)
        wait_loads<0>();
      else if (k + 2 >= runup)
        wait_loads<12>();
      else
        wait_loads<8>();
      __syncthreads();  // block k + 1 visible; the tiles of block k no longer read
      spare = set;
      set = set == 2 ? 0 : set + 1;
    }
    for (; k < run; ++k) {
      u32x4 yf[8], xf[8];
      if (q_active) {
        const char *from = smem + set * L::SET;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
          yf[ks] = lds16(from + L::Y + (y_at ^ (ks << 5)));
          xf[ks] = lds16(from + L::X + (x_at ^ (ks << 5)));
        }
      }
      if (k + 2 < run) fetch_yz(k + 2, spare);
      if (q_active) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) sc = E::mfma(yf[ks], xf[ks], sc);
      }
      __syncthreads();  // the scores of block k - 1 no longer read, its output staged
      if (q_active) write_scores();
      if (k > runup) {
        read_out(spare);
        store_out(k - 1);
      }
      if (k + 2 < run) fetch_x(k + 2, spare);
      // all but what was asked for since: four stores, 12 loads
      if (k + 2 < run) {
        if (k > runup)
          wait_loads<16>();
        else
          wait_loads<12>();
      } else if (k + 1 < run) {
        if (k > runup)
          wait_loads<4>();
        else
          wait_loads<0>();
      }
      __syncthreads();  // block k + 1 and the scores of block k visible; the tiles of block k no longer read
      spare = set;
      set = set == 2 ? 0 : set + 1;
    }
    __syncthreads();  // the last block's output staged
    read_out(spare);
    store_out(run - 1);
    return;
  }

  // ================================== math waves ==================================
  __builtin_amdgcn_s_setprio(2);  // a block waits for these waves: b*h = 16, n = 65536, backward sweep 460 us, 475 without
  // Registers and rows.  An accumulator tile holds rows 8g + 4hh + r in register 4g + r of lane (c, hh).  Which feature
  // of Y (state row) and which column of Z (state column, output column) a row or lane stands for is chosen by the addresses of
  // the transposing reads: state row 32T + 16(g / 2) + 8hh + 4(g % 2) + r, so that the eight rows of a k-step are eight
  // features in a row, as X has them in memory; column 16 hh' + 4 g + r for lane c = 8g + 4hh' + r, so that a lane of the output tile holds
  // 16 columns in a row of its token.
  const int col = 32 * w + 16 * ((c >> 2) & 1) + 4 * (c >> 3) + (c & 3);
  const float sl = S[head] * LOG2E;
  const float blockdec = decay(sl, (float)BLK);
  float qdec[2];
#pragma unroll
  for (int I = 0; I < 2; ++I) qdec[I] = decay(sl, REV ? (float)(BLK - 32 * I - c) : (float)(32 * I + c));
  floatx16 st[4];
#pragma unroll
  for (int T = 0; T < 4; ++T)
#pragma unroll
    for (int r = 0; r < 16; ++r) st[T][r] = 0.f;
  // st <- f * st + M (`fresh`: st <- M, which leaves the loads in flight until a product needs them), M being the W x W fp32
  // tile whose element (row, col) is src[row * ld + col], or for a transposed role src[col * ld + row]; `bounded`: src holds
  // only fa x fb (transposed: fb x fa) elements
  auto add_state_ld = [&](const float *src, int ld, float f, bool bounded, bool fresh) __attribute__((always_inline)) {
    typedef const __attribute__((address_space(1))) float *gmem_f32;
    const uint32_t lane_off = (uint32_t)(TRANS ? col * ld + 8 * hh : 8 * hh * ld + col) * (uint32_t)sizeof(float);
    const bool col_ok = !bounded || col < fb;
#pragma unroll
    for (int T = 0; T < 4; ++T)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int band = 32 * T + 16 * (gq >> 1) + 4 * (gq & 1);
        const gmem_ptr bp = uniform_ptr(reinterpret_cast<const char *>(src + (TRANS ? band : (int64_t)band * ld)));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool ok = col_ok && (!bounded || band + 8 * hh + r < fa);
          const float own =
              ok ? *reinterpret_cast<gmem_f32>(bp + lane_off + (uint32_t)(TRANS ? r : r * ld) * sizeof(float)) : 0.f;
          st[T][4 * gq + r] = fresh ? own : fmaf(f, st[T][4 * gq + r], own);
        }
      }
  };
  // a state of the workspace (W x W, zero beyond fa x fb) / the chunk's incoming state (fa x fb, unpadded)
  auto add_state = [&](const float *src, float f, bool fresh = false) __attribute__((always_inline)) {
    add_state_ld(src, W, f, false, fresh);
  };
  auto add_carry = [&]() __attribute__((always_inline)) {
    add_state_ld(carry_in + (int64_t)sw.bh * g.dt * g.e, NARROW ? (TRANS ? fa : fb) : W, 0.f, NARROW, true);
  };
  if (SRC == SRC_WALK) {
    const float *src = carry_in + (int64_t)sw.bh * g.dt * g.e;
    int ld = NARROW ? (TRANS ? fa : fb) : W;
    if (MAY_BE_KEPT && g.kept) {
      // the state that entered the chunk lies in the slot of the first piece, or of the last one for a head outside the scan (see below).
      // (By the slope at hand: asked for again it would have to arrive before these loads could leave.)
      const bool parked = state_dies_in_segment(slope, g);
      if (parked && g.kept == KEPT_STATES_ONLY) take_carry = false;
      src = carry_in + ((int64_t)sw.bh * g.pre_n + (parked ? g.pre_n - 1 : 0)) * (W * W);
      ld = W;
    }
    if (take_carry) add_state_ld(src, ld, 0.f, NARROW, true);
  } else if (SRC == SRC_SCANNED) {
    if (states) {
      // the scanned state of this segment, or for a head the scan leaves out (state_dies_in_segment), whose
      // own states are still where the pre-pass put them, the own state of the segment visited before it
      // (the chunk's incoming state for the first one)
      // The workspace holds one state per segment of the pre-pass, of which this sweep segment spans
      // `sub` (1 unless the plan cut long segments finer for the pre-pass, or a backward sweeps several of the
      // forward's in a row): the state that enters it is the one entering its first piece in sweep order.
      const int sub = g.seg_len / g.pre_len;
      const int piece = REV ? min(sw.seg * sub + sub, g.pre_n) - 1 : sw.seg * sub;
      const float *src = states + ((int64_t)sw.bh * g.pre_n + piece) * (W * W);
      bool from_carry = false;
      if (state_dies_in_segment(S[head], g)) {
        const int nb = REV ? piece + 1 : piece - 1;
        if (nb < 0 || nb >= g.pre_n)
          from_carry = true;
        else
          src = states + ((int64_t)sw.bh * g.pre_n + nb) * (W * W);
      }
      // (for such a head the scan kernel has parked the chunk's incoming state in the slot of the piece it
      // visits last, so that nothing reads `carry_in`'s memory once the outgoing state may have replaced it)
      if (from_carry) src = states + ((int64_t)sw.bh * g.pre_n + (REV ? 0 : g.pre_n - 1)) * (W * W);
      if (!from_carry || carry_in != nullptr) add_state(src, 0.f, true);
    }
  } else {
    // `states` holds the segments' OWN states.  The scan's recurrence, St <- l^len_j St + own_j over the
    // segments visited before this one, is run here -- over as many of them as the head's decay reaches:
    // an own state further back arrives weighted below 2^-SKIP_LOG2 (everything between it and this
    // segment is a full-length segment) and is left out, and so is the chunk's incoming state unless the
    // walk starts at the chunk's end.  These waves have the time: the feed waves are fetching block 0.
    const int n_before = REV ? g.n_seg - 1 - sw.seg : sw.seg;
    int first = 0;
    if (sl > 0.f) {
      const float segs = SKIP_LOG2 / (sl * (float)g.seg_len);  // full segments over which a weight falls to 2^-SKIP_LOG2
      if (segs < (float)n_before) first = n_before - ((int)segs + 1);
    }
    first = __builtin_amdgcn_readfirstlane(first);
    if (first == 0 && carry_in) add_carry();
    if (states) {
      const float *base = states + (int64_t)sw.bh * g.n_seg * (W * W);
      const float full = decay(sl, (float)g.seg_len);
      const float last = decay(sl, (float)(g.n - (int64_t)(g.n_seg - 1) * g.seg_len));
      for (int i = first; i < n_before; ++i) {
        const int j = REV ? g.n_seg - 1 - i : i;
        add_state(base + (int64_t)j * (W * W), j == g.n_seg - 1 ? last : full);
      }
    }
  }
  const int s16 = lane & 15, q4 = s16 & 3, ch = (lane >> 4) & 1;
  const int t_row = 8 * hh + (s16 >> 2), t_swz = swizzle(t_row);
  const int y_at = t_row * L::ROW + (((2 * ch + (q4 & 1)) ^ t_swz) << 4) + ((q4 >> 1) << 3);
  const int z_at = t_row * L::ROW + (((4 * w + 2 * (q4 & 1) + ch) ^ t_swz) << 4) + ((q4 >> 1) << 3);
  const int x_at = c * L::ROW + ((hh ^ swizzle(c)) << 4);
  const int sc_at = c * L::SC_ROW + ((hh ^ ((c >> 1) & 7)) << 4);
  // operand over tokens 16 u + 8 hh .. + 7 of a tile
  auto tokens = [&](const char *tile, int at, int u) __attribute__((always_inline)) {
    const u32x2 lo = lds_tr8(tile + at + 16 * u * L::ROW), hi = lds_tr8(tile + (at ^ 16) + (16 * u + 4) * L::ROW);
    u32x4 r;
    r.x = lo.x;
    r.y = lo.y;
    r.z = hi.x;
    r.w = hi.y;
    return r;
  };
  // Work for the vector unit is dealt out by hand between the products: one of 32 x 32 x 16 keeps the matrix unit busy for 32
  // cycles, in which the wave that issued it can issue some seven other instructions; the scheduler would put all of them in front.
  auto slot = [](floatx16 &sum, const u32x4 &a, const u32x4 &b, auto &&work) __attribute__((always_inline)) {
    sum = E::mfma(a, b, sum);
    work();
    __builtin_amdgcn_sched_barrier(0);
  };
  // rows r0 .. + 3 of tile T of the state
  auto decay_state = [&](int T, int r0, float bd) __attribute__((always_inline)) {
#pragma unroll
    for (int r = r0; r < r0 + 4; ++r) {
      float x = st[T][r] * bd;
      asm volatile("" : "+v"(x));
      st[T][r] = x;
    }
  };
  // operand of k-step ks of the state term
  auto pack_state = [&](int ks) __attribute__((always_inline)) {
    const int T = ks >> 1, r = 8 * (ks & 1);
    u32x4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t x = E::pack(st[T][r + 2 * i], st[T][r + 2 * i + 1]);
      asm volatile("" : "+v"(x));
      a[i] = x;
    }
    return a;
  };
  // Z^T scaled by its tokens' decay to the block's end: the decays of step u, pair i of it.  (Where a sweep leaves the state, the
  // tokens of the chunk's partial last block, going forwards, lie `len` - b before the end; elsewhere nothing after that block
  // uses the state.)
  const int kdec_at = L::KDEC + 32 * hh;
  auto read_kdec = [&](int u, int len, u32x4 (&kd)[2]) __attribute__((always_inline)) {
    const char *from = smem + kdec_at + (LEAVES_STATE && RAGGED && len != BLK ? L::KDEC_TAIL - L::KDEC : 0) + 64 * u;
    kd[0] = lds16(from);
    kd[1] = lds16(from + 16);
  };
  auto scale_z = [&](const u32x4 (&zf)[4], u32x4 (&zs)[4], const u32x4 (&kd)[2], int u, int i) __attribute__((always_inline)) {
    const u32x4 &q = kd[i >> 1];
    const float w0 = __uint_as_float((i & 1) ? q.z : q.x), w1 = __uint_as_float((i & 1) ? q.w : q.y);
    uint32_t x = E::pack(elem_f32<E>(zf[u], 2 * i) * w0, elem_f32<E>(zf[u], 2 * i + 1) * w1);
    asm volatile("" : "+v"(x));
    zs[u][i] = x;
  };
  // operand over tokens 16 u .. of the 32 rows of state tile T
  auto read_y = [&](const char *tile, int lane_at, int T, int u) __attribute__((always_inline)) {
    return tokens(tile, lane_at ^ (T << 6), u);
  };
  // an offset whose variants are worked out where they are used and not kept in registers
  auto fresh = [](int at) __attribute__((always_inline)) {
    asm volatile("" : "+v"(at));
    return at;
  };
  // Slices of a wide head after the first add to what the slices before them left in Out (its rows are whole
  // features of v, so only the non-transposed roles).  A block's old output is fetched while the block before it is
  // computed; the lane holds the columns that its accumulators hold.
  constexpr bool ADDS = MODE == M_ADDING && !TRANS;
  u32x4 old[2][2] = {};
  auto fetch_old = [&](int blk) __attribute__((always_inline)) {
    const rows_t rows = rows_of(Out + (row0 + (int64_t)blk * BLK) * zp, len_of(blk) * zp * 2);
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int first = 32 * w + 16 * hh + 8 * p;
        old[I][p] = __builtin_amdgcn_raw_buffer_load_b128(
            rows, first < fb ? (32 * I + c) * zp * 2 + first * 2 : (int)kOutside, 0, 0);
      }
  };
  // Unit j of 8 of a block's output on its way into an X tile: four for the 32 tokens that `first` names, then four for the others
  const int o_at = c * L::ROW + (((4 * w + 2 * hh) ^ swizzle(c)) << 4);
  auto pack_out = [&](const floatx16 (&acc)[2], int first, int j, char *tile, u32x4 &o) __attribute__((always_inline)) {
    const int lane_at = fresh(o_at);
    const int I = j < 4 ? first : 1 - first, i = j & 3;
    o[2 * (i & 1)] = E::pack(acc[I][4 * i], acc[I][4 * i + 1]);
    o[2 * (i & 1) + 1] = E::pack(acc[I][4 * i + 2], acc[I][4 * i + 3]);
    if (i & 1) *reinterpret_cast<u32x4 *>(tile + 32 * I * L::ROW + (lane_at ^ ((i >> 1) << 4))) = o;
  };
  if (NARROW && 32 * w >= fb) {  // a wave whose columns all lie past the width of Z only takes part in the barriers
    for (int i = 0; i < 2 + runup + 2 * nblk; ++i) __syncthreads();
    return;
  }
  __syncthreads();  // block 0 of the run visible
  int set_i = 0, k = 0;
  // What a block leaves to the next one's time: of its output, the scores' part (they are computed meanwhile), of the state
  // update, the upper half of the rows, whose products cover the time that the next block's first reads take.
  floatx16 acc[2];  // the output without that part, not yet scaled by ...
  float qd[2] = {1.f, 1.f};
  u32x4 zf[4], zs[4], yf1[4][2];
#pragma unroll
  for (int I = 0; I < 2; ++I)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[I][r] = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) zf[u] = zs[u] = yf1[u][0] = yf1[u][1] = u32x4{0u, 0u, 0u, 0u};
  // acc[I] += Z^T[32 w .., tokens] * score[a][tokens] of the block before
  auto read_scores = [&](const char *tile, u32x4 (&sf)[4][2]) __attribute__((always_inline)) {
    const int lane_at = fresh(sc_at);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int I = 0; I < 2; ++I)
        if (REV ? (I == 0 || u >= 2) : (I == 1 || u < 2)) sf[u][I] = lds16(tile + 32 * I * L::SC_ROW + (lane_at ^ (u << 5)));
  };
  // the six products of (row half I of the output, tokens 16 u ..) that the mask leaves
  constexpr int INTRA_U[2][6] = {{0, 1, 0, 1, 2, 3}, {2, 3, 0, 1, 2, 3}}, INTRA_I[2][6] = {{0, 0, 1, 1, 1, 1}, {1, 1, 0, 0, 0, 0}};
  constexpr int FIRST = REV ? 1 : 0;  // the half that is finished first
  auto scale_acc = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 4 * (j & 3); r < 4 * (j & 3) + 4; ++r) {
      float x = ADDS ? fmaf(acc[j >> 2][r], qd[j >> 2], elem_f32<E>(old[j >> 2][r >> 3], r & 7)) : acc[j >> 2][r] * qd[j >> 2];
      asm volatile("" : "+v"(x));
      acc[j >> 2][r] = x;
    }
  };
  if (SRC == SRC_WALK && runup > 0) {
    // A walk block: the upper half of the rows of the state update of the block before, whose products cover the time that this block's
    // first reads take, then the lower half of its own.  What bounds it is the issue of a math wave's instructions, alone on its SIMD but
    // for a feed wave: 16 products, 40 LDS reads and 190 on the vector unit, 0.57 us a block where reads, scaling and products that
    // followed one another took 0.69 (the loads alone would allow 0.35; scaling Z in the feed waves instead took 0.71, loads three blocks
    // ahead instead of two 0.57).  Backwards in one launch, in us: b*h = 24, n = 2048 36.8 -> 34.5, b*h = 20, n = 1024 21.5 -> 20.7;
    // forwards, b*h = 48, n = 1024 20.0 -> 18.5.
    u32x4 kd[4][2], zr[4], zt[4], yf0[4][2];
#pragma unroll
    for (int u = 0; u < 4; ++u) read_kdec(u, BLK, kd[u]);  // (partial only going backwards, where the tokens' decays are the same)
    auto walk = [&](u32x4 (&before)[4], u32x4 (&now)[4]) __attribute__((always_inline)) {
      const char *set = smem + set_i * L::SET;
      set_i = set_i == 2 ? 0 : set_i + 1;
      const int len = len_of(first_blk + k * step);
      const float bd = RAGGED && len != BLK ? decay(sl, (float)len) : blockdec;
      const int y_lane = fresh(y_at), z_lane = fresh(z_at);
#pragma unroll
      for (int u = 0; u < 2; ++u) zr[u] = tokens(set + L::Z, z_lane, u);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        slot(st[2 + (j & 1)], yf1[j >> 1][j & 1], before[j >> 1], [&]() __attribute__((always_inline)) {
          if (j < 2) zr[2 + j] = tokens(set + L::Z, z_lane, 2 + j);
          if (j >= 2 && j < 6) {
            yf0[j - 2][0] = read_y(set + L::Y, y_lane, 0, j - 2);
            yf0[j - 2][1] = read_y(set + L::Y, y_lane, 1, j - 2);
          }
          decay_state(j >> 2, 4 * (j & 3), bd);
          if (j >= 4) scale_z(zr, now, kd[(j - 4) >> 1], (j - 4) >> 1, 2 * (j & 1)), scale_z(zr, now, kd[(j - 4) >> 1], (j - 4) >> 1, 2 * (j & 1) + 1);
        });
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int u = j >> 1, T = j & 1;
        slot(st[T], yf0[u][T], now[u], [&]() __attribute__((always_inline)) {
          if (j < 4) scale_z(zr, now, kd[2 + (j >> 1)], 2 + (j >> 1), 2 * (j & 1)), scale_z(zr, now, kd[2 + (j >> 1)], 2 + (j >> 1), 2 * (j & 1) + 1);
          decay_state(2 + (j >> 2), 4 * (j & 3), bd);
          yf1[u][T] = read_y(set + L::Y, y_lane, 2 + T, u);
        });
      }
      __syncthreads();
      ++k;
    };
    for (; k + 1 < runup;) {
      walk(zs, zt);
      walk(zt, zs);
    }
    if (k < runup) {
      walk(zs, zt);
#pragma unroll
      for (int u = 0; u < 4; ++u) zs[u] = zt[u];
    }
  }
  for (; k < run; ++k) {
    const char *set = smem + set_i * L::SET;
    char *const staged = smem + (set_i == 0 ? 2 : set_i - 1) * L::SET + L::X;  // where the output of the block before goes
    set_i = set_i == 2 ? 0 : set_i + 1;
    const int blk = first_blk + k * step;
    const int len = len_of(blk);
    // A partial block is the chunk's last one.  Going forwards nothing after it uses the state (but the outgoing
    // state where the sweep leaves it); going backwards it comes first and the entering state sits `len` (not 64)
    // tokens ahead.
    float qn[2] = {qdec[0], qdec[1]};
    float bd = blockdec;
    if (RAGGED && REV && len != BLK) {
#pragma unroll
      for (int I = 0; I < 2; ++I) qn[I] = decay(sl, (float)max(len - 32 * I - c, 0));
      bd = decay(sl, (float)len);
    }
    if (LEAVES_STATE && RAGGED && !REV && len != BLK) bd = decay(sl, (float)len);
    {
      u32x4 sf[4][2], xf[2][4][2], yf0[4][2], zn[4], a[4], kd[4][2];
      const int x_lane = fresh(x_at), y_lane = fresh(y_at), z_lane = fresh(z_at);
      auto read_x = [&](int ks, int I) __attribute__((always_inline)) {
        return lds16(set + L::X + 32 * I * L::ROW + (x_lane ^ (ks << 5)));
      };
      read_scores(smem + L::SC, sf);
#pragma unroll
      for (int j = 0; j < 4; ++j) xf[0][j >> 1][j & 1] = read_x(j >> 1, j & 1);
      reads_first();
      // (1) the block before: the rest of its state update, the scores
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        slot(st[2 + (j & 1)], yf1[j >> 1][j & 1], zs[j >> 1], [&]() __attribute__((always_inline)) {
          scale_acc(j);
          if (j >= 4) xf[0][j >> 1][j & 1] = read_x(j >> 1, j & 1);
        });
      }
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        slot(acc[INTRA_I[REV][j]], zf[INTRA_U[REV][j]], sf[INTRA_U[REV][j]][INTRA_I[REV][j]], [&]() __attribute__((always_inline)) {
          if (j < 4) a[j] = pack_state(j);
          if (j >= 2) zn[j - 2] = tokens(set + L::Z, z_lane, j - 2);
          if (j >= 2 && j < 4) decay_state(0, 8 * (j - 2), bd), decay_state(0, 8 * (j - 2) + 4, bd);
          if (j >= 4) decay_state(1, 8 * (j - 4), bd), decay_state(1, 8 * (j - 4) + 4, bd);
        });
      }
      // (2) state term, transposed: term[I][4g+r] = sum_f St[f][column] x_a[f], a = 32 I + c
      floatx16 term[2];
#pragma unroll
      for (int I = 0; I < 2; ++I)
#pragma unroll
        for (int r = 0; r < 16; ++r) term[I][r] = 0.f;
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int ks = j >> 1, I = j & 1;
        slot(term[I], a[ks], xf[0][ks][I], [&]() __attribute__((always_inline)) {
          if (j >= 1 && j < 5) {
            pack_out(acc, FIRST, 2 * j - 2, staged, o);
            pack_out(acc, FIRST, 2 * j - 1, staged, o);
          }
          if (j == 2) read_kdec(0, len, kd[0]);
          if (j == 3) read_kdec(1, len, kd[1]);
          if (j == 4) __builtin_amdgcn_sched_barrier(0);
          if (j >= 4) {
            xf[1][j - 4][0] = read_x(j, 0);
            xf[1][j - 4][1] = read_x(j, 1);
          }
          if (j >= 5) a[j - 5] = pack_state(j - 1);
        });
      }
      if (ADDS) fetch_old(blk);
      barrier_before<8>();  // the scores are read and the output is staged (the eight youngest reads may be on their way)
      auto second_half = [&](int j) __attribute__((always_inline)) {
        decay_state(2 + (j >> 2), 4 * (j & 3), bd);
        yf0[j >> 1][j & 1] = read_y(set + L::Y, y_lane, j & 1, j >> 1);
        scale_z(zn, zs, kd[j >> 2], j >> 2, j & 3);
        if (j == 4) read_kdec(2, len, kd[2]), read_kdec(3, len, kd[3]);
      };
      a[3] = pack_state(7);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        slot(term[j & 1], a[j >> 1], xf[1][j >> 1][j & 1], [&]() __attribute__((always_inline)) { second_half(j); });
      // (3) state update, the lower half of the rows
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int u = j >> 1, T = j & 1;
        slot(st[T], yf0[u][T], zs[u], [&]() __attribute__((always_inline)) {
          if (j < 4) scale_z(zn, zs, kd[2], 2, j), scale_z(zn, zs, kd[3], 3, j);
          if (j < 4) {
            yf1[j][0] = read_y(set + L::Y, y_lane, 2, j);
            yf1[j][1] = read_y(set + L::Y, y_lane, 3, j);
          }
        });
      }
#pragma unroll
      for (int I = 0; I < 2; ++I) {
        acc[I] = term[I];
        qd[I] = qn[I];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) zf[u] = zn[u];
    }
    __syncthreads();
  }
  {
    u32x4 sf[4][2], o;
    read_scores(smem + L::SC, sf);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (LEAVES_STATE) st[2 + (j & 1)] = E::mfma(yf1[j >> 1][j & 1], zs[j >> 1], st[2 + (j & 1)]);
      scale_acc(j);
    }
#pragma unroll
    for (int j = 0; j < 6; ++j)
      acc[INTRA_I[REV][j]] = E::mfma(zf[INTRA_U[REV][j]], sf[INTRA_U[REV][j]][INTRA_I[REV][j]], acc[INTRA_I[REV][j]]);
#pragma unroll
    for (int j = 0; j < 8; ++j) pack_out(acc, FIRST, j, smem + (set_i == 0 ? 2 : set_i - 1) * L::SET + L::X, o);
    __syncthreads();
  }
  // the segment visited last leaves the chunk's outgoing state
  if (SRC != SRC_SCANNED && !TRANS && carry_out != nullptr && sw.seg == (REV ? 0 : g.n_seg - 1)) {
    float *cp = carry_out + (int64_t)sw.bh * g.dt * g.e, *tp = g.twin ? g.twin + (int64_t)sw.bh * g.dt * g.e : nullptr;
#pragma unroll
    for (int T = 0; T < 4; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * T + 16 * (r >> 3) + 8 * hh + 4 * ((r >> 2) & 1) + (r & 3);
        if (!NARROW || (row < fa && col < fb)) {
          cp[row * (NARROW ? fb : W) + col] = st[T][r];
          if (tp) tp[row * (NARROW ? fb : W) + col] = st[T][r];
        }
      }
  }
}

// (both round the same operand of every product and add in the same order: rows of 64 features give the bits of rows extended by zeros)
template <class E, bool REV, bool TRANS, int SRC, int MODE, int W>
__device__ __forceinline__ void
any_body(const elem16_t *__restrict__ X, const elem16_t *__restrict__ Y, const elem16_t *__restrict__ Z,
         const float *__restrict__ S, const float *__restrict__ states, elem16_t *__restrict__ Out, const Geom &g,
         int fa, int fb, int item, char *smem, const float *__restrict__ carry_in,
         float *__restrict__ carry_out = nullptr) {
  if constexpr (W == 128)
    sweep_body<E, REV, TRANS, SRC, MODE>(X, Y, Z, S, states, Out, g, fa, fb, item, smem, carry_in, carry_out);
  else
    ws_body<E, REV, TRANS, SRC, MODE>(X, Y, Z, S, states, Out, g, fa, fb, item, smem, carry_in, carry_out);
}
template <int W>
constexpr int sweep_lds() { return W == 128 ? SweepLds::BYTES : WsLds::BYTES; }

template <class E, bool REV, bool TRANS, int SRC, int MODE, int W>
__global__ void __launch_bounds__(WS_THREADS, ws_waves_per_simd(W))
la_apply(const elem16_t *__restrict__ X, const elem16_t *__restrict__ Y, const elem16_t *__restrict__ Z,
            const float *__restrict__ S, const float *__restrict__ states, const float *__restrict__ carry_in,
            float *__restrict__ carry_out, elem16_t *__restrict__ Out, Geom g) {
  extern __shared__ __align__(16) char smem[];
  // SRC_COMBINE: later segments have more states to gather first, so they are started first
  const int item = SRC == SRC_COMBINE ? g.b * g.h * g.n_seg - 1 - (int)blockIdx.x : (int)blockIdx.x;
  any_body<E, REV, TRANS, SRC, MODE, W>(X, Y, Z, S, states, Out, g, g.d, g.e, item, smem, carry_in, carry_out);
}

// A whole short chunk in one launch: every workgroup rebuilds the state entering its segment (SRC_WALK), so
// there is no pre-pass, no scan and no workspace.  Workgroups are dealt to the 8 XCDs round-robin: all
// segments of one (b, h) go to the same XCD, whose L2 then serves the repeated walks over that (b, h)'s K
// and V; later segments, which walk over more blocks first, are started first.
template <class E, int MODE, int W>
__global__ void __launch_bounds__(WS_THREADS, ws_waves_per_simd(W))
la_fused_fwd(const elem16_t *__restrict__ Q, const elem16_t *__restrict__ K, const elem16_t *__restrict__ V,
                const float *__restrict__ S, const float *__restrict__ kv_in, float *__restrict__ kv_out,
                elem16_t *__restrict__ O, Geom g) {
  extern __shared__ __align__(16) char smem[];
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int group = quotient(slot, g.by_seg), bh = group * 8 + xcd;
  if (bh >= g.b * g.h) return;
  const int item = bh * g.n_seg + (g.n_seg - 1 - (slot - group * g.n_seg));
  any_body<E, false, false, SRC_WALK, MODE, W>(Q, K, V, S, nullptr, O, g, g.d, g.e, item, smem, kv_in, kv_out);
}

// The (b, h) from bh0 on are cut into n_seg segments of their own, unequal ones as `cut` says: see fused_bwd_tail.
struct Fine {
  int bh0, n_seg;
  Divisor by_seg;
  Cut cut;
};

// roles as in la_bwd3 (the dV role leaves dKV_out); all roles and segments of one (b, h) on one XCD.  With g.kept set, kv_in holds the
// scanned states that the forward left, of which dQ takes the one that entered the chunk
template <class E, int MODE, int W>
__global__ void __launch_bounds__(WS_THREADS, ws_waves_per_simd(W))
la_fused_bwd(const elem16_t *__restrict__ Q, const elem16_t *__restrict__ K, const elem16_t *__restrict__ V,
                const elem16_t *__restrict__ DO, const float *__restrict__ S, const float *__restrict__ kv_in,
                const float *__restrict__ dkv_in, float *__restrict__ dkv_out, elem16_t *__restrict__ DQ,
                elem16_t *__restrict__ DK, elem16_t *__restrict__ DV, Geom g, Fine fine) {
  extern __shared__ __align__(16) char smem[];
  const int before = 3 * fine.bh0 * g.n_seg;  // workgroups of the (b, h) before bh0, a multiple of 8
  const bool cut = (int)blockIdx.x >= before;
  if (cut) {
    g.n_seg = fine.n_seg;
    g.by_seg = fine.by_seg;
    g.cut = fine.cut;
  }
  const int local = (int)blockIdx.x - (cut ? before : 0);
  const int xcd = local & 7, slot = local >> 3;
  const int triple = slot / 3, role = slot - 3 * triple;
  const int group = quotient(triple, g.by_seg), bh = (cut ? fine.bh0 : 0) + group * 8 + xcd;
  if (bh >= g.b * g.h) return;
  const int k = triple - group * g.n_seg;  // k-th longest walk of its role
  if (role == 0)
    any_body<E, false, true, SRC_WALK, MODE, W>(DO, V, K, S, nullptr, DQ, g, g.e, g.d, bh * g.n_seg + g.n_seg - 1 - k, smem,
                                            kv_in);
  else if (role == 1)
    any_body<E, true, false, SRC_WALK, MODE, W>(K, Q, DO, S, nullptr, DV, g, g.d, g.e, bh * g.n_seg + k, smem, dkv_in,
                                            dkv_out);
  else
    any_body<E, true, true, SRC_WALK, MODE, W>(V, DO, Q, S, nullptr, DK, g, g.e, g.d, bh * g.n_seg + k, smem, dkv_in);
}

// The three gradients in one launch.  Workgroups come in triples (dQ, dV, dK) that work on the same
// (b*h, segment) and therefore read the same Q, K, V, dO blocks; the triple is spread over block indices 8
// apart so that all three land on the same XCD (workgroups are dealt to the 8 XCDs round-robin) and share
// its L2.
template <class E, int SRC, int MODE, int W>
__global__ void __launch_bounds__(WS_THREADS, ws_waves_per_simd(W))
la_bwd3(const elem16_t *__restrict__ Q, const elem16_t *__restrict__ K, const elem16_t *__restrict__ V,
           const elem16_t *__restrict__ DO, const float *__restrict__ S, const float *__restrict__ kv_states,
           const float *__restrict__ dkv_states, const float *__restrict__ kv_in, const float *__restrict__ dkv_in,
           float *__restrict__ dkv_out, elem16_t *__restrict__ DQ, elem16_t *__restrict__ DK,
           elem16_t *__restrict__ DV, Geom g) {
  extern __shared__ __align__(16) char smem[];
  const int n_items = g.b * g.h * g.n_seg;
  const int grp = blockIdx.x / 24, r = blockIdx.x - grp * 24;
  const int role = r >> 3;
  const int item = n_items - 1 - (grp * 8 + (r & 7));
  if (item < 0) return;
  if (role == 0)
    any_body<E, false, true, SRC, MODE, W>(DO, V, K, S, kv_states, DQ, g, g.e, g.d, item, smem, kv_in);
  else if (role == 1)
    any_body<E, true, false, SRC, MODE, W>(K, Q, DO, S, dkv_states, DV, g, g.d, g.e, item, smem, dkv_in, dkv_out);
  else
    any_body<E, true, true, SRC, MODE, W>(V, DO, Q, S, dkv_states, DK, g, g.e, g.d, item, smem, dkv_in);
}

// ------------------------------------------------------------------------------
// A segment's own state:  causal  sum_b l^(L-b) y_b^T z_b ;  anti-causal  sum_b l^b y_b^T z_b
// (b from the segment start, L its length), written token-free as W x W fp32 (W = 64 or 128).  Y rows hold
// g.d features and Z rows g.e (M_NARROW; W otherwise).
//
// Blocks whose every token carries a weight below 2^-SKIP_LOG2 are neither read nor multiplied:
// with slope s a token that lies x tokens from the segment's far end weighs exp(-s x), so a
// fast-decaying head only needs the last (causal) or first (anti-causal) SKIP_LOG2 ln2 / s tokens
// of each segment.  What is dropped is below 2^-24 of a full-weight term, i.e. under the fp32
// rounding (2^-24) of the sum it would be added to.  s = 0 skips nothing.
//
// That leaves the workgroups unevenly loaded -- those of slow-decaying heads still read whole
// segments -- so one workgroup has to be able to pull more than an even share of the memory
// bandwidth.  512 threads (8 waves): threads 0-255 fetch the Y tile, 256-511 the Z tile, each
// keeping D blocks in flight in registers (16 registers per block) on top of the two LDS
// buffers; wave (wc, rh) owns rows [64 rh, 64 rh + 64) x columns [32 wc, 32 wc + 32) of the state
// as two accumulator tiles.
// W = 64: a step takes two blocks of the walk, i.e. the same bytes, and the four waves that fetch Z (and so have
// nothing to scale) own a 32 x 32 tile of the state each.  The blocks are weighted and added one after the other, as at
// W = 128, so that rows of 64 features give the bits that the same rows zero-extended to 128 give.
//
// Both tiles stay token-major in LDS, as they are in memory (16-byte copies, Y scaled by the decay
// weights on the way); the products contract over tokens, so the MFMA operands are fetched with
// the transposing LDS read.
constexpr int STATE_THREADS = 512;
template <int W>
struct StateLds {
  // Bytes per token row.  The four rows x 64 bytes that one transposing read touches per half-wave fall on
  // disjoint banks: W = 128 rows are 64 bytes longer than the data; W = 64 rows (two to a set of banks) swap their
  // 64-byte halves in every other pair of rows (see row_swap).
  static constexpr int LDR = W == 128 ? 320 : 128;
  static constexpr int BPS = W == 128 ? 1 : 2;  // blocks per step
  static constexpr int TILE = BPS * BLK * LDR;
  static constexpr int BYTES = 2 * 2 * TILE;  // double-buffered {Y scaled, Z}: 80 KiB, W = 64: 64 KiB
  static __device__ __forceinline__ int row_swap(int row) { return W == 128 ? 0 : ((row >> 1) & 1) << 6; }
};
// Blocks in flight per thread in registers (even).  Long walks gain from the deeper pipeline (b*h = 16,
// n = 65536, 2048-token pieces: 46 us per launch against 49); on short ones the longer start-up costs more
// than it gains (320-token segments: 13.1 us against 12.4).  The shallow form stays within 128 registers, so two
// workgroups share a CU; the deep one runs one per CU (squeezed into 128 registers it spills and measured slower).
constexpr int STATE_DEPTH_LONG = 4, STATE_DEPTH_SHORT = 2;
// Tokens per segment up to which every block is read, whatever the decay (forward with a state, b*h = 16, n = 2000, with the
// scan's shorter start-up: 24.1 us against 24.7; eight chained chunks of 2048 tokens, b*h = 24: 624 against 631).  Not where a wide
// head's slices run side by side: several workgroups per CU wait for one another's bytes, not for a slope (b*h = 8, n = 8192,
// d = 256, forward + backward: 186.3 us against 188.6 with every block read).
constexpr int STATE_WHOLE = 512;
constexpr int STATE_LONG_WALK = 1024;  // tokens per segment from which the deeper pipeline is used

// MFMA operand of lane (c, hh): feature f0 + c, tokens t0 + 8 hh .. + 7 (`lane_part` holds the lane's share
// of the address, see la_seg_state; rows LDR bytes apart)
template <int LDR>
__device__ __forceinline__ u32x4 token_fragment(const char *tile, int lane_part, int t0) {
  const char *p = tile + lane_part + t0 * LDR;
  const u32x2 lo = lds_tr8(p), hi = lds_tr8(p + 4 * LDR);
  u32x4 r;
  r.x = lo.x;
  r.y = lo.y;
  r.z = hi.x;
  r.w = hi.y;
  return r;
}

template <class E, bool REV, int MODE, int W, int D>
__global__ void __launch_bounds__(STATE_THREADS, 1)
la_seg_state(const elem16_t *__restrict__ Y, const elem16_t *__restrict__ Z, const float *__restrict__ S,
             float *__restrict__ states, Geom g, int skip_seg, int sub) {
  constexpr bool RAGGED = MODE != M_ALIGNED, NARROW = MODE == M_NARROW;
  using L = StateLds<W>;
  constexpr int BPS = L::BPS;              // blocks per step
  constexpr int NTILE = W == 128 ? 2 : 1;  // 32 x 32 tiles of the state per wave
  constexpr int ROWS = 2048 / W;           // token rows that 256 threads fetch at a time
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index, uniform: keeps it in an SGPR
  const int wc = W == 128 ? w8 & 3 : w8 & 1;                // column block ...
  const int row0s = W == 128 ? 64 * (w8 >> 2) : 32 * ((w8 >> 1) & 1);  // ... and first row of this wave's tiles
  const bool zgrp = w8 >= 4;                                // this wave fetches Z (else Y)
  const int c = lane & 31, hh = lane >> 5;
  // loader: W / 8 consecutive threads copy one row, the thread's 16 bytes are features 8 cq .. + 7 of rows
  // rq + ROWS * {0, 1, 2, 3}
  const int cq = tid & (W / 8 - 1), rq = (tid & 255) / (W / 8);

  // slow-decaying heads (the later ones in the usual slope schedules) have the most to read: first
  const int n_items = g.b * g.h * g.n_seg;
  const SegWork sw = seg_work(g, n_items - 1 - (int)blockIdx.x);
  if (sw.seg == skip_seg) return;  // the scan's final segment feeds only the outgoing carry
  // Short segments are walked whole: the few blocks that a fast-decaying head could leave out delay nobody, while the slope,
  // which says which, would have to arrive before the first load can leave.
  const bool whole = g.seg_len <= STATE_WHOLE && (!NARROW || g.dt <= W);
  const int head = sw.bh - quotient(sw.bh, g.by_h) * g.h;
  int lane_head = head;
  asm volatile("" : "+v"(lane_head));  // (a lane's load, waited for in order; see ws_body)
  const float lane_slope = S[lane_head];
  const float slope = whole ? 0.f : S[head];  // of the decisions which blocks to read
  // Where sweep segments span `sub` > 1 of these segments, a head that takes no part in the scan
  // (state_dies_in_segment) has readers for one state in `sub` only: a sweep reads the own state of the piece
  // next to its segment -- the last piece of the segment before it, or going backwards the first piece of the
  // segment after it -- and the outgoing state, if one is wanted (skip_seg < 0), is formed from the two pieces
  // visited last.  The other pieces are left out, and their slots in `states` unwritten.
  if (sub > 1 && state_dies_in_segment(slope, g)) {
    const int p = sw.seg;
    bool read = REV ? (p % sub == 0 && p >= sub) : (p % sub == sub - 1 && p + 1 < g.n_seg);
    if (skip_seg < 0) read = read || (REV ? p <= 1 : p >= g.n_seg - 2);
    if (!read) return;
  }
  const int64_t row0 = (int64_t)sw.bh * g.n + sw.tok0;
  // the feature slice of a wide head (blockIdx.y; rows of Y are g.dt features apart) and its width
  const int slice = NARROW && W == 128 ? (int)blockIdx.y : 0;
  const int gd = NARROW ? min(W, g.dt - slice * W) : W;
  states += (int64_t)slice * n_items * (W * W);
  const int yp = NARROW ? g.dt : W, zp = NARROW ? g.e : W;  // elements from row to row
  const int tw = NARROW ? (zgrp ? g.e : gd) : W;            // width of the tile this thread fetches
  const elem16_t *Tg = zgrp ? Z + row0 * zp : Y + row0 * yp + slice * W;
  const int row_bytes = (zgrp ? zp : yp) * 2;

  // row r of the thread's four: token row_of(r) of block half_of(r) of the step
  auto half_of = [](int r) { return BPS == 1 ? 0 : r >> 1; };
  auto row_of = [&](int r) __attribute__((always_inline)) { return rq + ROWS * (BPS == 1 ? r : r & 1); };
  u32x4 set[D][4];  // blocks in flight
  float sl, blockdec, kdec[4 / BPS];  // (set once the first loads are on their way)

  // blocks lo..hi of the segment are processed (uniform across the workgroup)
  int lo = 0, hi = sw.nblk - 1;
  if (slope > 0.f) {
    const float keep = SKIP_LOG2 / (slope * LOG2E);  // tokens whose weight is at least 2^-SKIP_LOG2
    if (!REV) {
      // the last token of block t lies (tokens - 64 t - 63) tokens before the segment end
      const float x = ((float)((sw.nblk - 1) * BLK + sw.tail) - 63.f - keep) * (1.f / BLK);
      if (x > 0.f) lo = min((int)ceilf(x), hi);
    } else {
      // the first token of block t lies 64 t tokens after the segment start
      const float x = keep * (1.f / BLK);
      if (x < (float)hi) hi = (int)x;
    }
  }
  // the float arithmetic above ran on the vector unit; put the (uniform) results back in scalar
  // registers so that the block addresses stay scalar
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  const int cnt = hi - lo + 1;

  floatx16 st[NTILE];
#pragma unroll
  for (int T = 0; T < NTILE; ++T)
#pragma unroll
    for (int r = 0; r < 16; ++r) st[T][r] = 0.f;

  // A partial block (the end of a ragged chunk) reads its missing rows as zeros; going
  // forwards it is the last block, and its tokens sit `len - b` (not 64 - b) before the
  // segment end.
  // the thread's four rows (see row_of); chunks past the row width read as zeros
  uint32_t t_off[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) t_off[r] = !NARROW || cq * 8 < tw ? (uint32_t)(row_of(r) * row_bytes + cq * 16) : kOutside;
  const int first = REV ? hi : lo;
  const int step = REV ? -1 : 1;
  auto block_of = [&](int i) __attribute__((always_inline)) { return first + min(i, cnt - 1) * step; };
  auto len_of = [&](int blk) __attribute__((always_inline)) { return RAGGED && blk == sw.nblk - 1 ? sw.tail : BLK; };
  auto issue_loads = [&](u32x4 (&nt)[4], int i) __attribute__((always_inline)) {
#pragma unroll
    for (int half = 0; half < BPS; ++half) {
      const int blk = block_of(BPS * i + half), len = len_of(blk);
      const rows_t rows = rows_of(Tg + (int64_t)blk * BLK * (row_bytes / 2), len * row_bytes);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (half_of(r) == half) nt[r] = __builtin_amdgcn_raw_buffer_load_b128(rows, (int)t_off[r], 0, 0);
    }
  };
  char *const my_rows = smem + (zgrp ? L::TILE : 0) + rq * L::LDR + ((cq * 16) ^ L::row_swap(rq));
  auto fill_lds = [&](int buf, const u32x4 (&nt)[4], int i) __attribute__((always_inline)) {
    char *dst = my_rows + buf * (2 * L::TILE);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int len = len_of(block_of(BPS * i + half_of(r)));
      const bool partial = RAGGED && !REV && len != BLK;
      u32x4 v = nt[r];
      if (!zgrp) v = scaled<E>(v, partial ? decay(sl, (float)max(len - row_of(r), 0)) : kdec[BPS == 1 ? r : r & 1]);
      *reinterpret_cast<u32x4 *>(dst + ROWS * r * L::LDR) = v;
    }
  };
  // M_NARROW: columns past the width of Z stay zero, as do rows past Y's
  const bool wave_active = (W == 128 || zgrp) && (!NARROW || (32 * wc < g.e && row0s < gd));
  // the lane's share of a fragment address: token 8 hh + (lane % 16) / 4, feature 16 ((lane / 16) % 2) + 4 (lane % 4)
  // (rows 4 apart, and the rows of different fragments, share their row_swap)
  const int lane_row = 8 * hh + ((lane & 15) >> 2), lane_feat = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  auto lane_part = [&](int f0) __attribute__((always_inline)) {
    return lane_row * L::LDR + ((2 * (f0 + lane_feat)) ^ L::row_swap(lane_row));
  };
  const int z_part = lane_part(32 * wc);
  int y_part[NTILE];
#pragma unroll
  for (int T = 0; T < NTILE; ++T) y_part[T] = lane_part(row0s + 32 * T);
  auto accumulate = [&](int buf, int i) __attribute__((always_inline)) {
    if (wave_active) {
#pragma unroll
      for (int half = 0; half < BPS; ++half) {
        if (half > 0 && BPS * i + half >= cnt) break;  // an odd block at the end of the walk
        const int len = len_of(block_of(BPS * i + half));
        const float bd = RAGGED && len != BLK ? decay(sl, (float)len) : blockdec;
        const char *yt = smem + buf * (2 * L::TILE) + half * (BLK * L::LDR);
        const char *zt = yt + L::TILE;
        u32x4 zf[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) zf[u] = token_fragment<L::LDR>(zt, z_part, 16 * u);
#pragma unroll
        for (int T = 0; T < NTILE; ++T) {
#pragma unroll
          for (int r = 0; r < 16; ++r) st[T][r] *= bd;
#pragma unroll
          for (int u = 0; u < 4; ++u)
            st[T] = E::mfma(token_fragment<L::LDR>(yt, y_part[T], 16 * u), zf[u], st[T]);
        }
      }
    }
  };

  // Step i of the walk (block i, or blocks 2 i and 2 i + 1) travels through register set i mod D.  Loads and LDS fills
  // past the end of the walk are not skipped but repeat its last block (served by the cache, never
  // used): with the same number of loads in flight on every path, the wait before a fill covers
  // exactly the oldest register set.
#pragma unroll
  for (int k = 0; k < D; ++k) issue_loads(set[k], k);
  __builtin_amdgcn_sched_barrier(0);
  sl = lane_slope * LOG2E;
  blockdec = decay(sl, (float)BLK);
#pragma unroll
  for (int r = 0; r < 4 / BPS; ++r) kdec[r] = decay(sl, REV ? (float)row_of(r) : (float)(BLK - row_of(r)));
  fill_lds(0, set[0], 0);
  issue_loads(set[0], D);
  __syncthreads();
  // The walk leaves the loop from the middle of the unrolled body.  Were the exit test left to the loop
  // head, the compiler would have to assume that any of the D positions can precede the first one, could
  // no longer tell which register set holds the oldest loads there, and would wait for all of them.
  for (int i = 0;; i += D) {
    bool last = false;
#pragma unroll
    for (int k = 0; k < D; ++k) {  // D is even: LDS buffer (i + k) & 1 == k & 1
      accumulate(k & 1, i + k);
      __builtin_amdgcn_sched_barrier(0);
      fill_lds((k + 1) & 1, set[(k + 1) % D], i + k + 1);
      __builtin_amdgcn_sched_barrier(0);
      issue_loads(set[(k + 1) % D], i + k + 1 + D);
      __syncthreads();
      if (BPS * (i + k + 1) >= cnt) {
        last = true;
        break;
      }
    }
    if (last) break;
  }

  if (W == 128 || zgrp)
  {
    float *sp = states + ((int64_t)sw.bh * g.n_seg + sw.seg) * (W * W);
#pragma unroll
    for (int T = 0; T < NTILE; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        sp[(row0s + 32 * T + 8 * (r >> 2) + 4 * hh + (r & 3)) * W + 32 * wc + c] = st[T][r];
  }
}

// What the loads of a sweep leave in the 256 MB memory-side cache.  A forward's q, k and v are read again by the backward, if that follows
// soon, and it begins at the ends of the segments.  Where they exceed the cache, only the last blocks of the segments are loaded as usual, as
// many as have 160 MB; the blocks before them, which would not last, are loaded as data that is read once (`nt`), and come faster for it.
// Forwards, us: b*h = 32, n = 16384 138 -> 126, b*h = 16, n = 65536 245 -> 222, b*h = 64, n = 8192 134 -> 126; with the backward 394 -> 385,
// 732 -> 698, 384 -> 378.  (Forwards one after the other, some of whose tensors the call before left in the cache; with the backwards between
// them and two sets of tensors in turn the sweep itself takes 198 -> 176 at b*h = 16, n = 65536, 6.1 TB/s, and 99 -> 91 at b*h = 32.)  With
// every block read once b*h = 32's forward takes 128 and its backward 16 more.  Tensors that fit the cache lose: b*h = 36, n = 5003, d = e =
// 128, every block read once 164.5 -> 168.1 in both directions, b*h = 16, n = 16384, 160 of 201 MB as usual, 237.7 -> 239.8.  Of 64, 96, 128,
// 160, 192 and 256 MB the forwards are the faster the less stays (b*h = 32: 0.91 of the time with 64, 0.95 with 192), the backwards the slower
// (b*h = 64, n = 4096: 1.03 of both with 64, 0.99 to 1.01 from 96 on).
// In a backward the three roles' workgroups of a round go over their segments' q, k, v and dO at about the same time, dQ's in the other
// direction: where these exceed the cache, dQ's loads leave nothing behind (b*h = 16, n = 65536: both directions 718 -> 706; b*h = 32, n = 16384,
// where they do not, 393 -> 396).
// Non-temporal loads in the pre-pass (0.95 of the speed at d = 256, 0.985 at n = 65536) or in all roles (0.90 to 0.96), and stores that are not
// non-temporal (0.95 to 0.98 beyond 200 MB of tensors) lose.
constexpr int64_t kCacheBytes = (int64_t)256 << 20, kStayBytes = (int64_t)160 << 20;
template <class E, bool REV, bool TRANS, int SRC, int MODE, int W>
int launch_apply(const void *x, const void *y, const void *z, const float *s, const float *states,
                    const float *carry_in, float *carry_out, void *out, const Geom &g_plan, hipStream_t st) {
  int rc = grant_lds<la_apply<E, REV, TRANS, SRC, MODE, W>>(sweep_lds<W>());
  if (rc) return rc;
  Geom g = g_plan;
  const int64_t row = (int64_t)g.b * g.h * 2 * (2 * g.d + g.e);  // bytes of a token's q, k and v
  if (row * g.n > kCacheBytes) g.stay = (int)(kStayBytes / (row * g.n_seg * BLK));
  const unsigned grid = (unsigned)((int64_t)g.b * g.h * g.n_seg);
  ProfScope prof(KC_APPLY, st);
  la_apply<E, REV, TRANS, SRC, MODE, W><<<grid, WS_THREADS, sweep_lds<W>(), st>>>(
      (const elem16_t *)x, (const elem16_t *)y, (const elem16_t *)z, s, states, carry_in, carry_out, (elem16_t *)out, g);
  return (int)hipGetLastError();
}

template <class E, int SRC, int MODE, int W>
int launch_bwd3(const BwdArgs &a, const float *kv_states, const float *dkv_states, const Geom &g_sweep,
                   hipStream_t st) {
  int rc = grant_lds<la_bwd3<E, SRC, MODE, W>>(sweep_lds<W>());
  if (rc) return rc;
  Geom g = g_sweep;
  if (256 / 3 * (int64_t)g.seg_len * 4 * (g.d + g.e) > kCacheBytes) g.stay = 0;  // dQ's
  const int64_t n_items = (int64_t)g.b * g.h * g.n_seg;
  const unsigned grid = (unsigned)(((n_items + 7) / 8) * 24);
  ProfScope prof(KC_BWD3, st);
  la_bwd3<E, SRC, MODE, W><<<grid, WS_THREADS, sweep_lds<W>(), st>>>((const elem16_t *)a.q, (const elem16_t *)a.k,
                                                         (const elem16_t *)a.v, (const elem16_t *)a.d_o, a.s,
                                                         kv_states, dkv_states, a.kv_in, a.dkv_in, a.dkv_out,
                                                         (elem16_t *)a.dq, (elem16_t *)a.dk, (elem16_t *)a.dv, g);
  return (int)hipGetLastError();
}

unsigned slices_of(const Geom &g) { return (unsigned)(g.dt + kMaxWidth - 1) / kMaxWidth; }

template <class E, bool REV, int MODE, int W, int D>
int launch_state_depth(const void *y, const void *z, const float *s, float *states, const Geom &g, int skip_seg,
                       int sub, hipStream_t st) {
  int rc = grant_lds<la_seg_state<E, REV, MODE, W, D>>(StateLds<W>::BYTES);
  if (rc) return rc;
  const unsigned grid = (unsigned)((int64_t)g.b * g.h * g.n_seg);
  ProfScope prof(KC_STATE, st);
  la_seg_state<E, REV, MODE, W, D><<<dim3(grid, slices_of(g)), STATE_THREADS, StateLds<W>::BYTES, st>>>((const elem16_t *)y, (const elem16_t *)z, s,
                                                                        states, g, skip_seg, sub);
  return (int)hipGetLastError();
}

// skip_seg: the segment whose own state nothing reads (-1: none); its workgroups leave at once.
// sub: segments of `g` per sweep segment (1 unless the plan cut the sweep segments finer for the pre-pass).
template <class E, bool REV, int MODE, int W>
int launch_state_skipping(const void *y, const void *z, const float *s, float *states, const Geom &g, int skip_seg,
                          hipStream_t st, int sub = 1) {
  return g.seg_len >= STATE_LONG_WALK
             ? launch_state_depth<E, REV, MODE, W, STATE_DEPTH_LONG>(y, z, s, states, g, skip_seg, sub, st)
             : launch_state_depth<E, REV, MODE, W, STATE_DEPTH_SHORT>(y, z, s, states, g, skip_seg, sub, st);
}

// carry_wanted: whether the scan that follows has to produce the outgoing carry; if not, the
// segment it visits last (whose own state feeds nothing else) is skipped.
template <class E, bool REV, int MODE, int W>
int launch_state(const void *y, const void *z, const float *s, float *states, const Geom &g,
                 bool carry_wanted, int sub, hipStream_t st) {
  return launch_state_skipping<E, REV, MODE, W>(y, z, s, states, g, carry_wanted ? -1 : (REV ? 0 : g.n_seg - 1), st, sub);
}

// How a single launch cuts a (b, h).  Segments of equal length leave the first one's workgroup idle while the last one's walks; so the
// first is the longest (32 blocks in three segments: 16, 10 and 6 and not 11, 11 and 10).  A walk block takes 0.57 us, a swept one 1.35;
// with 30 or 55 instead of 42 % the launches below take 0.99 - 1.09 of their time, with 70 % up to 1.25.  More than eight segments have
// nothing left to do.  In us, equal segments (forwards of 256 tokens, whatever the chip had room for) and these: forwards, b*h = 8, n = 256 8.5
// and 6.5, b*h = 16, n = 1024 17.6 and 15.6, b*h = 20, n = 700 14.7 and 13.2, b*h = 128, n = 1024 44.8 and 33.4, b*h = 160, n = 512 26.9 and
// 20.5; backwards, b*h = 8, n = 256 9.3 and 7.1, b*h = 24, n = 2048 33.2 and 30.2, b*h = 20, n = 1024 20.5 and 18.8, b*h = 36, n = 3000 63.5
// and 61.2; d = e = 64, b*h = 16, n = 1024 14.0 and 12.6 forwards, 13.6 and 13.4 backwards.  Of 31 such shapes none is slower by more than
// 1.6 %.
constexpr int CUT_MOST = 8;
constexpr int CUT_SWEEP = 100, CUT_WALK = 42;  // a block's time, swept and walked over
// A (b, h) of `total` blocks in at most `most` segments, each as long as the walk before it leaves it time: the least time in which that
// covers all of them.
void cut_in(int total, int64_t most, int *n_seg, Divisor *by_seg, Cut *cut) {
  const int m = (int)(most < 1 ? 1 : most > CUT_MOST ? CUT_MOST : most);
  // segments that cover the blocks in `time` (0: they don't), and where they start
  auto cover = [&](int64_t time, uint64_t (&starts)[2]) {
    starts[0] = starts[1] = 0;
    int64_t at = 0;
    for (int k = 0; k < m; ++k) {
      const int64_t len = (time - at * CUT_WALK) / CUT_SWEEP;
      if (len < 1) return 0;
      starts[k >> 2] |= (uint64_t)at << (16 * (k & 3));
      at += len;
      if (at >= total) return k + 1;
    }
    return 0;
  };
  uint64_t starts[2];
  int64_t lo = 0, hi = (int64_t)total * CUT_SWEEP;  // too little, enough
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) / 2;
    (cover(mid, starts) ? hi : lo) = mid;
  }
  const int k = cover(hi, starts);
  // equal segments take as long for a head that walks over this many blocks
  const int64_t spare = hi - (int64_t)((total + k - 1) / k) * CUT_SWEEP;
  *n_seg = k;
  *by_seg = divisor_of((uint32_t)k);
  *cut = Cut{starts[0], starts[1], k > 1 ? (int)(spare / CUT_WALK) + 1 : 0};
}
int blocks_of(const Geom &g) { return (int)((g.n + BLK - 1) / BLK); }

template <class E, int MODE, int W>
int launch_fused_fwd(const FwdArgs &a, const Geom &g_plan, hipStream_t st) {
  int rc = grant_lds<la_fused_fwd<E, MODE, W>>(sweep_lds<W>());
  if (rc) return rc;
  Geom g = g_plan;
  const int64_t bh8 = ((int64_t)g.b * g.h + 7) / 8 * 8;
  // (one segment that takes a state may be asked to leave it in its place: no other workgroup may have to read it)
  if (!(g.n_seg == 1 && a.kv_in)) cut_in(blocks_of(g), (W == 64 ? 512 : 256) / bh8, &g.n_seg, &g.by_seg, &g.cut);
  const unsigned grid = (unsigned)(bh8 * g.n_seg);  // whole groups of 8 (b, h)
  ProfScope prof(KC_FUSED, st);
  la_fused_fwd<E, MODE, W><<<grid, WS_THREADS, sweep_lds<W>(), st>>>((const elem16_t *)a.q, (const elem16_t *)a.k,
                                                         (const elem16_t *)a.v, a.s, a.kv_in, a.kv_out,
                                                         (elem16_t *)a.o, g);
  return (int)hipGetLastError();
}

// The backward's three workgroups per segment should fit the chip in one round (one workgroup per CU, two at W = 64), and
// nothing ties its segments to the forward's: no states are handed over on this path.
// All workgroups of a (b, h) run on one XCD, so from 20 (b, h) on it is the XCDs with most of them that have to have the places: bf16,
// d = e = 128, counted over the chip and by XCD: b*h = 20, n = 1024 27.5 and 22.6 us, b*h = 25, n = 768 23.9 and 19.9, b*h = 28, n =
// 1024 27.9 and 25.0, b*h = 42, n = 2048 61.6 and 57.8.  Fewer (b, h) have more, shorter segments, and those that wait for a place are
// the ones without a walk: b*h = 12, n = 1024 20.1 and 20.6, b*h = 18 21.6 and 22.2.  At W = 64 the two count alike (14.7 and 15.0 at
// worst).
constexpr int64_t kFitByXcd = 20;
int64_t fused_bwd_fit(const Geom &g) {  // segments per (b, h) in one round
  const int64_t bh = (int64_t)g.b * g.h, placed = g.width == 128 && bh >= kFitByXcd ? (bh + 7) / 8 * 8 : bh;
  return (g.width == 64 ? 512 : 256) / (3 * placed);
}
Geom fused_bwd_geom(const Geom &g) {
  Geom gb = g;
  cut_in(blocks_of(g), fused_bwd_fit(g), &gb.n_seg, &gb.by_seg, &gb.cut);
  return gb;
}

// Where whole chunks fill more than one round of the chip, the workgroups of the last, partly filled round would take as
// long as a full one.  Their (b, h) are cut into as many segments as fill the places that are left: walks over the blocks before
// a segment cost less than half of sweeping them.  Backward kernel, bf16, uncut and cut.  d = e = 128: n = 512, b*h = 88: 35.4 and
// 25.2 us, 96: 35.3 and 28.9, 120 (two segments only): 35.8 and 33.0, 172: 53.0 and 43.9; n = 1024, b*h = 96: 67.8 and 51.6, 120:
// 70.8 and 69.6; never slower over b*h = 88 ... 512, n = 64 ... 1536.  At W = 128 the places are counted by XCD (see fused_bwd_geom):
// 81 to 85 (b, h) overflow one of them, though 3 b*h <= 256 (b*h = 84: n = 512 uncut 34.9, cut 26.9; n = 2048 127 and 88), as 169 and
// 170 do with two rounds (n = 2048: 198 and 178).  d = e = 64: the places count one workgroup per CU, not
// two: a last round of at most 256 has the CUs to itself and runs at up to twice the pace of a full one, which is all that cutting
// it further can win (n = 1024: b*h = 171 uncut 50.2, cut for one per CU 38.5, for two 40.6; 200: 52.6, 50.4 and 51.1; 216, left
// uncut with one per CU: 53.8 and 57.1; 240: 58.3 and 63.9).
Fine fused_bwd_tail(const Geom &g) {
  const int64_t bh = (int64_t)g.b * g.h, slots = g.width == 64 ? 512 : 256, placed = g.width == 64 ? bh : (bh + 7) / 8 * 8;
  Fine f = {(int)((bh + 7) / 8 * 8), g.n_seg, g.by_seg, g.cut};  // nothing is cut
  if (g.n_seg > 1 || 3 * placed <= slots) return f;
  const int64_t whole = 3 * placed / slots * slots;  // workgroups in whole rounds
  const int64_t bh0 = whole / 24 * 8;            // whole groups of 8
  const int64_t rest = (bh - bh0 + 7) / 8 * 8, room = 256 + (g.width == 64 ? 0 : whole - 3 * bh0);
  if (rest <= 0 || room / (3 * rest) < 2) return f;
  cut_in(blocks_of(g), room / (3 * rest), &f.n_seg, &f.by_seg, &f.cut);
  if (f.n_seg > 1) f.bh0 = (int)bh0;
  return f;
}

template <class E, int MODE, int W>
int launch_fused_bwd(const BwdArgs &a, const Geom &g_fwd, hipStream_t st) {
  int rc = grant_lds<la_fused_bwd<E, MODE, W>>(sweep_lds<W>());
  if (rc) return rc;
  const Geom g = fused_bwd_geom(g_fwd);
  const Fine fine = fused_bwd_tail(g);
  const int64_t tail8 = ((int64_t)g.b * g.h - fine.bh0 + 7) / 8 * 8;
  const unsigned grid = (unsigned)(3 * ((int64_t)fine.bh0 * g.n_seg + tail8 * fine.n_seg));
  ProfScope prof(KC_FUSED, st);
  la_fused_bwd<E, MODE, W><<<grid, WS_THREADS, sweep_lds<W>(), st>>>((const elem16_t *)a.q, (const elem16_t *)a.k,
                                                         (const elem16_t *)a.v, (const elem16_t *)a.d_o, a.s,
                                                         a.kv_in, a.dkv_in, a.dkv_out, (elem16_t *)a.dq,
                                                         (elem16_t *)a.dk, (elem16_t *)a.dv, g, fine);
  return (int)hipGetLastError();
}

// The geometry the pre-pass and the scan work on: the chunk cut into g.pre_n segments of g.pre_len tokens
// (the sweeps' own segments unless the plan cut those finer for the pre-pass).
Geom pre_pass_geom(const Geom &g) {
  Geom gp = g;
  gp.seg_len = g.pre_len;
  gp.n_seg = g.pre_n;
  gp.by_seg = divisor_of((uint32_t)gp.n_seg);
  return gp;
}

// A wide head (d > 128) is swept one slice of 128 features of q and k after the other, straight from and to their rows
// (b*h = 8, n = 8192, d = 256, e = 128, forward + backward: 197 us, against 383 with slices copied out and summed outside):
// the scores and the state terms are sums over features, so every slice after the first adds its part of O (dV) to
// what is there, while dQ, dK and the states fall apart into slices.  The pre-pass and the scan take all slices in one launch.
Geom slice_geom(const Geom &g, int i) {
  Geom gs = g;
  gs.d = g.dt - i * kMaxWidth < kMaxWidth ? g.dt - i * kMaxWidth : kMaxWidth;
  if (g.twin) gs.twin = g.twin + (int64_t)i * kMaxWidth * g.e;
  return gs;
}
const void *row_slice(const void *p, int i) { return (const elem16_t *)p + i * kMaxWidth; }
void *row_slice(void *p, int i) { return (elem16_t *)p + i * kMaxWidth; }
template <class T>  // of the chunk's d x e states
T *carry_slice(T *p, const Geom &g, int i) { return p ? p + (int64_t)i * kMaxWidth * g.e : p; }
template <class T>  // of the workspace
T *state_slice(T *p, const Geom &g, int i) {
  return p ? p + (int64_t)i * g.b * g.h * g.pre_n * kMaxWidth * kMaxWidth : p;
}
FwdArgs slice_args(const FwdArgs &a, const Geom &g, int i) {
  FwdArgs r = a;
  r.q = row_slice(a.q, i);
  r.k = row_slice(a.k, i);
  r.kv_in = carry_slice(a.kv_in, g, i);
  r.kv_out = carry_slice(a.kv_out, g, i);
  return r;
}
BwdArgs slice_args(const BwdArgs &a, const Geom &g, int i) {
  BwdArgs r = a;
  r.q = row_slice(a.q, i);
  r.k = row_slice(a.k, i);
  r.dq = row_slice(a.dq, i);
  r.dk = row_slice(a.dk, i);
  r.kv_in = carry_slice(a.kv_in, g, i);
  r.dkv_in = carry_slice(a.dkv_in, g, i);
  r.dkv_out = carry_slice(a.dkv_out, g, i);
  return r;
}

template <class E, int MODE, int W>
int fwd_e(const FwdArgs &a, const Geom &g, hipStream_t st) {
  int rc = 0;
  const int slices = (int)slices_of(g);
  if (g.fused) {
    rc = launch_fused_fwd<E, MODE, W>(slice_args(a, g, 0), slice_geom(g, 0), st);
    if constexpr (MODE == M_NARROW && W == kMaxWidth)
      for (int i = 1; i < slices && !rc; ++i) rc = launch_fused_fwd<E, M_ADDING, W>(slice_args(a, g, i), slice_geom(g, i), st);
    return rc;
  }
  if constexpr (MODE != M_NARROW) if (g.combine) {  // (the plan combines full-width heads only)
    // few segments: the pre-pass leaves every segment's own state (the last one's is never read), each
    // sweep workgroup gathers the ones before it, and the last segment's sweep ends with KV_out
    if (g.n_seg > 1 &&
        (rc = launch_state_skipping<E, false, MODE, W>(a.k, a.v, a.s, a.seg_states, g, g.n_seg - 1, st)))
      return rc;
    return launch_apply<E, false, false, SRC_COMBINE, MODE, W>(a.q, a.k, a.v, a.s, g.n_seg > 1 ? a.seg_states : nullptr,
                                                               a.kv_in, a.kv_out, a.o, g, st);
  }
  const bool need_states = g.n_seg > 1 || a.kv_in || a.kv_out;
  const Geom gp = pre_pass_geom(g);
  const int sub = g.seg_len / g.pre_len;  // pre-pass segments per sweep segment
  if (need_states) {
    if ((rc = launch_state<E, false, MODE, W>(a.k, a.v, a.s, a.seg_states, gp, a.kv_out != nullptr, sub, st))) return rc;
    if ((rc = launch_segment_scan(a.seg_states, a.kv_in, a.kv_out, a.s, gp, 0, st))) return rc;
  }
  auto sweep = [&](auto mode, int i) {
    const FwdArgs as = slice_args(a, g, i);
    return launch_apply<E, false, false, SRC_SCANNED, decltype(mode)::value, W>(
        as.q, as.k, as.v, as.s, need_states ? state_slice(as.seg_states, g, i) : nullptr, as.kv_in, nullptr, as.o,
        slice_geom(g, i), st);
  };
  rc = sweep(std::integral_constant<int, MODE>(), 0);
  if constexpr (MODE == M_NARROW && W == kMaxWidth)
    for (int i = 1; i < slices && !rc; ++i) rc = sweep(std::integral_constant<int, M_ADDING>(), i);
  return rc;
}

// Chunks whose forward takes pre-pass, scan and sweep run their backward in one launch all the same where that is faster: it reads q
// and dO once less, passes no states through memory, and three workgroups per segment fill the chip with a third of the segments,
// so that little is walked twice.  Its time goes with the chunk's length, as a workgroup walks and sweeps all of it, that of the
// three kernels with n b h: no chunk beyond n = 88 b*h.  Up to there, bf16, backward with states, three kernels and one launch in us:
//   Whole rows, all (b, h) in one round (up to 80): always.  b*h = 24, n = 2048 40.9 and 35.1, n = 2112 42 and 37; b*h = 36, n = 2048
// 59.0 and 42.3; b*h = 48, n = 4224 118 and 111 (the nearest); b*h = 60, n = 4096 131 and 119; b*h = 80, n = 6144 247 and 234.
//   Whole rows, more rounds than one: the three kernels come down to few, well-filled rounds too, above all where they gather four
// segments or fewer.  Up to 4096 tokens the one launch is at worst even (b*h = 104: 216 and 217) and as a rule faster (b*h = 88,
// n = 3072 154 and 149, b*h = 112, n = 4096 239 and 227, b*h = 160, n = 3072 257 and 222); beyond, it is where they scan and b*h > 128
// (b*h = 144, n = 6144 449 and 425, b*h = 192, n = 5003 500 and 479), and elsewhere it may lose what it wins (b*h = 128, n = 4608 296
// and 305, n = 6144 386 and 400, b*h = 192, n = 4608 423 and 441, b*h = 168, n = 5632 443 and 454, but b*h = 144, n = 4608 348 and 322,
// b*h = 256 573 and 547).  81 to 85 (b, h) are one round of three segments for the three kernels and one and a half here: up to
// 2560 tokens (b*h = 84 120 and 103; b*h = 82 118 and 120, n = 3072 135 and 141).
//   Narrow rows, whose three kernels scan whatever the number of segments: with more rounds than one always (d = e = 96, b*h = 128,
// n = 3072 185 and 160, b*h = 84, n = 4096 154 and 133); with one, by the blocks that a workgroup of either form goes through in a row --
// one launch a segment and the longest walk before it, at 0.35 of a block swept, the three kernels their rounds of segments, three
// blocks more for each start, and pre-pass and scan.  Fitted over 631 shapes, four widths (b*h = 18 ... 80, n = 1100 ... 6144), 4 %
// off at one deviation.  d = 128, e = 64: b*h = 24, n = 2048 40.1 and 38.5; b*h = 28, n = 2464 45 and 47; b*h = 44, n = 3872 91 and 96;
// b*h = 60, n = 4096 132 and 102.
// Of 1034 measured shapes 831 take one launch, the slowest beside its three kernels at 1.024.  Heads of up to 64 features stay (b*h = 24,
// n = 2048: 23.1 and 29.1).
// DKV_out is summed over the whole chunk in one accumulator of 32 bits: without decay, b*h = 24, n = 2048, it is 2.9e-7 off (2-norm, against
// 64 bits) where sums of segments are 1.0e-7, at n = 6144, b*h = 80, 5.0e-7 and 4.3e-7; as chunks of that length are in one launch
// of either direction.  With decay it is 1.6e-3 off either way (bf16), the rounding of its decayed operand, and no other output differs.
// Only with the segments of the library's own plan (others are asked for to get the three kernels), and not where the
// outgoing state lies over an incoming one: nothing orders the workgroup that writes it and those that read the other.
constexpr int64_t kWholeBwdPerHead = 88, kWholeBwdMax = 6144;
constexpr int64_t kWholeBwdRounds = 4096, kWholeBwdOverXcd = 2560, kWholeBwdMany = 128;
bool whole_bwd_pays(const Geom &g) {
  const int64_t bh = (int64_t)g.b * g.h, placed = (bh + 7) / 8 * 8;
  if (g.n > kWholeBwdMax || g.n > kWholeBwdPerHead * bh) return false;
  const bool one_round = 3 * placed <= 256;
  if (g.dt == kMaxWidth && g.e == kMaxWidth) {
    if (one_round) return true;
    if (3 * bh <= 256) return g.n <= kWholeBwdOverXcd;
    return g.n <= kWholeBwdRounds || (bh > kWholeBwdMany && !g.combine);
  }
  if (!one_round) return true;
  // (counted with segments of equal length, as when the rule was fitted)
  const int64_t fit = fused_bwd_fit(g), segs = fit < 1 ? 1 : fit < g.n_seg ? fit : g.n_seg, seg_blk = (blocks_of(g) + segs - 1) / segs;
  const double len = fit < g.n_seg ? (double)seg_blk : g.seg_len / BLK, walk = ((fit < g.n_seg ? (blocks_of(g) + seg_blk - 1) / seg_blk : g.n_seg) - 1) * len;
  const double blocks = blocks_of(g);
  const double rounds = (double)((3 * bh * g.n_seg + 255) / 256);
  const double three = rounds * (g.seg_len / BLK + 3) + (double)(bh * g.n_seg) / 13 + (double)bh * blocks / 116;
  return 1.44 * (len + 0.35 * walk) + 6 < three;
}
bool whole_bwd(const BwdArgs &a, const Geom &g) {
  if (!a.planned || g.width != kMaxWidth || g.dt > kMaxWidth || !whole_bwd_pays(g)) return false;
  const size_t bytes = sizeof(float) * (size_t)g.b * g.h * g.dt * g.e;
  auto apart = [&](const float *in, const float *out) {
    const uintptr_t i = (uintptr_t)in, o = (uintptr_t)out;
    return !in || !out || i + bytes <= o || o + bytes <= i;
  };
  return apart(a.dkv_in, a.dkv_out) && apart(a.kv_in, a.dkv_out) && apart(a.kv_in, g.twin);
}

// A forward that keeps no states may run in one launch as well, where the three kernels are not faster: each workgroup walks or sweeps all
// of its (b, h), so again up to n = 88 b*h (80 for narrow rows) and 6144 tokens.  Up to 64 (b, h) and beyond 4096 tokens four gathered
// segments fill the chip as well (b*h = 60, n = 4700 75.8 and 79.7 us).  bf16, forward with states, three kernels and one launch in us:
// b*h = 24, n = 2048 27.9 and 24.9, b*h = 48, n = 2048 39.9 and 28.2, b*h = 64, n = 3100 61.9 and 57.2, b*h = 56, n = 3600 62.6 and 61.8 (the
// nearest), b*h = 112, n = 3600 115 and 99, b*h = 200, n = 5400 295 and 222; d = 96, b*h = 80, n = 2600 72.9 and 47.1.  Of 160 shapes that
// take it (four widths, b*h = 13 ... 512, n = 1100 ... 6144) the slowest is at 1.006 of its three kernels, the mean at 0.84.
// KV_out is one sum over the whole chunk, as DKV_out is backwards: without decay 2.9e-7 off 64 bits at b*h = 24, n = 2048 where sums of
// segments are 1.0e-7, 5.0e-7 and 3.7e-7 at b*h = 120, n = 6000, so the operators take it only where no state leaves; with decay 1.66e-3
// (bf16) and 2.07e-4 (fp16) either way, the rounding of its operand, and O 1.7e-3 to 2.7e-3 either way.
constexpr int64_t kWholeFwdNarrow = 80, kWholeFwdGathered = 64;
bool whole_fwd_pays(const Geom &g) {
  const int64_t bh = (int64_t)g.b * g.h;
  const bool full = g.dt == kMaxWidth && g.e == kMaxWidth;
  if (g.n > kWholeBwdMax || g.n > (full ? kWholeBwdPerHead : kWholeFwdNarrow) * bh) return false;
  return !full || bh > kWholeFwdGathered || g.n <= kWholeBwdRounds;
}

// Segments of the backward sweeps: m of the plan's in a row.  The plan's segments give the forward a workgroup per CU; three roles of them
// take one round and a half to three, each with its start-up -- the first tiles, the entering state, the last stores -- of about five
// blocks' time, and half of a last round is empty.  The states lie at the plan's segments either way (a sweep takes the one that enters its
// first), so the forward, the pre-passes and the scans stay as they are but for the states that nothing reads.  m is the one with the least
// rounds x (blocks + 5), a round being 32 workgroups on each XCD, as launch_bwd3 deals items out, if that saves 3 %.  bf16, backward with kept
// states, us, m = 1 and m: b*h = 4, n = 8192 38.2 and 34.0 (m = 2: one round of 8 blocks for two of 4), b*h = 8, n = 3784 35.5 and 31.1 (2),
// b*h = 16, n = 8192 87.9 and 81.2 (4: one round of 32 for three of 8), b*h = 20, n = 3757, d = 96 52.7 and 43.3 (3), b*h = 16, n = 1536, d =
// 192 55.9 and 47.9 (2). A last segment of the plan's less than a fifth full makes no round of its own (b*h = 10, n = 8226: 3.4 % slower with
// m = 3).  Over 225 shapes (b*h = 3 ... 48, n = 1523 ... 31484) 0.956 of the time on average, 0.954 with the best m of each, none slower.
// Slices of a wide head, whose sweeps fetch narrow rows, lose from 28 blocks on (b*h = 32, n = 4096, d = 256 1.012 and up).  Heads of up to 64
// features run two workgroups to a CU and lose with any m (1.03 and up on 24 shapes).
// Tried: DKV states as far apart as the sweeps start, which only they read (b*h = 8, n = 8192, d = 256 102.2 and 94.8 us backwards).  DKV_out is
// then a sum of longer pieces, without decay up to 1.13 times as far from 64 bits (fp16, b*h = 16, n = 1536, d = 192 1.09e-7 and 0.96e-7), and
// where that keeps to calls that leave no state, gradients depend on whether one is asked for.
constexpr int kSweepStart = 5, kSweepBlocks = 40, kSweepBlocksSlice = 24, kSweepRow = 8;
template <int W>
Geom bwd_sweep_geom(const Geom &g) {
  Geom gs = g;
  if (W != kMaxWidth) return gs;
  const int64_t blk = g.seg_len / BLK, most = g.dt > kMaxWidth ? kSweepBlocksSlice : kSweepBlocks;
  const bool sliver = g.n_seg > 1 && (g.n - (int64_t)(g.n_seg - 1) * g.seg_len) * 5 < g.seg_len;
  auto cost = [&](int m) {
    const int segs = m > 1 ? (g.n_seg + m - 1) / m : sliver ? g.n_seg - 1 : g.n_seg;
    const int64_t items = (int64_t)g.b * g.h * segs, per_xcd = 3 * ((items + 7) / 8);
    return (per_xcd + 31) / 32 * (m * blk + kSweepStart);
  };
  int best = 1;
  for (int m = 2; m <= kSweepRow && m <= g.n_seg && m * blk <= most; ++m)
    if (best == 1 ? cost(m) * 100 < cost(1) * 97 : cost(m) < cost(best)) best = m;
  gs.seg_len = best * g.seg_len;
  gs.n_seg = (g.n_seg + best - 1) / best;
  gs.by_seg = divisor_of((uint32_t)gs.n_seg);
  return gs;
}

template <class E, int MODE, int W>
int bwd_e(const BwdArgs &a, const Geom &g, hipStream_t st) {
  int rc = 0;
  const int slices = (int)slices_of(g);
  if (g.fused) {
    rc = launch_fused_bwd<E, MODE, W>(slice_args(a, g, 0), slice_geom(g, 0), st);
    if constexpr (MODE == M_NARROW && W == kMaxWidth)
      for (int i = 1; i < slices && !rc; ++i) rc = launch_fused_bwd<E, M_ADDING, W>(slice_args(a, g, i), slice_geom(g, i), st);
    return rc;
  }
  if (whole_bwd(a, g)) {
    // Kept states say what entered the chunk, whatever kv_in's memory holds by now (gathered ones do not: there kv_in is read, as
    // their sweeps do).  They come in kv_in's place: a pointer of their own among the kernel's arguments, read before the state can
    // be, took the launch at b*h = 16, n = 1024 from 19.4 to 19.9 us.
    BwdArgs aw = a;
    Geom gw = slice_geom(g, 0);
    if (a.kv_seg_states && !g.combine) {
      gw.kept = a.kv_in ? KEPT_STATES : KEPT_STATES_ONLY;
      aw.kv_in = a.kv_seg_states;
    }
    return launch_fused_bwd<E, MODE, W>(aw, gw, st);
  }
  if constexpr (MODE != M_NARROW) if (g.combine) {
    const float *kv_states = a.kv_seg_states;
    if (!kv_states && g.n_seg > 1) {
      if ((rc = launch_state_skipping<E, false, MODE, W>(a.k, a.v, a.s, a.ws_kv, g, g.n_seg - 1, st))) return rc;
      kv_states = a.ws_kv;
    }
    if (g.n_seg > 1 && (rc = launch_state_skipping<E, true, MODE, W>(a.q, a.d_o, a.s, a.ws_dkv, g, 0, st))) return rc;
    return launch_bwd3<E, SRC_COMBINE, MODE, W>(a, g.n_seg > 1 ? kv_states : nullptr,
                                                g.n_seg > 1 ? a.ws_dkv : nullptr, g, st);
  }
  const Geom gp = pre_pass_geom(g), gw = bwd_sweep_geom<W>(g);
  const int sub = gw.seg_len / g.pre_len;  // pre-pass segments per sweep segment
  const float *kv_states = a.kv_seg_states;
  if (!kv_states && (g.n_seg > 1 || a.kv_in)) {
    if ((rc = launch_state<E, false, MODE, W>(a.k, a.v, a.s, a.ws_kv, gp, false, sub, st))) return rc;
    if ((rc = launch_segment_scan(a.ws_kv, a.kv_in, nullptr, a.s, gp, 0, st))) return rc;
    kv_states = a.ws_kv;
  }
  const float *dkv_states = nullptr;
  if (g.n_seg > 1 || a.dkv_in || a.dkv_out) {
    if ((rc = launch_state<E, true, MODE, W>(a.q, a.d_o, a.s, a.ws_dkv, gp, a.dkv_out != nullptr, sub, st))) return rc;
    if ((rc = launch_segment_scan(a.ws_dkv, a.dkv_in, a.dkv_out, a.s, gp, 1, st))) return rc;
    dkv_states = a.ws_dkv;
  }
  auto sweep = [&](auto mode, int i) {
    return launch_bwd3<E, SRC_SCANNED, decltype(mode)::value, W>(slice_args(a, g, i), state_slice(kv_states, g, i),
                                                                 state_slice(dkv_states, g, i), slice_geom(gw, i), st);
  };
  rc = sweep(std::integral_constant<int, MODE>(), 0);
  if constexpr (MODE == M_NARROW && W == kMaxWidth)
    for (int i = 1; i < slices && !rc; ++i) rc = sweep(std::integral_constant<int, M_ADDING>(), i);
  return rc;
}


// rows of g.sd = g.se features (64 or 128) run without the bookkeeping of narrower ones and of slices
int mode_of(const Geom &g) {
  if (g.dt != g.sd || g.e != g.se) return M_NARROW;
  return g.n % BLK != 0 ? M_RAGGED : M_ALIGNED;
}

template <class E, int W>
int fwd_m(const FwdArgs &a, const Geom &g, hipStream_t st) {
  switch (mode_of(g)) {
    case M_ALIGNED: return fwd_e<E, M_ALIGNED, W>(a, g, st);
    case M_RAGGED: return fwd_e<E, M_RAGGED, W>(a, g, st);
    default: return fwd_e<E, M_NARROW, W>(a, g, st);
  }
}
template <class E, int W>
int bwd_m(const BwdArgs &a, const Geom &g, hipStream_t st) {
  switch (mode_of(g)) {
    case M_ALIGNED: return bwd_e<E, M_ALIGNED, W>(a, g, st);
    case M_RAGGED: return bwd_e<E, M_RAGGED, W>(a, g, st);
    default: return bwd_e<E, M_NARROW, W>(a, g, st);
  }
}
template <class E>
int fwd_w(const FwdArgs &a, const Geom &g, hipStream_t st) {
  return g.width == 64 ? fwd_m<E, 64>(a, g, st) : fwd_m<E, 128>(a, g, st);
}
template <class E>
int bwd_w(const BwdArgs &a, const Geom &g, hipStream_t st) {
  return g.width == 64 ? bwd_m<E, 64>(a, g, st) : bwd_m<E, 128>(a, g, st);
}
template <class E>
int whole_fwd_w(const FwdArgs &a, const Geom &g, hipStream_t st) {
  switch (mode_of(g)) {
    case M_ALIGNED: return launch_fused_fwd<E, M_ALIGNED, kMaxWidth>(a, g, st);
    case M_RAGGED: return launch_fused_fwd<E, M_RAGGED, kMaxWidth>(a, g, st);
    default: return launch_fused_fwd<E, M_NARROW, kMaxWidth>(a, g, st);
  }
}

}  // namespace

// This file is compiled once per element type: as it stands for bf16, and through lasp_mfma_f16.hip for fp16.
#ifdef LASP_MFMA_F16
int mfma_f16_fwd(const FwdArgs &a, const Geom &g, hipStream_t st) { return fwd_w<ElemF16>(a, g, st); }
int mfma_f16_bwd(const BwdArgs &a, const Geom &g, hipStream_t st) { return bwd_w<ElemF16>(a, g, st); }
int mfma_f16_whole_fwd(const FwdArgs &a, const Geom &g, hipStream_t st) { return whole_fwd_w<ElemF16>(a, g, st); }
#else
int mfma_fwd(const FwdArgs &a, const Geom &g, int dtype, hipStream_t st) {
  return dtype == LASP_DTYPE_F16 ? mfma_f16_fwd(a, g, st) : fwd_w<ElemBF16>(a, g, st);
}
int mfma_bwd(const BwdArgs &a, const Geom &g, int dtype, hipStream_t st) {
  return dtype == LASP_DTYPE_F16 ? mfma_f16_bwd(a, g, st) : bwd_w<ElemBF16>(a, g, st);
}
int mfma_bwd_row(const Geom &g, bool planned) {
  if (g.fused || g.combine || (planned && g.width == kMaxWidth && g.dt <= kMaxWidth && whole_bwd_pays(g))) return 0;
  return (g.width == 64 ? bwd_sweep_geom<64>(g) : bwd_sweep_geom<kMaxWidth>(g)).seg_len;
}
bool mfma_whole(const Geom &g, bool backward_follows) {
  return !g.fused && g.width == kMaxWidth && g.dt <= kMaxWidth && whole_fwd_pays(g) && (!backward_follows || whole_bwd_pays(g));
}
int mfma_whole_fwd(const FwdArgs &a, const Geom &g, int dtype, hipStream_t st) {
  return dtype == LASP_DTYPE_F16 ? mfma_f16_whole_fwd(a, g, st) : whole_fwd_w<ElemBF16>(a, g, st);
}
#endif

}  // namespace lasp
