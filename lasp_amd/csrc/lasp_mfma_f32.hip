// fp32 MFMA kernels for d, e <= 128, laid out for 128 (gfx950, wave64): the same decomposition
// as the 16-bit kernels -- one routine evaluates a causal or anti-causal decayed linear
// attention over a segment given the state entering it, and the four outputs of the
// operator are instances of it (O: x=Q y=K z=V; dQ: x=dO y=V z=K with the state transposed;
// dV: x=K y=Q z=dO anti-causal; dK: x=V y=dO z=Q anti-causal, state transposed) -- but with
// full-precision arithmetic, for inputs whose tolerance (1e-3) rules out 16-bit operands.
//
// The matrix unit multiplies fp32 at a sixteenth of its bf16 rate, so every operand is split into three bf16 numbers (Henry,
// Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019), x = h
// + m + l: h is x cut off after 8 bits, m what is left rounded to 8 bits, l the rest.  The three hold x exactly from 2^-110 on;
// below, where l and then m fall under bf16's smallest number, 2^-133, they are off by up to 2^-134 (1e-6 of an operand at
// 2^-115, 4e-5 at 2^-120).  A product is the six of the nine partial products that reach 2^-24 of the whole, the small ones
// first, in the unit's fp32 accumulators; m l and l m, left out, are 2^-25 of a term as a rule and of either sign, and at most
// 2^-22 together.  With these two added the errors are the same within 5 % from n = 16 on and up to a quarter less below, and
// 0.6 - 1.04 of themselves for rows of equal numbers, whose errors do not average. Sums of a few wide products round less often
// than sums of many narrow ones: 2-norms of the errors against 64 bits are 0.62 - 0.86 of those with v_mfma_f32_32x32x2_f32,
// used before, for random numbers, d = 64 and 128, n = 2 ... 2048 (n = 1: 0.64 - 1.03; no decay, n = 2048: 3.7e-7 against
// 4.4e-7), and 0.09 - 1.0 for rows of equal numbers.  Products of single features go either way (n = 1: dv 6.9e-8 against
// 3.3e-8, dq 1.0e-7 against 1.6e-7).  All finite numbers are taken; an infinite one, or a sum that overflows, makes NaN of what
// it takes part in, where the fp32 instruction could leave an infinity.  Neither reaches a token that does not see it through a
// score, but a row of Z that is not finite meets the masked scores, zeros, of its block in a product.
//
// The state tiles feed the state-term product straight from registers (see the order of features below), each split anew for
// every block.  The LDS holds the X and Y rows of a block, split, and the masked 32 x 32 score tile, split, of which each of the
// four waves computes one 16 x 16 quadrant (v_mfma_f32_16x16x32_bf16); a wave's 32 columns of Z, which no other wave
// needs, come from memory in operand order.  The scaled Y^T of the state update is not made: its operands are read from the Y
// rows with the transposing LDS read, and the decay goes to Z instead.  Blocks are 32 tokens.
//
// What bounds it: a wave and block take 132 matrix instructions (3840 cycles of its SIMD's matrix unit) and some 870 others on
// the vector unit, two thirds of them for splitting; one of those costs about 4 cycles of issue and a matrix instruction 11, so
// that a block cannot take less than 4900 cycles.  At n = 16384, with two workgroups per CU, it takes a CU 8200 in the forward
// sweep and 7000 in the backward, the matrix units busy 47 and 55 % of the time (75 and 81 % of 13 700 and 12 600 with
// v_mfma_f32_32x32x2_f32, 10 240 cycles of matrix unit per block).  The splitting stands between the matrix instructions, one
// by one: 9200 with each operand split in one go. Against v_mfma_f32_32x32x2_f32, forward + backward: b*h = 24, n = 2048: 172 -
// 182 us against 227 - 231; n = 16384: 1034 - 1072 against 1365.
#include "lasp_common.h"

namespace lasp {
namespace {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;

constexpr int F = 128;
constexpr int BLK = 32;
constexpr int NTHR = 256;
constexpr int ROW = 2 * F;           // bytes per row of one part of a tile (128 bf16)
constexpr int PART = BLK * ROW;      // h, m and l of a tile lie PART bytes apart
constexpr int TILE = 3 * PART;
constexpr int SC_ROW = 2 * BLK;      // the score tile: a row per token of X, 32 tokens of Y
constexpr int SC_PART = BLK * SC_ROW;
constexpr int OFF_X = 0, OFF_Y = TILE, OFF_SC = 2 * TILE;
constexpr int OFF_W = OFF_SC + 3 * SC_PART;  // the decay between each token of a block and the state that the block leaves
constexpr int OFF_Z = OFF_W + BLK * 4;        // each wave's columns of Z, parked
constexpr int APPLY_LDS = OFF_Z + BLK * F * 4;  // 71 808 B: two workgroups per CU
constexpr float LOG2E = 1.4426950408889634f;

__device__ __forceinline__ float decay(float s_log2e, float x) {
  return __builtin_amdgcn_exp2f(-s_log2e * x);
}
// of arguments that are the same for every lane, in a scalar register
__device__ __forceinline__ float uniform_decay(float s_log2e, float x) {
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(decay(s_log2e, x))));
}
__device__ __forceinline__ u32x4 lds16(const char *p) { return *reinterpret_cast<const u32x4 *>(p); }

// Eight numbers as three bf16 parts each
struct Split {
  u32x4 h, m, l;
};
__device__ __forceinline__ uint32_t pack(float lo, float hi) {
  float2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ float high_half(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }
// h is cut off, not rounded, which would turn the largest finite numbers into infinities
__device__ __forceinline__ void split2(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l) {
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b);
  h = __builtin_amdgcn_perm(y, x, 0x07060302);  // their upper halves
  a -= high_half(x);
  b -= high_half(y);
  m = pack(a, b);
  a -= __uint_as_float(m << 16);
  b -= high_half(m);
  l = pack(a, b);
}
// numbers 2 i and 2 i + 1 of eight, here and not where they are used
__device__ __forceinline__ void split_pair(Split &s, int i, float a, float b) {
  uint32_t h, m, l;
  split2(a, b, h, m, l);
  asm volatile("" : "+v"(h), "+v"(m), "+v"(l));
  s.h[i] = h;
  s.m[i] = m;
  s.l[i] = l;
}
__device__ __forceinline__ floatx16 mfma(u32x4 a, u32x4 b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 mfma(u32x4 a, u32x4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// c + a b.  A product of 32 x 32 x 16 keeps the matrix unit busy for 32 cycles, in which the wave that issued it can issue eight
// instructions to the vector unit; the scheduler would have all six products wait for all of the next operand's splitting and
// the splitting for the products.  work(i) goes behind product i and stays there.
template <class C, class Work>
__device__ __forceinline__ C product(const Split &a, const Split &b, C c, Work &&work) {
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const u32x4 x = i == 0 ? a.l : i == 2 || i == 3 ? a.m : a.h, y = i == 1 ? b.l : i == 2 || i == 4 ? b.m : b.h;
    c = mfma(x, y, c);
    work(i);
    __builtin_amdgcn_sched_barrier(0);
  }
  return c;
}

// Rows of the X and Y tiles.  A 16-byte unit holds eight features: of each group of 16, unit 0 has features 0-3 and 8-11, unit 1
// features 4-7 and 12-15, which is the order in which lane half hh = 0, 1 of an accumulator tile holds rows (8 g + 4 hh + r in
// register 4 g + r), so that an accumulator tile is multiplied against rows without a shuffle.  Unit u of row r lies at unit
// u ^ swizzle(r): eight consecutive rows read at one unit, and the four rows x 64 bytes that half a wave reads transposed,
// fall on disjoint banks.
__device__ __forceinline__ int swizzle(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
// 16 bytes at `off` of a tile's three parts
__device__ __forceinline__ Split parts(const char *tile, int off, int part) {
  return {lds16(tile + off), lds16(tile + off + part), lds16(tile + off + 2 * part)};
}
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 *lds_v4i16;
// The transposing 8-byte read works in groups of 16 lanes: lane i of a group receives, as element j, element (i % 4) of what
// lane (4 j + i / 4) of the group addressed.  With lane s addressing token T + s / 4, features f + 4 (s % 4) .. + 3, lane i ends
// up with feature f + i of tokens T .. T + 3; two such reads are eight tokens.
__device__ __forceinline__ u32x4 transposed(const char *lo, const char *hi) {
  const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(lo)));
  const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16)(hi)));
  return {a.x, a.y, b.x, b.y};
}
// Operand of lane (c, hh) over tokens: features 32 T + c of tokens 16 u + 8 hh .. + 7 of a tile
struct TokenReader {
  int lo, hi;  // the lane's offsets in the first 32 features and 16 tokens
  __device__ __forceinline__ explicit TokenReader(int lane) {
    const int s = lane & 15, ch = (lane >> 4) & 1, hh = lane >> 5, p = s & 3;
    const int row = 8 * hh + (s >> 2), unit = 2 * ch + (p & 1);
    lo = row * ROW + ((unit ^ swizzle(row)) << 4) + ((p >> 1) << 3);
    hi = (row + 4) * ROW + ((unit ^ swizzle(row + 4)) << 4) + ((p >> 1) << 3);
  }
  __device__ __forceinline__ Split read(const char *tile, int T, int u) const {
    const char *a = tile + (lo ^ (T << 6)) + 16 * u * ROW, *b = tile + (hi ^ (T << 6)) + 16 * u * ROW;
    return {transposed(a, b), transposed(a + PART, b + PART), transposed(a + 2 * PART, b + 2 * PART)};
  }
};

// Nothing is moved across this line: the reads above it are in flight while the products below run.  (The scheduler by itself
// reads an operand right before the product that needs it.)
__device__ __forceinline__ void reads_first() { __builtin_amdgcn_sched_barrier(0); }

// A block of token rows as a buffer that ends with them: rows that a partial block does not have read as zeros and are not
// stored, without a branch per access (after which a wait for the oldest access would have to wait for all of them).
typedef __amdgpu_buffer_rsrc_t rows_t;
__device__ __forceinline__ rows_t buffer_of(const float *p, int bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);  // the same for every lane
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0, bytes, 0x00020000);
}
__device__ __forceinline__ rows_t rows_of(const float *p, int count, int width) { return buffer_of(p, count * width * 4); }
constexpr int NOWHERE = 1 << 30;  // an offset past the end of every such buffer: features that a narrow row does not have
__device__ __forceinline__ f32x4 load16(rows_t rows, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, off, 0, 0));
}

struct SegWork {
  int bh, seg;
  int64_t tok0;
  int nblk;  // 32-token blocks, the last one possibly partial
  int tail;  // tokens in the last block (1..32); below 32 only at the end of a ragged chunk
};
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

// An offset that is worked out here, and not once for all blocks: the offsets of narrow rows are no constants, and registers are short
template <bool NARROW>
__device__ __forceinline__ int fresh(int off) {
  if (NARROW) asm volatile("" : "+v"(off));
  return off;
}
// The X (or Y) rows of a block: thread (cq, rq) holds features 4 cq .. + 3 of rows rq + 8 it
struct Loader {
  int from, to, step;  // the thread's place in a block of rows and in a tile; eight rows on
  __device__ __forceinline__ Loader(int tid, int width) {
    const int cq = tid & 31, rq = tid >> 5, p = cq & 3;
    from = width == F || 4 * cq < width ? rq * (width * 4) + cq * 16 : NOWHERE;
    step = 8 * width * 4;
    to = rq * ROW + (((2 * (cq >> 2) + (p & 1)) ^ swizzle(rq)) << 4) + ((p >> 1) << 3);
  }
  template <bool NARROW>
  __device__ __forceinline__ void load(rows_t rows, f32x4 (&n)[4]) const {
    const int at = fresh<NARROW>(from);
#pragma unroll
    for (int it = 0; it < 4; ++it) n[it] = load16(rows, at + it * step);
  }
  // half `k & 1` of row k >> 1, into `row`; the second half writes the row
  __device__ __forceinline__ void fill_half(char *tile, const f32x4 (&n)[4], int k, u32x2 (&row)[3]) const {
    const int it = k >> 1, half = k & 1;
    uint32_t h, m, l;
    if (half == 0)
      split2(n[it].x, n[it].y, h, m, l);
    else
      split2(n[it].z, n[it].w, h, m, l);
    row[0][half] = h;
    row[1][half] = m;
    row[2][half] = l;
    if (half == 0) return;
    char *at = tile + (to ^ ((it & 1) << 5)) + it * (8 * ROW);  // (eight rows on, bit 1 of the swizzle flips)
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x2 *>(at + i * PART) = row[i];
  }
  __device__ __forceinline__ void fill(char *tile, const f32x4 (&n)[4]) const {
    u32x2 row[3];
#pragma unroll
    for (int k = 0; k < 8; ++k) fill_half(tile, n, k, row);
  }
};
// A wave's own 32 columns of Z come straight from memory: lane (c, hh) holds tokens 16 u + 8 hh + j of column c in z[8 u + j]
__device__ __forceinline__ int column_off(int lane, int w, int width) {
  const int col = 32 * w + (lane & 31);
  return width == F || col < width ? 8 * (lane >> 5) * (width * 4) + col * 4 : NOWHERE;
}
template <bool NARROW>
__device__ __forceinline__ void load_columns(rows_t rows, int lane_off, int width, float (&z)[16]) {
  const int at = fresh<NARROW>(lane_off);
#pragma unroll
  for (int i = 0; i < 16; ++i)
    z[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rows, at + (16 * (i >> 3) + (i & 7)) * (width * 4), 0, 0));
}

enum Mode {
  M_ALIGNED,  // n is a multiple of 32, rows of 128 features
  M_RAGGED,   // any n
  // any n and rows of any multiples of 4 features, d and e, that 2, 3 or 4 tiles of 32 features hold
  M_NARROW2,
  M_NARROW3,
  M_NARROW4,
};
constexpr bool narrow(int mode) { return mode >= M_NARROW2; }
constexpr int tiles(int mode) { return narrow(mode) ? mode - M_NARROW2 + 2 : 4; }  // of 32 features
// Narrow rows end after g.d (g.e) features: what is missing reads as zeros and is not stored, and stored states are d x e.  With two or
// three tiles the state has as many rows, and the waves whose columns of Z are all missing only help with rows and scores.
// Against rows padded to 128 features before the call (five tensors copied in, four copied out, and products of zeros), forward +
// backward: b*h = 24, n = 2048: d = e = 64 348 -> 105 us, 80 359 -> 121, 96 371 -> 133, d = 128, e = 64 282 -> 146; n = 8192, d = e =
// 64: 1035 -> 303.  Bound as above; with two tiles the matrix units of two SIMDs idle in the state's products.  The kernels are
// instances per number of tiles because a number known only at run time cost up to 110 spilled registers.
//
// RAGGED: the chunk length is not a multiple of 32, so the last block of the last segment is
// partial (missing rows read as zeros, stores masked, and -- going backwards, where that block
// comes first -- the entering state sits `len` tokens ahead instead of 32).
template <bool REV, bool TRANS, int MODE>
__device__ __forceinline__ void
sweep_body(const float *__restrict__ X, const float *__restrict__ Y, const float *__restrict__ Z,
           const float *__restrict__ S, const float *__restrict__ states, float *__restrict__ Out,
           const Geom &g, int item, char *smem) {
  constexpr bool RAGGED = MODE != M_ALIGNED, NARROW = narrow(MODE);
  constexpr int NT = tiles(MODE);
  const int tid = fresh<NARROW>(threadIdx.x);  // (nothing of it is kept for another role's sweep)
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index, uniform: keeps it in an SGPR
  const int c = lane & 31, hh = lane >> 5;

  // features of X and Y, and of Z and Out
  const int xw = !NARROW ? F : TRANS ? g.e : g.d, zw = !NARROW ? F : TRANS ? g.d : g.e;
  const bool active = NT == 4 || w < NT;

  const SegWork sw = seg_work(g, item);
  const int64_t row0 = (int64_t)sw.bh * g.n + sw.tok0;
  const Loader loader(tid, xw);
  const TokenReader tokens(lane);
  const int z_off = column_off(lane, w, zw);

  f32x4 nx[4], ny[4];
  float z[16];
  auto len_of = [&](int blk) __attribute__((always_inline)) { return RAGGED && blk == sw.nblk - 1 ? sw.tail : BLK; };
  auto rows = [&](const float *p, int blk, int width) __attribute__((always_inline)) {
    return rows_of(p + (row0 + (int64_t)blk * BLK) * width, len_of(blk), width);
  };
  const int first = REV ? sw.nblk - 1 : 0;
  const int step = REV ? -1 : 1;
  loader.load<NARROW>(rows(X, first, xw), nx);
  loader.load<NARROW>(rows(Y, first, xw), ny);
  load_columns<NARROW>(rows(Z, first, zw), z_off, zw, z);

  const float sl = S[sw.bh - quotient(sw.bh, g.by_h) * g.h] * LOG2E;
  // ---- constants (all exponents <= 0)
  const float blockdec = uniform_decay(sl, (float)BLK);
  const float qdec = decay(sl, REV ? (float)(BLK - c) : (float)c);
  if (tid < BLK) *reinterpret_cast<float *>(smem + OFF_W + 4 * tid) = decay(sl, REV ? (float)tid : (float)(BLK - tid));
  // this wave's quadrant of the score tile: tokens b = 16 qb .. of Y, a = 16 qa .. of X
  const int qb = w >> 1, qa = w & 1;
  const int q_lane = lane & 15, q_grp = lane >> 4;
  // the lane's operands: a token of quadrant row q of X or Y, and token lane % 32 of X
  auto quadrant_at = [](int lane, int q) {
    const int token = 16 * q + (lane & 15);
    return token * ROW + (((lane >> 4) ^ swizzle(token)) << 4);
  };
  auto row_at = [](int lane) { return (lane & 31) * ROW + (((lane >> 5) ^ swizzle(lane & 31)) << 4); };
  const int xq = quadrant_at(lane, qa), yq = quadrant_at(lane, qb);
  // decay between the tokens of a score; -1: masked.  Such a score is left out and not multiplied by zero, which would take an
  // infinity or a NaN (or what overflowed on the way to this score only) to tokens that do not see it.
  float qmask[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int dist = (16 * qa + q_lane - 16 * qb - 4 * q_grp - r) * (REV ? -1 : 1);
    qmask[r] = dist >= 0 ? decay(sl, (float)dist) : -1.f;
  }
  // (selected before the product, which the compiler fuses with the first subtraction of the split: its rounding is not felt)
  auto masked = [&](float score, int r) __attribute__((always_inline)) { return (qmask[r] < 0.f ? 0.f : score) * qmask[r]; };
  // rows of 64 bytes; unit u of row a lies at u ^ ((a >> 2) & 3)
  auto quadrant_scores_at = [&](int lane) __attribute__((always_inline)) {
    const int q_lane = lane & 15, q_grp = lane >> 4;
    return (16 * qa + q_lane) * SC_ROW + (((2 * qb + (q_grp >> 1)) ^ ((q_lane >> 2) & 3)) << 4) + ((q_grp & 1) << 3);
  };
  const int sc_at = quadrant_scores_at(lane);
  auto scores_at = [](int lane) { return (lane & 31) * SC_ROW + (((lane >> 5) ^ ((lane >> 2) & 3)) << 4); };  // token lane % 32's
  const int sc_from = scores_at(lane);
  char *const z_park = smem + OFF_Z + w * 4096 + lane * 16;
  const int x_from = row_at(lane);

  // ---- state entering the segment: st[T][4g+r] = St[32T+8g+4hh+r][32w+c]
  floatx16 st[NT];
  if (NARROW && states) {
    // (rows come in fours: a row that is missing is in a group of four that is)
    const rows_t sp = buffer_of(states + ((int64_t)sw.bh * g.n_seg + sw.seg) * (g.d * g.e), g.d * g.e * 4);
    const int col = 32 * w + c;
    const int at = col < zw ? (TRANS ? col * xw : col) * 4 : NOWHERE;
#pragma unroll
    for (int T = 0; T < NT; ++T) {
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int row = 32 * T + 8 * gq + 4 * hh;
        const int off = row < xw ? at + (TRANS ? row : row * zw) * 4 : NOWHERE;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          st[T][4 * gq + r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sp, off + (TRANS ? r : r * zw) * 4, 0, 0));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  } else if (states) {
    const float *sp = states + ((int64_t)sw.bh * g.n_seg + sw.seg) * (F * F);
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * T + 8 * (r >> 2) + 4 * hh + (r & 3);
        const int col = 32 * w + c;
        st[T][r] = TRANS ? sp[col * F + row] : sp[row * F + col];
      }
  } else {
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r) st[T][r] = 0.f;
  }
  loader.fill(smem + OFF_X, nx);
  loader.fill(smem + OFF_Y, ny);
  __syncthreads();

  // output: lane (c, hh) holds, for token c, four consecutive columns per g
  auto store = [&](const floatx16 &acc, int blk, int lane) __attribute__((always_inline)) {
    const int c = lane & 31, col0 = fresh<NARROW>(32 * w + 4 * (lane >> 5));
    const rows_t out = rows_of(Out + (row0 + (int64_t)blk * BLK) * zw, len_of(blk), zw);
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      f32x4 o;
      o.x = acc[4 * gq + 0];
      o.y = acc[4 * gq + 1];
      o.z = acc[4 * gq + 2];
      o.w = acc[4 * gq + 3];
      const int col = col0 + 8 * gq, off = !NARROW || col < zw ? c * (zw * 4) + col * 4 : NOWHERE;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), out, off, 0, 0);
    }
  };

  int blk = first;
#pragma unroll 1
  for (int it = 0; it < sw.nblk - 1; ++it, blk += step) {
    const int len = len_of(blk);
    float qd = qdec, bd = blockdec;
    if (RAGGED && REV && len != BLK) {
      qd = decay(sl, (float)max(len - c, 0));
      bd = uniform_decay(sl, (float)len);
    }

    // Z as the state update takes it, between the products of the scores
    Split zs[2];
    f32x4 wz[4];  // (kept in LDS: registers are short here)
#pragma unroll
    for (int i = 0; i < 4; ++i) wz[i] = *reinterpret_cast<const f32x4 *>(smem + OFF_W + (16 * (i >> 1) + 8 * hh + 4 * (i & 1)) * 4);
    auto scale_z = [&](int i) __attribute__((always_inline)) {  // pair i of 8
      const f32x4 &v = wz[i >> 1];
      const float w0 = (i & 1) ? v.z : v.x, w1 = (i & 1) ? v.w : v.y;
      split_pair(zs[i >> 2], i & 3, z[2 * i] * w0, z[2 * i + 1] * w1);
    };
    // (1) scores of the quadrant, masked: sc[r] = y_b . x_a, b = 16 qb + 4 q_grp + r, a = 16 qa + q_lane
    Split xf[2], yf[2];
    {
      floatx4 sc = {0.f, 0.f, 0.f, 0.f};
      Split ys[2], xs[2];
      xs[0] = parts(smem + OFF_X, xq, PART);
      ys[0] = parts(smem + OFF_Y, yq, PART);
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        if (m < NT - 1) {
          xs[(m + 1) & 1] = parts(smem + OFF_X, xq ^ ((m + 1) << 6), PART);
          ys[(m + 1) & 1] = parts(smem + OFF_Y, yq ^ ((m + 1) << 6), PART);
        } else {
#pragma unroll
          for (int u = 0; u < 2; ++u) xf[u] = parts(smem + OFF_X, x_from ^ (u << 5), PART);
        }
        reads_first();
        sc = product(ys[m & 1], xs[m & 1], sc, [&](int i) __attribute__((always_inline)) {
          constexpr int PER = (8 + NT - 1) / NT;  // pairs of Z for each of the NT products
          const int pair = m * PER + i / (6 / PER);
          if (i % (6 / PER) == 0 && i / (6 / PER) < PER && pair < 8) scale_z(pair);
        });
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) yf[u] = tokens.read(smem + OFF_Y, 0, u);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4 *>(z_park + 1024 * i) = f32x4{z[4 * i], z[4 * i + 1], z[4 * i + 2], z[4 * i + 3]};
      reads_first();
      u32x2 h, m, l;
      uint32_t a, b, d;
      split2(masked(sc[0], 0), masked(sc[1], 1), a, b, d);
      h.x = a, m.x = b, l.x = d;
      split2(masked(sc[2], 2), masked(sc[3], 3), a, b, d);
      h.y = a, m.y = b, l.y = d;
      char *at = smem + OFF_SC + sc_at;
      *reinterpret_cast<u32x2 *>(at) = h;
      *reinterpret_cast<u32x2 *>(at + SC_PART) = m;
      *reinterpret_cast<u32x2 *>(at + 2 * SC_PART) = l;
    }
    // (2) state term, acc[4g+r] = sum_f St[f][32w+8g+4hh+r] x_a[f] (a = c), and (3) the state update, 32 features at a time
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    loader.load<NARROW>(rows(X, blk + step, xw), nx);
    Split a0, a1, zu[2];
    f32x4 zp[4];
    if (active) {
#pragma unroll
      for (int i = 0; i < 4; ++i) split_pair(a0, i, st[0][2 * i], st[0][2 * i + 1]);
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        acc = product(a0, xf[0], acc, [&](int i) __attribute__((always_inline)) {
          if (i < 4) split_pair(a1, i, st[T][8 + 2 * i], st[T][9 + 2 * i]);
        });
        acc = product(a1, xf[1], acc, [&](int i) __attribute__((always_inline)) {
#pragma unroll
          for (int r = 3 * i; r < 3 * i + 3 && r < 16; ++r) st[T][r] *= bd;
        });
        if (T < NT - 1) {
#pragma unroll
          for (int u = 0; u < 2; ++u) xf[u] = parts(smem + OFF_X, x_from ^ ((2 * T + 2 + u) << 5), PART);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) zp[i] = *reinterpret_cast<const f32x4 *>(z_park + 1024 * i);
        }
        reads_first();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          st[T] = product(yf[u], zs[u], st[T], [&](int i) __attribute__((always_inline)) {
            if (T < NT - 1) {
              if (u == 0 && i < 4) split_pair(a0, i, st[T + 1][2 * i], st[T + 1][2 * i + 1]);
            } else if (i < 4) {
              const f32x4 &v = zp[2 * u + (i >> 1)];
              split_pair(zu[u], i, (i & 1) ? v.z : v.x, (i & 1) ? v.w : v.y);
            }
          });
          if (T < NT - 1) yf[u] = tokens.read(smem + OFF_Y, T + 1, u);
          reads_first();
        }
        if (T == (NT == 3 ? 2 : 1)) loader.load<NARROW>(rows(Y, blk + step, xw), ny);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] *= qd;
    } else {
      loader.load<NARROW>(rows(Y, blk + step, xw), ny);
    }
    __syncthreads();  // the score tile is complete; X and Y are no longer read
    // (4) intra-block term
    load_columns<NARROW>(rows(Z, blk + step, zw), z_off, zw, z);
    if (active) {
      Split sf[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) sf[u] = parts(smem + OFF_SC, sc_from ^ (u << 5), SC_PART);
      reads_first();
      u32x2 row[3];
#pragma unroll
      for (int u = 0; u < 2; ++u)
        acc = product(zu[u], sf[u], acc, [&](int i) __attribute__((always_inline)) {  // and the next block's X
          if (6 * u + i < 8) loader.fill_half(smem + OFF_X, nx, 6 * u + i, row);
        });
    } else {
      loader.fill(smem + OFF_X, nx);
    }
    loader.fill(smem + OFF_Y, ny);
    store(acc, blk, lane);  // (5)
    __syncthreads();  // the next block's X and Y are complete; the score tile is no longer read
  }
  // The segment's last block leaves no state behind: its update, 48 of 132 products, and what is split and scaled for it are left out.
  // Forward + backward in us, with that update and without, the same bits: b*h = 24, n = 2048 (four blocks to a segment) 183.7 and 174.8,
  // n = 16384 (16 blocks) 1061 and 1045; b*h = 16, n = 1024 (two) 85.6 and 79.9.
  {
    float qd = qdec;
    if (RAGGED && REV && len_of(blk) != BLK) qd = decay(sl, (float)max(len_of(blk) - c, 0));
    Split xf[2][2], zu[2];
    // (the lane's offsets are worked out here: kept through the blocks before, they would go to scratch)
    const int late = fresh<true>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    const int x_at = row_at(late);
    {
      floatx4 sc = {0.f, 0.f, 0.f, 0.f};
      Split ys[2], xs[2];
      const int xl = quadrant_at(late, qa), yl = quadrant_at(late, qb);
      xs[0] = parts(smem + OFF_X, xl, PART);
      ys[0] = parts(smem + OFF_Y, yl, PART);
#pragma unroll
      for (int m = 0; m < NT; ++m) {
        if (m < NT - 1) {
          xs[(m + 1) & 1] = parts(smem + OFF_X, xl ^ ((m + 1) << 6), PART);
          ys[(m + 1) & 1] = parts(smem + OFF_Y, yl ^ ((m + 1) << 6), PART);
        } else {
#pragma unroll
          for (int u = 0; u < 2; ++u) xf[0][u] = parts(smem + OFF_X, x_at ^ (u << 5), PART);
        }
        reads_first();
        sc = product(ys[m & 1], xs[m & 1], sc, [](int) {});
      }
      u32x2 h, m, l;
      uint32_t a, b, d;
      split2(masked(sc[0], 0), masked(sc[1], 1), a, b, d);
      h.x = a, m.x = b, l.x = d;
      split2(masked(sc[2], 2), masked(sc[3], 3), a, b, d);
      h.y = a, m.y = b, l.y = d;
      char *at = smem + OFF_SC + quadrant_scores_at(late);
      *reinterpret_cast<u32x2 *>(at) = h;
      *reinterpret_cast<u32x2 *>(at + SC_PART) = m;
      *reinterpret_cast<u32x2 *>(at + 2 * SC_PART) = l;
    }
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (active) {
      Split a0, a1;
#pragma unroll
      for (int i = 0; i < 4; ++i) split_pair(a0, i, st[0][2 * i], st[0][2 * i + 1]);
#pragma unroll
      for (int T = 0; T < NT; ++T) {
        if (T < NT - 1)
#pragma unroll
          for (int u = 0; u < 2; ++u) xf[(T + 1) & 1][u] = parts(smem + OFF_X, x_at ^ ((2 * T + 2 + u) << 5), PART);
        reads_first();
        auto split_z = [&](int k) __attribute__((always_inline)) {
          if (k < 8) split_pair(zu[k >> 2], k & 3, z[2 * k], z[2 * k + 1]);
        };
        constexpr int PER = 8 / NT + (8 % NT > 0);  // pairs of Z beside each of the NT pairs of products
        acc = product(a0, xf[T & 1][0], acc, [&](int i) __attribute__((always_inline)) {
          if (i < 4) split_pair(a1, i, st[T][8 + 2 * i], st[T][9 + 2 * i]);
          if (i >= 4 && i - 4 < PER) split_z(T * PER + i - 4);
        });
        acc = product(a1, xf[T & 1][1], acc, [&](int i) __attribute__((always_inline)) {
          if (T < NT - 1 && i < 4) split_pair(a0, i, st[T < NT - 1 ? T + 1 : T][2 * i], st[T < NT - 1 ? T + 1 : T][2 * i + 1]);
          if (i >= 4 && i - 2 < PER) split_z(T * PER + i - 2);
        });
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] *= qd;
    }
    __syncthreads();  // the score tile is complete
    if (active) {
      Split sf[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) sf[u] = parts(smem + OFF_SC, scores_at(late) ^ (u << 5), SC_PART);
      reads_first();
#pragma unroll
      for (int u = 0; u < 2; ++u) acc = product(zu[u], sf[u], acc, [](int) {});
    }
    store(acc, blk, late);
  }
}

template <bool REV, bool TRANS, int MODE>
__global__ void __launch_bounds__(NTHR, 2)
la32_apply(const float *__restrict__ X, const float *__restrict__ Y, const float *__restrict__ Z,
           const float *__restrict__ S, const float *__restrict__ states, float *__restrict__ Out, Geom g) {
  extern __shared__ __align__(16) char smem[];
  sweep_body<REV, TRANS, MODE>(X, Y, Z, S, states, Out, g, (int)blockIdx.x, smem);
}

// dQ, dV and dK in one launch; the three workgroups of a (b*h, segment) sit 8 block indices
// apart, i.e. on the same XCD
template <int MODE>
__global__ void __launch_bounds__(NTHR, 2)
la32_bwd3(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V,
          const float *__restrict__ DO, const float *__restrict__ S, const float *__restrict__ kv_states,
          const float *__restrict__ dkv_states, float *__restrict__ DQ, float *__restrict__ DK,
          float *__restrict__ DV, Geom g) {
  extern __shared__ __align__(16) char smem[];
  const int n_items = g.b * g.h * g.n_seg;
  const int grp = blockIdx.x / 24, r = blockIdx.x - grp * 24;
  const int role = r >> 3;
  const int item = n_items - 1 - (grp * 8 + (r & 7));
  if (item < 0) return;
  if (role == 0)
    sweep_body<false, true, MODE>(DO, V, K, S, kv_states, DQ, g, item, smem);
  else if (role == 1)
    sweep_body<true, false, MODE>(K, Q, DO, S, dkv_states, DV, g, item, smem);
  else
    sweep_body<true, true, MODE>(V, DO, Q, S, dkv_states, DK, g, item, smem);
}

// a segment's own state: causal sum_b l^(L-b) y_b^T z_b ; anti-causal sum_b l^b y_b^T z_b
template <bool REV, int MODE>
__global__ void __launch_bounds__(NTHR, 2)
la32_seg_state(const float *__restrict__ Y, const float *__restrict__ Z, const float *__restrict__ S,
               float *__restrict__ states, Geom g, int skip_seg) {
  constexpr bool RAGGED = MODE != M_ALIGNED, NARROW = narrow(MODE);
  constexpr int NT = tiles(MODE);
  __shared__ __align__(256) char smem[2][TILE];  // double-buffered Y
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index, uniform: keeps it in an SGPR
  const int c = lane & 31, hh = lane >> 5;

  const SegWork sw = seg_work(g, (int)blockIdx.x);
  if (sw.seg == skip_seg) return;
  const int64_t row0 = (int64_t)sw.bh * g.n + sw.tok0;
  const int yw = NARROW ? g.d : F, zw = NARROW ? g.e : F;
  const bool active = NT == 4 || w < NT;
  const Loader loader(tid, yw);
  const TokenReader tokens(lane);
  const int z_off = column_off(lane, w, zw);
  auto len_of = [&](int blk) __attribute__((always_inline)) { return RAGGED && blk == sw.nblk - 1 ? sw.tail : BLK; };
  auto rows = [&](const float *p, int blk, int width) __attribute__((always_inline)) {
    return rows_of(p + (row0 + (int64_t)blk * BLK) * width, len_of(blk), width);
  };
  f32x4 ny[4];
  float z[16];
  const int first = REV ? sw.nblk - 1 : 0;
  const int step = REV ? -1 : 1;
  loader.load<NARROW>(rows(Y, first, yw), ny);
  load_columns<NARROW>(rows(Z, first, zw), z_off, zw, z);

  const float sl = S[sw.bh - quotient(sw.bh, g.by_h) * g.h] * LOG2E;
  const float blockdec = uniform_decay(sl, (float)BLK);
  float zdec[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int b = 16 * (i >> 3) + 8 * hh + (i & 7);
    zdec[i] = decay(sl, REV ? (float)b : (float)(BLK - b));
  }
  floatx16 st[NT];
#pragma unroll
  for (int T = 0; T < NT; ++T)
#pragma unroll
    for (int r = 0; r < 16; ++r) st[T][r] = 0.f;
  loader.fill(smem[0], ny);
  __syncthreads();
  for (int it = 0, blk = first; it < sw.nblk; ++it, blk += step) {
    const bool more = it + 1 < sw.nblk;
    if (more) loader.load<NARROW>(rows(Y, blk + step, yw), ny);
    const int len = len_of(blk);
    const float bd = RAGGED && len != BLK ? uniform_decay(sl, (float)len) : blockdec;
    if (RAGGED && !REV && len != BLK)  // going forwards a partial block is the last one: its tokens sit `len - b` before the segment's end
#pragma unroll
      for (int i = 0; i < 16; ++i) zdec[i] = decay(sl, (float)max(len - 16 * (i >> 3) - 8 * hh - (i & 7), 0));
    const char *tile = smem[it & 1];
    Split yf[2][2], zs[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) yf[0][u] = tokens.read(tile, 0, u);
#pragma unroll
    for (int i = 0; i < 8; ++i) split_pair(zs[i >> 2], i & 3, z[2 * i] * zdec[2 * i], z[2 * i + 1] * zdec[2 * i + 1]);
    if (more) load_columns<NARROW>(rows(Z, blk + step, zw), z_off, zw, z);
#pragma unroll
    for (int r = 0; r < 16; ++r) st[0][r] *= bd;
#pragma unroll
    for (int T = 0; T < NT; ++T) {
      if (!active) break;
      if (T < NT - 1)
#pragma unroll
        for (int u = 0; u < 2; ++u) yf[(T + 1) & 1][u] = tokens.read(tile, T + 1, u);
      reads_first();
#pragma unroll
      for (int u = 0; u < 2; ++u)
        st[T] = product(yf[T & 1][u], zs[u], st[T], [&](int i) __attribute__((always_inline)) {
          if (T < NT - 1 && u == 0)
#pragma unroll
            for (int r = 3 * i; r < 3 * i + 3 && r < 16; ++r) st[T + 1][r] *= bd;
        });
    }
    if (more) loader.fill(smem[(it + 1) & 1], ny);
    __syncthreads();
  }
  if (NARROW) {
    const rows_t sp = buffer_of(states + ((int64_t)sw.bh * g.n_seg + sw.seg) * (yw * zw), yw * zw * 4);
#pragma unroll
    for (int T = 0; T < NT; ++T)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 32 * T + 8 * (r >> 2) + 4 * hh + (r & 3), col = 32 * w + c;
        const int off = row < yw && col < zw ? (row * zw + col) * 4 : NOWHERE;
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, (float)st[T][r]), sp, off, 0, 0);
      }
    return;
  }
  float *sp = states + ((int64_t)sw.bh * g.n_seg + sw.seg) * (F * F);
#pragma unroll
  for (int T = 0; T < NT; ++T)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      sp[(32 * T + 8 * (r >> 2) + 4 * hh + (r & 3)) * F + 32 * w + c] = st[T][r];
}

template <bool REV, int MODE>
int launch_state(const void *y, const void *z, const float *s, float *states, const Geom &g,
                 bool carry_wanted, hipStream_t st) {
  const unsigned grid = (unsigned)((int64_t)g.b * g.h * g.n_seg);
  const int skip_seg = carry_wanted ? -1 : (REV ? 0 : g.n_seg - 1);
  ProfScope prof(KC_STATE, st);
  la32_seg_state<REV, MODE><<<grid, NTHR, 0, st>>>((const float *)y, (const float *)z, s, states, g,
                                                     skip_seg);
  return (int)hipGetLastError();
}

template <int MODE>
int fwd_r(const FwdArgs &a, const Geom &g, hipStream_t st) {
  int rc;
  const bool need_states = g.n_seg > 1 || a.kv_in || a.kv_out;
  if (need_states) {
    if ((rc = launch_state<false, MODE>(a.k, a.v, a.s, a.seg_states, g, a.kv_out != nullptr, st))) return rc;
    if ((rc = launch_segment_scan(a.seg_states, a.kv_in, a.kv_out, a.s, g, 0, st))) return rc;
  }
  if ((rc = grant_lds<la32_apply<false, false, MODE>>(APPLY_LDS))) return rc;
  const unsigned grid = (unsigned)((int64_t)g.b * g.h * g.n_seg);
  ProfScope prof(KC_APPLY, st);
  la32_apply<false, false, MODE><<<grid, NTHR, APPLY_LDS, st>>>((const float *)a.q, (const float *)a.k,
                                                                  (const float *)a.v, a.s,
                                                                  need_states ? a.seg_states : nullptr,
                                                                  (float *)a.o, g);
  return (int)hipGetLastError();
}

template <int MODE>
int bwd_r(const BwdArgs &a, const Geom &g, hipStream_t st) {
  int rc;
  const float *kv_states = a.kv_seg_states;
  if (!kv_states && (g.n_seg > 1 || a.kv_in)) {
    if ((rc = launch_state<false, MODE>(a.k, a.v, a.s, a.ws_kv, g, false, st))) return rc;
    if ((rc = launch_segment_scan(a.ws_kv, a.kv_in, nullptr, a.s, g, 0, st))) return rc;
    kv_states = a.ws_kv;
  }
  const float *dkv_states = nullptr;
  if (g.n_seg > 1 || a.dkv_in || a.dkv_out) {
    if ((rc = launch_state<true, MODE>(a.q, a.d_o, a.s, a.ws_dkv, g, a.dkv_out != nullptr, st))) return rc;
    if ((rc = launch_segment_scan(a.ws_dkv, a.dkv_in, a.dkv_out, a.s, g, 1, st))) return rc;
    dkv_states = a.ws_dkv;
  }
  if ((rc = grant_lds<la32_bwd3<MODE>>(APPLY_LDS))) return rc;
  const int64_t n_items = (int64_t)g.b * g.h * g.n_seg;
  const unsigned grid = (unsigned)(((n_items + 7) / 8) * 24);
  ProfScope prof(KC_BWD3, st);
  la32_bwd3<MODE><<<grid, NTHR, APPLY_LDS, st>>>((const float *)a.q, (const float *)a.k,
                                                   (const float *)a.v, (const float *)a.d_o, a.s, kv_states,
                                                   dkv_states, (float *)a.dq, (float *)a.dk, (float *)a.dv, g);
  return (int)hipGetLastError();
}

}  // namespace

int mfma_f32_fwd(const FwdArgs &a, const Geom &g, hipStream_t st) {
  if (g.d == F && g.e == F) return g.n % BLK != 0 ? fwd_r<M_RAGGED>(a, g, st) : fwd_r<M_ALIGNED>(a, g, st);
  const int widest = g.d > g.e ? g.d : g.e;
  return widest <= 64 ? fwd_r<M_NARROW2>(a, g, st) : widest <= 96 ? fwd_r<M_NARROW3>(a, g, st) : fwd_r<M_NARROW4>(a, g, st);
}

int mfma_f32_bwd(const BwdArgs &a, const Geom &g, hipStream_t st) {
  if (g.d == F && g.e == F) return g.n % BLK != 0 ? bwd_r<M_RAGGED>(a, g, st) : bwd_r<M_ALIGNED>(a, g, st);
  const int widest = g.d > g.e ? g.d : g.e;
  return widest <= 64 ? bwd_r<M_NARROW2>(a, g, st) : widest <= 96 ? bwd_r<M_NARROW3>(a, g, st) : bwd_r<M_NARROW4>(a, g, st);
}

}  // namespace lasp
