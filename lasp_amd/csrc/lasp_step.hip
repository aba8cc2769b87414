// A few tokens at a time (decoding): n <= LASP_STEP_TOKENS tokens for every (b, h), d <= 128, any element type.
//
//   per token:  A = St + k^T v;   o = q A;   St <- l A          (l = exp(-s); lasp/lasp_fuse.py:104-127 with one-token blocks)
//
// What bounds it: the states.  A token moves 3 d + e elements of q, k, v and o but reads and writes d x e floats, so the
// kernel is a copy of the states with a rank-one update on the way.  A workgroup holds the state of one (b, h), or a slab
// of its columns, in registers: every thread has all its 16-byte pieces in flight at once, applies the tokens to them and
// writes them back; nothing passes through LDS but q, k, v and the partial outputs.  All arithmetic is fp32.
//
// Slabs of 32 columns: small workgroups keep reads and writes of different slabs mixed on the memory bus, and give one
// sequence's 16 heads 64 workgroups.  b*h = 512, d = e = 128, one token: 11.9 us (5.7 TB/s) against 12.2 for slabs of 64 and
// 14.0 for whole rows; b*h = 16: 3.6, 4.3 and 5.9.  The sweep kernels, where such calls ran before, hold a CU with a
// 64-token block of which one row is real: 17.0 us and 6.0; in fp32 (pre-pass, scan and sweep) 54 us against 11.7.
//
// The tokens are taken one after the other, so the sweep kernels win again from about five on (b*h = 512: 4 tokens 16.0 us
// against 18.1, 8 tokens 23.4 against 18.3; b*h = 16: 5.0 against 6.2 and 6.7 against 6.2): hence LASP_STEP_TOKENS = 4.
#include "lasp_common.h"

namespace lasp {
namespace {

constexpr int NT = 256;
// states need only start on a 4-byte boundary; global 16-byte accesses ask for no more
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// A row's LC lanes span a slab of 4 LC columns; the workgroup's NT / LC groups of lanes take every (NT / LC)-th row.
// TOK: tokens the LDS arrays hold (n <= TOK).
template <class T, int LC, int TOK>
__global__ void __launch_bounds__(NT)
la_step(const T *__restrict__ Q, const T *__restrict__ K, const T *__restrict__ V, const float *__restrict__ S,
        const float *kv_in, float *kv_out, T *__restrict__ O, Geom g) {
  constexpr int RG = NT / LC, R = kMaxWidth / RG;  // groups of rows; rows per thread
  __shared__ float sq[TOK][kMaxWidth], sk[TOK][kMaxWidth];
  __shared__ __align__(16) float sv[TOK][kMaxWidth];
  __shared__ __align__(16) float red[TOK][NT / 64][4 * LC];
  const int tid = threadIdx.x, bh = blockIdx.x, n = (int)g.n, d = g.d, e = g.e;
  const int col0 = blockIdx.y * 4 * LC, col = col0 + 4 * (tid % LC), rg = tid / LC;
  const bool col_ok = col < e;  // e is a multiple of 4

  // q, k and v first, then the state: the counter that a wait reads runs in issue order
  const int f = tid & (kMaxWidth - 1), t0 = tid / kMaxWidth;
  constexpr int PER = (TOK + 1) / 2;
  float xq[PER], xk[PER], xv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int t = t0 + 2 * i;
    const int64_t row = (int64_t)bh * n + t;
    xq[i] = t < n && f < d ? elem<T>::load(Q + row * d + f) : 0.f;
    xk[i] = t < n && f < d ? elem<T>::load(K + row * d + f) : 0.f;
    xv[i] = t < n && f < e ? elem<T>::load(V + row * e + f) : 0.f;
  }
  const float lam = __builtin_amdgcn_exp2f(-S[bh % g.h] * kLog2e);
  const int64_t base = (int64_t)bh * d * e + col;
  f32x4 st[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int r = rg + RG * i;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    st[i] = kv_in && col_ok && r < d ? (f32x4)*reinterpret_cast<const f32x4u *>(kv_in + base + (int64_t)r * e) : zero;
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int t = t0 + 2 * i;
    if (t < TOK) {
      sq[t][f] = xq[i];
      sk[t][f] = xk[i];
      sv[t][f] = xv[i];
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int t = 0; t < n; ++t) {
    const f32x4 v = *reinterpret_cast<const f32x4 *>(&sv[t][col & (kMaxWidth - 1)]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = rg + RG * i;
      const float qr = sq[t][r], kr = sk[t][r];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float a = fmaf(kr, v[x], st[i][x]);
        o[x] = fmaf(qr, a, o[x]);
        st[i][x] = lam * a;
      }
    }
    // the groups of rows of a wave, then (below) of the four waves
#pragma unroll
    for (int m = LC; m < 64; m *= 2)
#pragma unroll
      for (int x = 0; x < 4; ++x) o[x] += __shfl_xor(o[x], m);
    if ((tid & 63) < LC) *reinterpret_cast<f32x4 *>(&red[t][tid / 64][4 * (tid % LC)]) = o;
  }
  if (kv_out && col_ok) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = rg + RG * i;
      if (r < d) {
        *reinterpret_cast<f32x4u *>(kv_out + base + (int64_t)r * e) = st[i];
        if (g.twin) *reinterpret_cast<f32x4u *>(g.twin + base + (int64_t)r * e) = st[i];
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < n * 4 * LC; i += NT) {
    const int t = i / (4 * LC), c = i % (4 * LC);
    if (col0 + c < e)
      elem<T>::store(O + ((int64_t)bh * n + t) * e + col0 + c, (red[t][0][c] + red[t][1][c]) + (red[t][2][c] + red[t][3][c]));
  }
}

template <class T, int LC, int TOK>
int launch(const FwdArgs &a, const Geom &g, hipStream_t st) {
  const dim3 grid((unsigned)(g.b * g.h), (unsigned)((g.e + 4 * LC - 1) / (4 * LC)));
  ProfScope prof(KC_FUSED, st);
  la_step<T, LC, TOK><<<grid, NT, 0, st>>>((const T *)a.q, (const T *)a.k, (const T *)a.v, a.s, a.kv_in, a.kv_out, (T *)a.o, g);
  return (int)hipGetLastError();
}

template <class T>
int step_t(const FwdArgs &a, const Geom &g, hipStream_t st) {
  return g.n == 1 ? launch<T, 8, 1>(a, g, st) : launch<T, 8, LASP_STEP_TOKENS>(a, g, st);
}

}  // namespace

bool step_eligible(const Geom &g) { return g.n <= LASP_STEP_TOKENS && g.dt <= kMaxWidth && g.e % 4 == 0; }

int step_fwd(const FwdArgs &a, const Geom &g, int dtype, hipStream_t st) {
  switch (dtype) {
    case LASP_DTYPE_F32: return step_t<float>(a, g, st);
    case LASP_DTYPE_BF16: return step_t<bf16_tag>(a, g, st);
    case LASP_DTYPE_F16: return step_t<_Float16>(a, g, st);
  }
  return LASP_E_DTYPE;
}

}  // namespace lasp
