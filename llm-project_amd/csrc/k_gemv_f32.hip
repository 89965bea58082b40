// k_gemv_f32.hip - the fp32 (LLMA) decode path's kernels: the f32 matmul of one
// row (matrix.c:178-190) with the reference's summation order, and the small
// elementwise pieces of llama.c:296-362.
//
// Order: the reference forms c[j] = ((0 + a_0*W_0j) + a_1*W_1j) + ... in k order
// (the k loop is outer, j inner), every product rounded before its add.  Here
// each output column is one serial chain of K dependent adds, kept by one lane.
//
// Device layout of W ("panels of 16"): the reference's (K, N) row-major matrix is
// stored as ceil(N/16) panels of 16 columns, a panel as tiles of 16 k rows (K
// padded to 16 with zeros, columns past N zero).  A tile is 256 floats, lane l of
// a wave owning the four at 4*l: with l = 16*a + 4*s + b these are the k rows
// 4*s .. 4*s+3 of column 4*a + b.  One 16-byte load a lane moves a whole tile, and
// within a row of 16 lanes the four values of s (the next k rows of the same four
// columns) sit 4, 8 and 12 lanes up, where a DPP row shift reaches them.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "qdev_math.h"
#include "qdev_norm.h"
#include "qhip.h"
#include "qhip_internal.h"

namespace {

constexpr int kFC = 16;                        // columns (chains) per panel
constexpr int kFK = 16;                        // k rows per tile of a panel
constexpr int kFTile = kFC * kFK;              // floats per tile
constexpr int kFDepth = 8;                     // groups of four tiles in flight

enum { FMODE_PLAIN = 0, FMODE_RESID = 1, FMODE_RESID_BIAS = 2, FMODE_GELU_BIAS = 3, FMODE_SWIGLU = 4 };
enum { FPRO_NONE = 0, FPRO_RMS = 1, FPRO_LN = 2 };

// p, moved by a DPP control (row_shl:n is 0x100 + n: lane i takes lane i + n of
// its row of 16; a quad permutation that broadcasts lane c of each quad is
// 0x55 * c).  The compiler folds the move into the add or multiply that uses it.
template <int CTRL>
__device__ __forceinline__ float f_dpp(float p) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(p), CTRL, 0xf, 0xf, true));
}

// The lane's four products of tile C of a group.  x holds, in lane (s, c) of each
// row of 16, x[k0 + 16*c + 4*s .. +3] of the group's 64 k rows; tile C's are those
// of c = C.  Four multiplies form the 16 products of 16 columns.
template <int C>
__device__ __forceinline__ float4 f_products(const float4 &w, const float4 &x) {
  return make_float4(f_dpp<0x55 * C>(x.x) * w.x, f_dpp<0x55 * C>(x.y) * w.y, f_dpp<0x55 * C>(x.z) * w.z,
                     f_dpp<0x55 * C>(x.w) * w.w);
}

// acc takes the 16 products p of one tile in k order, in the lanes with s = 0
// (lane % 16 < 4; the other lanes' sums are never used); mid(i), i = 0..3, is work
// that does not touch acc or p.  A DPP operand must be two instructions old, and
// the compiler keeps that distance for the running sum as well: the work goes
// where it would otherwise put idle slots.
template <typename Mid>
__device__ __forceinline__ void f_sum(float &acc, const float4 &p, Mid mid) {
  acc += p.x; acc += p.y; acc += p.z; acc += p.w;
  __builtin_amdgcn_sched_barrier(0);
  mid(0);
  __builtin_amdgcn_sched_barrier(0);
  acc += f_dpp<0x104>(p.x);
  __builtin_amdgcn_sched_barrier(0);
  mid(1);
  __builtin_amdgcn_sched_barrier(0);
  acc += f_dpp<0x104>(p.y);
  __builtin_amdgcn_sched_barrier(0);
  mid(2);
  __builtin_amdgcn_sched_barrier(0);
  acc += f_dpp<0x104>(p.z);
  __builtin_amdgcn_sched_barrier(0);
  mid(3);
  __builtin_amdgcn_sched_barrier(0);
  acc += f_dpp<0x104>(p.w);
  acc += f_dpp<0x108>(p.x); acc += f_dpp<0x108>(p.y); acc += f_dpp<0x108>(p.z); acc += f_dpp<0x108>(p.w);
  acc += f_dpp<0x10c>(p.x); acc += f_dpp<0x10c>(p.y); acc += f_dpp<0x10c>(p.z); acc += f_dpp<0x10c>(p.w);
  __builtin_amdgcn_sched_barrier(0);
}

// 16 bytes of a buffer resource at the lane's offset vo (bytes); 0, and no memory
// traffic, past the resource's end.  The whole offset is in the vector operand: the
// range check does not cover the scalar one.
__device__ __forceinline__ float4 f_load16(__amdgpu_buffer_rsrc_t rs, int vo) {
  const auto r = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, 0, 0);
  float4 v;
  __builtin_memcpy(&v, &r, 16);
  return v;
}

// One wave per panel of 16 columns, no LDS and no barrier: the wave multiplies and
// adds a group of four tiles (64 k rows) while the loads of the next kFD groups
// (4 KiB of W and 256 bytes of x each) are in flight in registers.
// Bound: few columns (2048, 8192 inputs): the chain, 4.6 ns a k row (a dependent
// v_add_f32 alone takes 3.5 ns on a wave by itself, every other instruction or
// idle slot 1.7); many columns: HBM.  Against a block of 16 chain lanes fed with
// product tiles through LDS by seven producer waves: 8192 x 2048 40.7 -> 39.9 us,
// 2048 x 16384 32.0 -> 25.2, 2048 x 3072 13.2 -> 12.5, 2048 x 32000 52.9 -> 45.6
// (5.7 TB/s), 3072 x 768 15.9 -> 16.2.
//   out[j] = c[j] (+ bias[j]) or out[j] = out[j] + c[j] (llama.c:319-321, 347, 352);
// GPT-2 (model.c:505-514, feedforward.c:23-37): out[j] = out[j] + (c[j] + bias[j])
// and out[j] = gelu(c[j] + bias[j]) (activation.c:43-50)
template <int MODE, int kFD>
__global__ __launch_bounds__(64) void k_gemv_f32(const float *x, int K, const float *W, int N, float *out,
                                                const float *bias) {
  const int lane = threadIdx.x, s = (lane >> 2) & 3, c = lane & 3;
  const int kt = (K + kFK - 1) / kFK;                   // tiles of the panel
  const int ng = K / (4 * kFK);                         // whole groups of four
  const float *Wp = W + (size_t)blockIdx.x * kt * kFTile;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)Wp, (short)0, kt * kFTile * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, K * 4, 0x00020000);
  const int vw = lane * 16, vx = (16 * c + 4 * s) * 4;
  float4 w[kFD][4], xv[kFD];
  // the offsets of the group to request next: one register each, the tile a constant beside it
  int ow = vw, ox = vx;
  auto loadw = [&](int d, int t) __attribute__((always_inline)) { w[d][t] = f_load16(rw, ow + t * kFTile * 4); };
  auto loadx = [&](int d) __attribute__((always_inline)) { xv[d] = f_load16(rx, ox); };
  auto next = [&]() __attribute__((always_inline)) {
    ow += 4 * kFTile * 4;
    ox += 4 * kFK * 4;
    asm volatile("" : "+v"(ow), "+v"(ox));
  };
  float acc = 0.0f;
#pragma unroll
  for (int d = 0; d < kFD; d++) {
#pragma unroll
    for (int t = 0; t < 4; t++) loadw(d, t);
    loadx(d);
    next();
    __builtin_amdgcn_sched_barrier(0);      // groups arrive in order: a wait for one leaves the later ones in flight
  }
  int g0 = 0;
  // The products of a tile are formed during the sums of the one before it; a
  // group's registers take group g + kFD as their tiles' products are formed.
  float4 p = f_products<0>(w[0][0], xv[0]);
  for (; g0 + kFD < ng; g0 += kFD) {        // whole rounds: no branch inside, so the waits name only the loads in use
#pragma unroll
    for (int d = 0; d < kFD; d++) {
      const int e = (d + 1) % kFD;
      float4 q;
      f_sum(acc, p, [&](int i) {
        if (i == 0) q.x = f_dpp<0x55>(xv[d].x) * w[d][1].x;
        if (i == 1) q.y = f_dpp<0x55>(xv[d].y) * w[d][1].y;
        if (i == 2) q.z = f_dpp<0x55>(xv[d].z) * w[d][1].z;
        if (i == 3) q.w = f_dpp<0x55>(xv[d].w) * w[d][1].w;
      });
      f_sum(acc, q, [&](int i) {
        if (i == 1) loadw(d, 0);
        if (i == 0) p.x = f_dpp<0xaa>(xv[d].x) * w[d][2].x;
        if (i == 1) p.y = f_dpp<0xaa>(xv[d].y) * w[d][2].y;
        if (i == 2) p.z = f_dpp<0xaa>(xv[d].z) * w[d][2].z;
        if (i == 3) p.w = f_dpp<0xaa>(xv[d].w) * w[d][2].w;
      });
      f_sum(acc, p, [&](int i) {
        if (i == 1) loadw(d, 1);
        if (i == 0) q.x = f_dpp<0xff>(xv[d].x) * w[d][3].x;
        if (i == 1) q.y = f_dpp<0xff>(xv[d].y) * w[d][3].y;
        if (i == 2) q.z = f_dpp<0xff>(xv[d].z) * w[d][3].z;
        if (i == 3) q.w = f_dpp<0xff>(xv[d].w) * w[d][3].w;
      });
      f_sum(acc, q, [&](int i) {
        if (i == 1) loadw(d, 2);
        if (i == 2) loadw(d, 3);
        if (i == 3) {
          loadx(d);
          next();
        }
        if (i == 0) p.x = f_dpp<0>(xv[e].x) * w[e][0].x;
        if (i == 1) p.y = f_dpp<0>(xv[e].y) * w[e][0].y;
        if (i == 2) p.z = f_dpp<0>(xv[e].z) * w[e][0].z;
        if (i == 3) p.w = f_dpp<0>(xv[e].w) * w[e][0].w;
      });
    }
  }
  auto none = [](int) {};
#pragma unroll
  for (int d = 0; d < kFD; d++) {           // the last 1 .. kFD groups: nothing left to load
    if (g0 + d < ng) {
      f_sum(acc, f_products<0>(w[d][0], xv[d]), none);
      f_sum(acc, f_products<1>(w[d][1], xv[d]), none);
      f_sum(acc, f_products<2>(w[d][2], xv[d]), none);
      f_sum(acc, f_products<3>(w[d][3], xv[d]), none);
    }
  }
  if (ng * 4 < kt) {       // the rest: up to four tiles, x zero past K (a zero product leaves the chain as it is)
    const int k0 = ng * 4 * kFK + 16 * c + 4 * s;
    float4 wt[4], xt;
#pragma unroll
    for (int t = 0; t < 4; t++) wt[t] = f_load16(rw, vw + (4 * ng + t) * kFTile * 4);       // 0 past the panel
    xt.x = k0 < K ? x[k0] : 0.0f;
    xt.y = k0 + 1 < K ? x[k0 + 1] : 0.0f;
    xt.z = k0 + 2 < K ? x[k0 + 2] : 0.0f;
    xt.w = k0 + 3 < K ? x[k0 + 3] : 0.0f;
    f_sum(acc, f_products<0>(wt[0], xt), none);
    f_sum(acc, f_products<1>(wt[1], xt), none);
    f_sum(acc, f_products<2>(wt[2], xt), none);
    f_sum(acc, f_products<3>(wt[3], xt), none);
  }
  const int j = blockIdx.x * kFC + 4 * (lane >> 4) + c;
  if (s == 0 && j < N) {
    if (MODE == FMODE_RESID) out[j] = out[j] + acc;
    else if (MODE == FMODE_RESID_BIAS) out[j] = out[j] + (acc + bias[j]);
    else if (MODE == FMODE_GELU_BIAS) out[j] = qd::gelu_tanh(acc + bias[j]);
    else out[j] = bias ? acc + bias[j] : acc;
  }
}

// Two chains at once (the gate and the up panel of one column group): the other
// chain's adds are the work between a chain's DPP adds.
template <typename Mid>
__device__ __forceinline__ void f_sum2(float &a0, float &a1, const float4 &p, const float4 &q, Mid mid) {
#define F_PAIR(ctrl, e)                                                     \
  a0 += f_dpp<ctrl>(p.e);                                                   \
  __builtin_amdgcn_sched_barrier(0);                                        \
  a1 += f_dpp<ctrl>(q.e);                                                   \
  __builtin_amdgcn_sched_barrier(0)
  a0 += p.x; a1 += q.x; a0 += p.y; a1 += q.y; a0 += p.z; a1 += q.z; a0 += p.w; a1 += q.w;
  __builtin_amdgcn_sched_barrier(0);
  F_PAIR(0x104, x); mid(0); F_PAIR(0x104, y); mid(1); F_PAIR(0x104, z); mid(2); F_PAIR(0x104, w); mid(3);
  F_PAIR(0x108, x); mid(4); F_PAIR(0x108, y); mid(5); F_PAIR(0x108, z); mid(6); F_PAIR(0x108, w); mid(7);
  F_PAIR(0x10c, x); F_PAIR(0x10c, y); F_PAIR(0x10c, z); F_PAIR(0x10c, w);
#undef F_PAIR
}

// Product m of tile C (f_products, one at a time).
template <int C>
__device__ __forceinline__ float f_product1(const float4 &w, const float4 &x, int m) {
  return m == 0 ? f_dpp<0x55 * C>(x.x) * w.x : m == 1 ? f_dpp<0x55 * C>(x.y) * w.y
       : m == 2 ? f_dpp<0x55 * C>(x.z) * w.z : f_dpp<0x55 * C>(x.w) * w.w;
}
__device__ __forceinline__ void f_set(float4 &v, int m, float x) {
  if (m == 0) v.x = x;
  else if (m == 1) v.y = x;
  else if (m == 2) v.z = x;
  else v.w = x;
}

// Where a GEMV of [q | k | v] (GPT-2) also appends the new position's rows
// (model.c:481-482) to the caches laid out [head][max_seq][head_dim].
struct FAppend {
  const int *d_state;
  float *kc, *vc;
  int dm, hd, max_seq;
};

// The GEMV over a row that each block normalizes for itself (K <= 256 * CM): rmsnorm
// (rmsnorm.c:7-21) or LayerNorm into LDS by its four waves, while the first groups of
// the panel's W are in flight; then wave 0 sums the panel as k_gemv_f32 does, x from
// LDS, and the others end.  SwiGLU (swiglu.c:7-10, 36-39): the wave sums a gate panel
// and the matching up panel, one chain's adds between the other's, and stores h.
// Bound: the norm's serial sum, then the panel's chains; what it saves is a one-block
// kernel and its boundaries, after which the GEMV would first wait for its loads.
// Kernel times, against the separate kernels': K = 2048, rmsnorm + 3072 columns
// 5.3 + 12.5 -> 15.4 us, rmsnorm + 2 x 8192 + SwiGLU 5.3 + 25.2 + 4.7 -> 26.8;
// K = 768, LayerNorm + 2304 columns + append 7.4 + 6.4 + 1.6 -> 12.8, LayerNorm +
// 3072 with GELU 7.4 + 8.0 -> 14.0.  One wave a block forming the norm alone: 18.2,
// 30.0, 13.7, 15.4; four panels a block (all four waves sum, a quarter of the
// CUs): 17.1, 30.6, 13.9, 15.8.
constexpr int kFNW = 4;           // waves per block, for the norm; wave 0 then sums the panel

template <int MODE, int PRO, int CM, int kFD>
__global__ __launch_bounds__(64 * kFNW) void k_gemv_f32_norm(const float *x, int K, const float *gamma,
                                                            const float *beta, float eps, const float *W, int N,
                                                            float *out, const float *bias, FAppend ap) {
  constexpr int NP = MODE == FMODE_SWIGLU ? 2 : 1, NT = 64 * kFNW;
  __shared__ __attribute__((aligned(16))) float xs[NT * CM];
  __shared__ qd::SeqScratch seq;
  __shared__ float red[kFNW];
  const int lane = threadIdx.x & 63, s = (lane >> 2) & 3, c = lane & 3, j0 = threadIdx.x * CM;
  const int kt = (K + kFK - 1) / kFK, ng = (kt + 3) / 4;               // tiles; groups of four, the last perhaps short
  const int np = (N + kFC - 1) / kFC;
  const int panel = blockIdx.x;
  const bool chains = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0;
  float y[CM], gm[CM], be[PRO == FPRO_LN ? CM : 1];
  qd::rmsnorm_load<CM>(x, K, gamma, y, gm);
  if constexpr (PRO == FPRO_LN) {
#pragma unroll
    for (int i = 0; i < CM; i++) be[i] = j0 + i < K ? beta[j0 + i] : 0.0f;
  }
  __builtin_amdgcn_sched_barrier(0);          // the row first: loads return in order
  __amdgpu_buffer_rsrc_t rw[NP];
#pragma unroll
  for (int n = 0; n < NP; n++) {
    const float *Wp = W + ((size_t)panel + (size_t)n * np) * kt * kFTile;
    rw[n] = __builtin_amdgcn_make_buffer_rsrc((void *)Wp, (short)0, chains ? kt * kFTile * 4 : 0, 0x00020000);
  }
  const int vw = lane * 16;
  float4 w[kFD][NP][4], xv[kFD];
  int ow = vw;                                // of the group to request next
  auto loadw = [&](int d, int t) __attribute__((always_inline)) {       // past the panel's end: reads 0, no traffic
#pragma unroll
    for (int n = 0; n < NP; n++) w[d][n][t] = f_load16(rw[n], ow + t * kFTile * 4);
  };
  auto next = [&]() __attribute__((always_inline)) {
    ow += 4 * kFTile * 4;
    asm volatile("" : "+v"(ow));
  };
  auto loadx = [&](int d, int g) __attribute__((always_inline)) {              // groups past the last: the last again
    xv[d] = *reinterpret_cast<const float4 *>(&xs[min(g, ng - 1) * 4 * kFK + 16 * c + 4 * s]);
  };
#pragma unroll
  for (int d = 0; d < kFD; d++) {
#pragma unroll
    for (int t = 0; t < 4; t++) loadw(d, t);
    next();
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (PRO == FPRO_LN) qd::layernorm_apply<NT, CM>(x, K, eps, y, gm, be, xs, &red[0], seq);
  else (void)qd::rmsnorm_apply<NT, CM>(x, K, eps, y, gm, red, seq);
#pragma unroll
  for (int i = 0; i < CM; i += 4) {
    float4 v = make_float4(y[i], y[i + 1], y[i + 2], y[i + 3]);
    if (j0 + i >= K) v.x = 0.0f;                // LayerNorm leaves garbage past K
    if (j0 + i + 1 >= K) v.y = 0.0f;
    if (j0 + i + 2 >= K) v.z = 0.0f;
    if (j0 + i + 3 >= K) v.w = 0.0f;
    *reinterpret_cast<float4 *>(&xs[j0 + i]) = v;
  }
  qd::lds_sync();                               // the last barrier
  if (!chains) return;
#pragma unroll
  for (int d = 0; d < kFD; d++) loadx(d, d);

  float acc[NP];
#pragma unroll
  for (int n = 0; n < NP; n++) acc[n] = 0.0f;
  // one tile's sums, with the products of the next formed and `more` requested meanwhile
  float4 p[2][NP];
  auto tile = [&](auto cv, auto &cur, auto &nxt, const float4 (&wn)[NP][4], const float4 &xn, auto more)
      __attribute__((always_inline)) {
    constexpr int C = decltype(cv)::value;      // tile of its group that `nxt` is of
    if constexpr (NP == 1) {
      f_sum(acc[0], cur[0], [&](int i) __attribute__((always_inline)) {
        f_set(nxt[0], i, f_product1<C>(wn[0][C], xn, i));
        more(i);
      });
    } else {
      f_sum2(acc[0], acc[NP - 1], cur[0], cur[NP - 1], [&](int i) __attribute__((always_inline)) {
        f_set(nxt[i >> 2], i & 3, f_product1<C>(wn[i >> 2][C], xn, i & 3));
        if (i < 4) more(i);
      });
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;
  auto none = [](int) {};
#pragma unroll
  for (int n = 0; n < NP; n++) p[0][n] = f_products<0>(w[0][n][0], xv[0]);
  int g0 = 0;
  for (; g0 + kFD < ng; g0 += kFD) {
#pragma unroll
    for (int d = 0; d < kFD; d++) {
      const int g = g0 + d + kFD, e = (d + 1) % kFD;
      tile(C1(), p[0], p[1], w[d], xv[d], none);
      tile(C2(), p[1], p[0], w[d], xv[d], [&](int i) __attribute__((always_inline)) { if (i == 1) loadw(d, 0); });
      tile(C3(), p[0], p[1], w[d], xv[d], [&](int i) __attribute__((always_inline)) { if (i == 1) loadw(d, 1); });
      tile(C0(), p[1], p[0], w[e], xv[e], [&](int i) __attribute__((always_inline)) {
        if (i == 1) loadw(d, 2);
        if (i == 2) loadw(d, 3);
        if (i == 3) {
          loadx(d, g);
          next();
        }
      });
    }
  }
#pragma unroll
  for (int d = 0; d < kFD; d++) {               // the last 1 .. kFD groups (a short one's missing tiles are 0)
    if (g0 + d < ng) {
      const int e = (d + 1) % kFD;
      tile(C1(), p[0], p[1], w[d], xv[d], none);
      tile(C2(), p[1], p[0], w[d], xv[d], none);
      tile(C3(), p[0], p[1], w[d], xv[d], none);
      tile(C0(), p[1], p[0], w[e], xv[e], none);
    }
  }
  const int j = panel * kFC + 4 * (lane >> 4) + c;
  if (s == 0 && j < N) {
    if (MODE == FMODE_SWIGLU) {
      const float z = acc[0], sg = 1.0f / (1.0f + qd::expf_glibc(-z));
      out[j] = (z * sg) * acc[NP - 1];
    } else if (MODE == FMODE_GELU_BIAS) {
      out[j] = qd::gelu_tanh(acc[0] + bias[j]);
    } else {
      const float v = bias ? acc[0] + bias[j] : acc[0];
      out[j] = v;
      if (PRO == FPRO_LN && ap.d_state && j >= ap.dm) {
        const int i = j < 2 * ap.dm ? j - ap.dm : j - 2 * ap.dm, h = i / ap.hd;
        (j < 2 * ap.dm ? ap.kc : ap.vc)[((size_t)h * ap.max_seq + ap.d_state[0]) * ap.hd + (i - h * ap.hd)] = v;
      }
    }
  }
}

// (K, N) row-major -> panels of 16 columns (see the top of this file).  A block
// takes 16 k rows of 256 columns, read row by row and written tile by tile.
__global__ __launch_bounds__(256) void k_to_panels(const float *src, int K, int N, float *dst) {
  __shared__ float t[kFK][256 + 1];
  const int kt = (K + kFK - 1) / kFK, k0 = blockIdx.y * kFK, j0 = blockIdx.x * 256, tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < kFK; i++) t[i][tid] = k0 + i < K && j0 + tid < N ? src[(size_t)(k0 + i) * N + j0 + tid] : 0.0f;
  __syncthreads();
  const int l = tid >> 2, k = 4 * ((l >> 2) & 3) + (tid & 3), j = 4 * (l >> 4) + (l & 3);
  for (int p = 0; p < 256 / kFC && j0 + p * kFC < N; p++)
    dst[((size_t)(j0 / kFC + p) * kt + blockIdx.y) * kFTile + tid] = t[k][p * kFC + j];
}

// x = wte[token] (llama.c:304), token = d_in[d_state[0]]
__global__ void k_embed_f32(const float *wte, int dm, const int *d_in, const int *d_state, float *x) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= dm) return;
  x[j] = wte[(size_t)d_in[d_state[0]] * dm + j];
}

// Row r of x = wte[ids[r]] (llama.c:172-174)
__global__ void k_embed_f32_rows(const float *wte, int dm, const int *ids, float *x) {
  const int j = blockIdx.x * 256 + threadIdx.x, r = blockIdx.y;
  if (j >= dm) return;
  x[(size_t)r * dm + j] = wte[(size_t)ids[r] * dm + j];
}

// y = rmsnorm(x) (rmsnorm.c:7-21), one block per row of dm floats
template <int NT, int CM>
__global__ __launch_bounds__(NT) void k_rmsnorm_f32(const float *x, int dm, const float *gamma, float eps, float *y) {
  __shared__ float red[NT / 64];
  __shared__ qd::SeqScratch seq;
  x += (size_t)blockIdx.x * dm;
  y += (size_t)blockIdx.x * dm;
  float v[CM];
  (void)qd::rmsnorm_row<NT, CM>(x, dm, gamma, eps, v, red, seq);
  const int j0 = threadIdx.x * CM;
#pragma unroll
  for (int c = 0; c < CM; c++)
    if (j0 + c < dm) y[j0 + c] = v[c];
}

// h = SiLU(g) * u = (g * (1 / (1 + expf(-g)))) * u over gu = [g | u] (swiglu.c:7-10, 36-39),
// row blockIdx.y of gu [rows][2 dff] into h [rows][dff]
__global__ void k_swiglu_f32(const float *gu, int dff, float *h) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= dff) return;
  gu += (size_t)blockIdx.y * 2 * dff;
  h += (size_t)blockIdx.y * dff;
  const float z = gu[j];
  const float s = 1.0f / (1.0f + qd::expf_glibc(-z));
  h[j] = (z * s) * gu[dff + j];
}

// ---------------------------------------------------------------------------
// Many-row f32 matmul (matrix.c:178-190 over M rows): the GEMMs of the batched
// forward.  Every output element is one serial chain in k order, the reference's,
// with each product rounded before its add: a v_mul_f32 and a v_add_f32 a k row.
//
// A lane owns one column and R rows, a wave 64 columns (four panels), a block of
// eight waves 8 * R rows of the same columns.  A row's value at a k row is the
// same for the whole wave, so it comes through the scalar cache into SGPRs and is
// the multiply's scalar operand: it costs no vector register, no LDS read and no
// vector issue slot.  For that A is first packed by groups of R rows,
// [ceil(M/R)][K][R], so that a wave reads one contiguous stream (R = 1: A itself).
// W goes through LDS, 32 k rows a stage in two buffers with two more stages in
// flight in registers, and a lane reads four k rows of its column at a time.
// Bound: the VALU, two instructions a multiply-add without FMA (65 T lane-ops/s
// reached by multiplies and adds alone), where eight waves a SIMD cover the scalar
// loads; the loads' latency where a narrow output leaves fewer.  512 rows: K = 2048,
// N = 16384 814 -> 626 us (54.9 TFLOP/s), N = 32000 1522 -> 1230, N = 3072
// 264 -> 134; K = 8192, N = 2048 960 -> 377 (45.6), against 64 x 64 tiles of
// 4 x 4 sums a thread with both operands read from LDS.
// ---------------------------------------------------------------------------
constexpr int kGW = 8;            // waves per block
constexpr int kGN = 64;           // columns per block: four panels
constexpr int kGK = 2 * kFK;      // k rows per LDS stage

// rows of A -> groups of R rows, k rows outermost within a group (rows past M zero)
template <int R>
__global__ __launch_bounds__(256) void k_pack_rows(const float *A, int M, int K, float *P) {
  const int k = blockIdx.x * 256 + threadIdx.x, i0 = blockIdx.y * R;
  if (k >= K) return;
  float v[R];
#pragma unroll
  for (int r = 0; r < R; r++) v[r] = i0 + r < M ? A[(size_t)(i0 + r) * K + k] : 0.0f;
  float *o = P + ((size_t)blockIdx.y * K + k) * R;
#pragma unroll
  for (int r = 0; r < R; r++) o[r] = v[r];
}

// N floats from a wave-uniform address, into SGPRs
template <int N>
struct SRow { typedef float V __attribute__((ext_vector_type(N), aligned(4))); };

template <int MODE, int R>
__global__ __launch_bounds__(64 * kGW) void k_gemm_f32(const float *Ap, int M, int K, const float *W, int N, float *out,
                                                      const float *bias, int mt, int nt) {
  constexpr int KB = R >= 8 ? 4 : 8, QB = KB / 4;     // k rows of a scalar batch
  typedef typename SRow<R * KB>::V Batch;
  typedef const __attribute__((address_space(4))) Batch *BatchPtr;
  typedef const __attribute__((address_space(4))) float *ScalarPtr;
  __shared__ float4 ws[2][kGK * kGN / 4];
  const int b8 = blockIdx.x >> 3, mtile = b8 % mt, ntile = 8 * (b8 / mt) + (blockIdx.x & 7);
  if (ntile >= nt) return;                            // uniform for the block
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = (mtile * kGW + wave) * R, np = (N + kFC - 1) / kFC, kt = (K + kFK - 1) / kFK;
  const bool work = i0 < M;                           // a wave past the last row only helps to stage
  // staging: float4 tid of a stage is panel tid / 128, tile (tid / 64) % 2, part l of the tile; part
  // l = 16*a + 4*s + b goes to slot 16*a + 4*(s ^ a) + b, so that the 16 columns of a panel, read at
  // one s, fall in distinct banks
  const int l = lane, pnl = ntile * 4 + (tid >> 7), tsub = (tid >> 6) & 1;
  const int wslot = (tid & ~63) + (l & 48) + 4 * (((l >> 2) & 3) ^ (l >> 4)) + (l & 3);
  const float4 *Wl = reinterpret_cast<const float4 *>(W) + ((size_t)min(pnl, np - 1) * kt) * (kFTile / 4) + l;
  auto gload = [&](int st) __attribute__((always_inline)) {
    return Wl[(size_t)min(2 * st + tsub, kt - 1) * (kFTile / 4)];     // past the last tile or panel: staged, never summed or stored
  };
  // this lane's column: slot of k rows 4*s .. +3 of tile t of a stage
  const int ca = (lane >> 2) & 3, cslot = (lane >> 4) * 128 + 16 * ca + (lane & 3);
  int rslot[4];
#pragma unroll
  for (int s = 0; s < 4; s++) rslot[s] = cslot + 4 * (s ^ ca);
  const ScalarPtr As = (ScalarPtr)(uintptr_t)(Ap + (size_t)(i0 / R) * K * R);
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = 0.0f;

  Batch av[2];
  float4 wv[2][QB];
  // nb batches of KB k rows of the stage at k0, from LDS buffer buf; av[0] holds the first on entry and
  // the next stage's first on exit
  auto sum = [&](int buf, int k0, int nb) __attribute__((always_inline)) {
    constexpr int NB = kGK / KB;
    ScalarPtr p = As + (size_t)k0 * R;
    // the batch after the last: the next stage's first, or (nothing follows) one this wave has read
    ScalarPtr pn = k0 + (nb + 1) * KB <= K ? p + nb * KB * R : As;
    auto wload = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < QB; i++) wv[u & 1][i] = ws[buf][rslot[(u * QB + i) & 3] + ((u * QB + i) >> 2) * 64];
    };
    wload(0);
#pragma unroll
    for (int u = 0; u < NB; u++) {
      if (u < nb) {
        // scalar loads return out of order, so a wait is for all of them: this batch's, requested a
        // batch ago, before the next one's are requested
        __builtin_amdgcn_s_waitcnt(0xC07F);
        if (u + 1 < NB) wload(u + 1);
        av[(u + 1) & 1] = *(BatchPtr)(u + 1 < NB && u + 1 < nb ? p + (u + 1) * KB * R : pn);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < KB; e++) {
          const float4 w4 = wv[u & 1][e >> 2];
          const float w = (e & 3) == 0 ? w4.x : (e & 3) == 1 ? w4.y : (e & 3) == 2 ? w4.z : w4.w;
          float m[R];
#pragma unroll
          for (int r = 0; r < R; r++) m[r] = av[u & 1][e * R + r] * w;
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int r = 0; r < R; r++) acc[r] = acc[r] + m[r];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  // the wave's part of stage t of A, touched (one value a 128-byte line) so that its scalar loads find it in L2
  const float *At = Ap + (size_t)(work ? i0 / R : 0) * K * R;
  auto touch = [&](int t) __attribute__((always_inline)) {
    return At[(unsigned)min(t * kGK * R + (lane & (R - 1)) * 32, K * R - 1)];
  };

  float4 g[2];
  g[0] = gload(0);
  g[1] = gload(1);
  float pf = touch(1);
  if (work && K >= KB) av[0] = *(BatchPtr)As;
  ws[0][wslot] = g[0];
  g[0] = gload(2);
  qd::lds_sync();
  const int nst = K / kGK;
  auto stage = [&](auto par, int t) __attribute__((always_inline)) {   // stage t, parity par
    constexpr int P = decltype(par)::value;
    ws[P ^ 1][wslot] = g[P ^ 1];                      // that buffer was last read in stage t - 1
    asm volatile("" ::"v"(pf));
    pf = touch(t + 2);
    g[P ^ 1] = gload(t + 3);
    __builtin_amdgcn_sched_barrier(0);
    if (work) sum(P, t * kGK, kGK / KB);
    qd::lds_sync();
  };
  int t = 0;
  for (; t + 2 <= nst; t += 2) {
    stage(std::integral_constant<int, 0>(), t);
    stage(std::integral_constant<int, 1>(), t + 1);
  }
  ws[1][wslot] = g[1];                                // t is even: buffer 0 holds stage t, and t + 1 is the last
  for (; t * kGK < K; t++) {                          // a whole stage, a partial one, or both (a chain takes exactly K terms)
    const int kn = min(kGK, K - t * kGK), nb = kn / KB, buf = t & 1;
    if (buf) qd::lds_sync();
    if (!work) continue;
    sum(buf, t * kGK, nb);
    for (int k = nb * KB; k < kn; k++) {
      const float w = reinterpret_cast<const float *>(&ws[buf][cslot + 4 * (((k >> 2) & 3) ^ ca) + (k >> 4) * 64])[k & 3];
#pragma unroll
      for (int r = 0; r < R; r++) acc[r] = acc[r] + As[(size_t)(t * kGK + k) * R + r] * w;
    }
  }
  if (!work) return;
  const int j = ntile * kGN + lane;
  if (j >= N) return;
  const float bj = MODE == FMODE_PLAIN && bias ? bias[j] : 0.0f;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (i0 + r >= M) break;
    float *o = out + (size_t)(i0 + r) * N + j;
    if (MODE == FMODE_RESID) *o = *o + acc[r];
    else *o = bias ? acc[r] + bj : acc[r];
  }
}

template <int R>
int launch_gemm(int mode, int cls, const float *A, int M, int K, const float *W, int N, float *out, const float *bias,
                float *pack) {
  const int mt = (M + kGW * R - 1) / (kGW * R), nt = (N + kGN - 1) / kGN;
  const dim3 grid(8 * mt * ((nt + 7) / 8)), block(64 * kGW);
  if (R > 1) {
    QH_LAUNCH(cls, k_pack_rows<R>, dim3((K + 255) / 256, (M + R - 1) / R), dim3(256), 0, A, M, K, pack);
    A = pack;
  }
  if (mode == 0) QH_LAUNCH(cls, (k_gemm_f32<FMODE_PLAIN, R>), grid, block, 0, A, M, K, W, N, out, bias, mt, nt);
  else QH_LAUNCH(cls, (k_gemm_f32<FMODE_RESID, R>), grid, block, 0, A, M, K, W, N, out, bias, mt, nt);
  return 0;
}

}  // namespace

// Largest K the fp32 GEMV takes (a panel stays within a buffer resource's 32-bit offsets).
extern "C" int qhip_gemv_f32_max_k(void) { return 32768; }

extern "C" int qhip_gemv_f32(int mode, int cls, const float *x, int K, const float *W, int N, float *out,
                             const float *bias) {
  if (K <= 0 || N <= 0 || K > qhip_gemv_f32_max_k()) return qh::fail_msg("gemv_f32: bad shape");
  if (mode < 0 || mode > 3 || (mode >= 2 && !bias)) return qh::fail_msg("gemv_f32: bad mode");
  const dim3 grid((N + kFC - 1) / kFC), block(64);
  switch (mode) {
    case 0: QH_LAUNCH(cls, (k_gemv_f32<FMODE_PLAIN, kFDepth>), grid, block, 0, x, K, W, N, out, bias); break;
    case 1: QH_LAUNCH(cls, (k_gemv_f32<FMODE_RESID, kFDepth>), grid, block, 0, x, K, W, N, out, bias); break;
    case 2: QH_LAUNCH(cls, (k_gemv_f32<FMODE_RESID_BIAS, kFDepth>), grid, block, 0, x, K, W, N, out, bias); break;
    default: QH_LAUNCH(cls, (k_gemv_f32<FMODE_GELU_BIAS, kFDepth>), grid, block, 0, x, K, W, N, out, bias); break;
  }
  return 0;
}

// Whether qhip_gemv_f32_norm takes this shape: panels that do not mix gate and up
// columns (SwiGLU), at most 1024 of them (four blocks a CU: every block forms the
// norm at once, none waits for another's to end), and K up to 2048 (measured ahead
// of the separate kernels from 48 to 2048, at the head of this kernel; a longer row's
// weights stream for much longer than the kernel that this saves).
extern "C" int qhip_gemv_f32_norm_ok(int mode, int K, int N) {
  return K >= 1 && K <= 64 * kFNW * 8 && (mode != FMODE_SWIGLU || N % kFC == 0) && (N + kFC - 1) / kFC <= 1024;
}

extern "C" int qhip_gemv_f32_norm(int pro, int mode, int cls, const float *x, int K, const float *gamma,
                                  const float *beta, float eps, const float *W, int N, float *out, const float *bias,
                                  const int *d_state, float *kc, float *vc, int hd, int max_seq) {
  if (!qhip_gemv_f32_norm_ok(mode, K, N) || N <= 0) return qh::fail_msg("gemv_f32_norm: unsupported shape");
  const int np = (N + kFC - 1) / kFC;
  const dim3 grid(np), block(64 * kFNW);
  const FAppend ap{d_state, kc, vc, N / 3, hd, max_seq};
#define F_NORM(MODE, PRO, FD)                                                                                         \
  do {                                                                                                                \
    if (K <= 64 * kFNW * 4) QH_LAUNCH(cls, (k_gemv_f32_norm<MODE, PRO, 4, FD>), grid, block, 0, x, K, gamma, beta,   \
                                      eps, W, N, out, bias, ap);                                                     \
    else QH_LAUNCH(cls, (k_gemv_f32_norm<MODE, PRO, 8, FD>), grid, block, 0, x, K, gamma, beta, eps, W, N, out, bias, \
                   ap);                                                                                               \
    return 0;                                                                                                         \
  } while (0)
  if (pro == FPRO_RMS && mode == FMODE_PLAIN) F_NORM(FMODE_PLAIN, FPRO_RMS, kFDepth);
  if (pro == FPRO_RMS && mode == FMODE_SWIGLU) F_NORM(FMODE_SWIGLU, FPRO_RMS, 5);
  if (pro == FPRO_LN && mode == FMODE_PLAIN) F_NORM(FMODE_PLAIN, FPRO_LN, kFDepth);
  if (pro == FPRO_LN && mode == FMODE_GELU_BIAS && bias) F_NORM(FMODE_GELU_BIAS, FPRO_LN, kFDepth);
#undef F_NORM
  return qh::fail_msg("gemv_f32_norm: bad mode");
}

// Floats of a (K, N) matrix in the panel layout.
extern "C" size_t qhip_panels_f32_size(int K, int N) { return (size_t)((K + kFK - 1) / kFK) * ((N + kFC - 1) / kFC) * kFTile; }

extern "C" int qhip_to_panels_f32(const float *src, int K, int N, float *dst) {
  if (K <= 0 || N <= 0 || K > qhip_gemv_f32_max_k()) return qh::fail_msg("to_panels_f32: bad shape");
  QH_LAUNCH(QK_OTHER, k_to_panels, dim3((N + 255) / 256, (K + kFK - 1) / kFK), dim3(256), 0, src, K, N, dst);
  return 0;
}

extern "C" int qhip_embed_f32(const float *wte, int dm, const int *d_in, const int *d_state, float *x) {
  QH_LAUNCH(QK_EMBED, k_embed_f32, dim3((dm + 255) / 256), dim3(256), 0, wte, dm, d_in, d_state, x);
  return 0;
}

extern "C" int qhip_rmsnorm_f32_rows(const float *x, int R, int dm, const float *gamma, float eps, float *y) {
  const dim3 g(R);
  if (R <= 0) return qh::fail_msg("rmsnorm_f32: no rows");
  if (dm <= 256 * 4) QH_LAUNCH(QK_RMSNORM, (k_rmsnorm_f32<256, 4>), g, dim3(256), 0, x, dm, gamma, eps, y);
  else if (dm <= 256 * 8) QH_LAUNCH(QK_RMSNORM, (k_rmsnorm_f32<256, 8>), g, dim3(256), 0, x, dm, gamma, eps, y);
  else if (dm <= 256 * 16) QH_LAUNCH(QK_RMSNORM, (k_rmsnorm_f32<256, 16>), g, dim3(256), 0, x, dm, gamma, eps, y);
  else if (dm <= 256 * 32) QH_LAUNCH(QK_RMSNORM, (k_rmsnorm_f32<256, 32>), g, dim3(256), 0, x, dm, gamma, eps, y);
  else if (dm <= 1024 * 16) QH_LAUNCH(QK_RMSNORM, (k_rmsnorm_f32<1024, 16>), g, dim3(1024), 0, x, dm, gamma, eps, y);
  else return qh::fail_msg("rmsnorm_f32: d_model above 16384");
  return 0;
}

extern "C" int qhip_rmsnorm_f32(const float *x, int dm, const float *gamma, float eps, float *y) {
  return qhip_rmsnorm_f32_rows(x, 1, dm, gamma, eps, y);
}

extern "C" int qhip_swiglu_f32_rows(const float *gu, int R, int dff, float *h) {
  QH_LAUNCH(QK_SWIGLU, k_swiglu_f32, dim3((dff + 255) / 256, R), dim3(256), 0, gu, dff, h);
  return 0;
}

extern "C" int qhip_swiglu_f32(const float *gu, int dff, float *h) { return qhip_swiglu_f32_rows(gu, 1, dff, h); }

extern "C" int qhip_embed_f32_rows(const float *wte, int dm, const int *ids, int R, float *x) {
  QH_LAUNCH(QK_EMBED, k_embed_f32_rows, dim3((dm + 255) / 256, R), dim3(256), 0, wte, dm, ids, x);
  return 0;
}

// Floats of qhip_gemm_f32's pack workspace.
extern "C" size_t qhip_gemm_f32_pack(int M, int K) { return (size_t)((M + 7) / 8) * 8 * K; }

extern "C" int qhip_gemm_f32(int mode, int cls, const float *A, int M, int K, const float *W, int N, float *out,
                             const float *bias, float *pack) {
  if (M <= 0 || K <= 0 || N <= 0) return qh::fail_msg("gemm_f32: bad shape");
  if (mode != 0 && mode != 1) return qh::fail_msg("gemm_f32: bad mode");
  // Rows per wave.  A CU spends R + 0.65 units (4.4 ns) a k row on each of its blocks (R multiply-add
  // pairs, and the reads around them), but no less than a batch of scalar loads takes to come back,
  // which only other waves can cover: with one block a CU at least 3.0, 3.5, 4.7 and 14 units for R = 1,
  // 2, 4, 8.  The R of the least time, the largest of equals (W is then read by fewer blocks).
  // Measured, us (K = 8192, N = 2048): 50 rows 110 134 177 306 for R = 1 2 4 8, 130 rows 183 185 189 451,
  // 512 rows 513 423 377 529; (K = 2048, N = 16384) 512 rows 986 784 662 626.
  static const int least[4] = {300, 350, 470, 1400};
  const int cus = qh::num_cus() > 0 ? qh::num_cus() : 256, nt = (N + kGN - 1) / kGN;
  int best = 1;
  long long cost = 0;
  for (int i = 0; i < 4; i++) {
    const int R = 1 << i;
    const long long blocks = (long long)((M + kGW * R - 1) / (kGW * R)) * nt;
    long long c = ((blocks + cus - 1) / cus) * (100 * R + 65);
    if (c < least[i]) c = least[i];
    if (i == 0 || c <= cost) { best = R; cost = c; }
  }
  switch (best) {
    case 1: return launch_gemm<1>(mode, cls, A, M, K, W, N, out, bias, pack);
    case 2: return launch_gemm<2>(mode, cls, A, M, K, W, N, out, bias, pack);
    case 4: return launch_gemm<4>(mode, cls, A, M, K, W, N, out, bias, pack);
    default: return launch_gemm<8>(mode, cls, A, M, K, W, N, out, bias, pack);
  }
}
