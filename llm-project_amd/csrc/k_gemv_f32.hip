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

#include "qdev_math.h"
#include "qdev_norm.h"
#include "qhip.h"
#include "qhip_internal.h"

namespace {

constexpr int kFC = 16;                        // columns (chains) per panel
constexpr int kFK = 16;                        // k rows per tile of a panel
constexpr int kFTile = kFC * kFK;              // floats per tile
constexpr int kFDepth = 8;                     // groups of four tiles in flight

enum { FMODE_PLAIN = 0, FMODE_RESID = 1, FMODE_RESID_BIAS = 2, FMODE_GELU_BIAS = 3 };

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

// 16 bytes of a buffer resource at the lane's offset vo plus the wave's so (bytes);
// 0 past the resource's end.
__device__ __forceinline__ float4 f_load16(__amdgpu_buffer_rsrc_t rs, int vo, int so) {
  const auto r = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0);
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
  auto loadw = [&](int d, int g, int t) { w[d][t] = f_load16(rw, vw + t * kFTile * 4, g * 4 * kFTile * 4); };
  auto loadx = [&](int d, int g) { xv[d] = f_load16(rx, vx, g * 4 * kFK * 4); };   // past the last group: reads 0, no traffic
  float acc = 0.0f;
#pragma unroll
  for (int d = 0; d < kFD; d++) {
#pragma unroll
    for (int t = 0; t < 4; t++) loadw(d, d, t);
    loadx(d, d);
    __builtin_amdgcn_sched_barrier(0);      // groups arrive in order: a wait for one leaves the later ones in flight
  }
  int g0 = 0;
  // The products of a tile are formed during the sums of the one before it; a
  // group's registers take group g + kFD as their tiles' products are formed.
  float4 p = f_products<0>(w[0][0], xv[0]);
  for (; g0 + kFD < ng; g0 += kFD) {        // whole rounds: no branch inside, so the waits name only the loads in use
#pragma unroll
    for (int d = 0; d < kFD; d++) {
      const int g = g0 + d + kFD, e = (d + 1) % kFD;
      float4 q;
      f_sum(acc, p, [&](int i) {
        if (i == 0) q.x = f_dpp<0x55>(xv[d].x) * w[d][1].x;
        if (i == 1) q.y = f_dpp<0x55>(xv[d].y) * w[d][1].y;
        if (i == 2) q.z = f_dpp<0x55>(xv[d].z) * w[d][1].z;
        if (i == 3) q.w = f_dpp<0x55>(xv[d].w) * w[d][1].w;
      });
      f_sum(acc, q, [&](int i) {
        if (i == 1) loadw(d, g, 0);
        if (i == 0) p.x = f_dpp<0xaa>(xv[d].x) * w[d][2].x;
        if (i == 1) p.y = f_dpp<0xaa>(xv[d].y) * w[d][2].y;
        if (i == 2) p.z = f_dpp<0xaa>(xv[d].z) * w[d][2].z;
        if (i == 3) p.w = f_dpp<0xaa>(xv[d].w) * w[d][2].w;
      });
      f_sum(acc, p, [&](int i) {
        if (i == 1) loadw(d, g, 1);
        if (i == 0) q.x = f_dpp<0xff>(xv[d].x) * w[d][3].x;
        if (i == 1) q.y = f_dpp<0xff>(xv[d].y) * w[d][3].y;
        if (i == 2) q.z = f_dpp<0xff>(xv[d].z) * w[d][3].z;
        if (i == 3) q.w = f_dpp<0xff>(xv[d].w) * w[d][3].w;
      });
      f_sum(acc, q, [&](int i) {
        if (i == 1) loadw(d, g, 2);
        if (i == 2) loadw(d, g, 3);
        if (i == 3) loadx(d, g);
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
    for (int t = 0; t < 4; t++) wt[t] = f_load16(rw, vw + t * kFTile * 4, 4 * ng * kFTile * 4);
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
// forward.  Every output element is one serial chain in k order, the
// reference's, with each product rounded before its add.  A 64 x 64 block tile
// gives each of 256 threads 4 rows x 4 columns, 16 independent chains; K is
// staged kKT rows at a time through LDS (A transposed to [k][row], W from the
// block's four panels as [k][column]), and the next stage's global loads are in
// flight while the current one is summed.  A chain takes exactly K terms: a
// padded 0 * w term would turn a -0 sum into +0.
// ---------------------------------------------------------------------------
constexpr int kMT = 64;           // rows per block tile
constexpr int kNT = 4 * kFC;      // columns per block tile: four panels
constexpr int kKT = 32;           // k rows per LDS stage
constexpr int kAS = kMT + 4;      // LDS stride of a k row of A
constexpr int kWS = kNT + 4;      // LDS stride of a k row of W

template <int MODE>
__global__ __launch_bounds__(256) void k_gemm_f32(const float *A, int M, int K, const float *W, int N, float *out,
                                                  const float *bias) {
  __shared__ __align__(16) float As[kKT * kAS];
  __shared__ __align__(16) float Ws[kKT * kWS];
  const int tid = threadIdx.x;
  const int i0 = blockIdx.y * kMT, j0 = blockIdx.x * kNT;
  const int np = (N + kFC - 1) / kFC, kt = (K + kFK - 1) / kFK;
  const bool vec = (K & 3) == 0 && (reinterpret_cast<uintptr_t>(A) & 15) == 0;   // whole aligned float4s
  // staging of A: thread -> row ar, k offsets ak .. ak+7 of the stage
  const int ar = tid >> 2, ak = (tid & 3) * 8;
  const bool arow = i0 + ar < M;
  const float *Ar = A + (size_t)(arow ? i0 + ar : 0) * K;
  // staging of W: float4 f = tid + 256 g is panel f / 128, tile (f % 128) / 64, lane part f % 64 of the tile
  float av[8];
  float4 wv[2];
  auto gload = [&](int k0) {
    if (vec) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int k = k0 + ak + 4 * h;
        const float4 v = arow && k < K ? *reinterpret_cast<const float4 *>(Ar + k) : make_float4(0.f, 0.f, 0.f, 0.f);
        av[4 * h] = v.x; av[4 * h + 1] = v.y; av[4 * h + 2] = v.z; av[4 * h + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) av[e] = arow && k0 + ak + e < K ? Ar[k0 + ak + e] : 0.0f;
    }
#pragma unroll
    for (int g = 0; g < 2; g++) {
      const int f = tid + 256 * g, p = blockIdx.x * 4 + (f >> 7), t = k0 / kFK + ((f >> 6) & 1);
      wv[g] = p < np && t < kt ? *reinterpret_cast<const float4 *>(W + ((size_t)p * kt + t) * kFTile + (f & 63) * 4)
                               : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  const int ty = tid >> 4, tx = tid & 15;
  float acc[4][4];
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[r][c] = 0.0f;
  gload(0);
  for (int k0 = 0; k0 < K; k0 += kKT) {
    __syncthreads();                              // the previous stage is summed
#pragma unroll
    for (int e = 0; e < 8; e++) As[(ak + e) * kAS + ar] = av[e];
#pragma unroll
    for (int g = 0; g < 2; g++) {
      const int f = tid + 256 * g;
      const int l = f & 63, k = ((f >> 6) & 1) * kFK + 4 * ((l >> 2) & 3), j = (f >> 7) * kFC + 4 * (l >> 4) + (l & 3);
      Ws[k * kWS + j] = wv[g].x;
      Ws[(k + 1) * kWS + j] = wv[g].y;
      Ws[(k + 2) * kWS + j] = wv[g].z;
      Ws[(k + 3) * kWS + j] = wv[g].w;
    }
    __syncthreads();
    if (k0 + kKT < K) gload(k0 + kKT);
    const int kn = min(kKT, K - k0);
    auto step = [&](int kk) {
      const float4 a = *reinterpret_cast<const float4 *>(&As[kk * kAS + ty * 4]);
      const float4 w = *reinterpret_cast<const float4 *>(&Ws[kk * kWS + tx * 4]);
      const float ar4[4] = {a.x, a.y, a.z, a.w}, wr4[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[r][c] = acc[r][c] + ar4[r] * wr4[c];
    };
    if (kn == kKT) {
#pragma unroll 8
      for (int kk = 0; kk < kKT; kk++) step(kk);
    } else {
      for (int kk = 0; kk < kn; kk++) step(kk);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int i = i0 + ty * 4 + r;
    if (i >= M) continue;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int j = j0 + tx * 4 + c;
      if (j >= N) continue;
      float *o = out + (size_t)i * N + j;
      if (MODE == FMODE_RESID) *o = *o + acc[r][c];
      else *o = bias ? acc[r][c] + bias[j] : acc[r][c];
    }
  }
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

extern "C" int qhip_gemm_f32(int mode, int cls, const float *A, int M, int K, const float *W, int N, float *out,
                             const float *bias) {
  if (M <= 0 || K <= 0 || N <= 0 || M > 65535 * kMT) return qh::fail_msg("gemm_f32: bad shape");
  const dim3 grid((N + kNT - 1) / kNT, (M + kMT - 1) / kMT);
  if (mode == 0) QH_LAUNCH(cls, k_gemm_f32<FMODE_PLAIN>, grid, dim3(256), 0, A, M, K, W, N, out, bias);
  else if (mode == 1) QH_LAUNCH(cls, k_gemm_f32<FMODE_RESID>, grid, dim3(256), 0, A, M, K, W, N, out, bias);
  else return qh::fail_msg("gemm_f32: bad mode");
  return 0;
}
