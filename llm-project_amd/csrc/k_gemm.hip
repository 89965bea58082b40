// k_gemm.hip - int8 MFMA GEMM for prompt ingestion: quant.c:60-85 over many
// activation rows at once (qmatmul with M = the prompt length).
//
// C[i][j] = (as[i] * ws[j]) * (float)acc[i][j],  acc = sum_k qa[i][k] * W[j][k]
//
// acc is an exact int32 sum (|acc| <= 127^2 * K < 2^31), so the MFMA order of
// accumulation changes nothing: every row equals the decode GEMV's result, and
// the epilogues below are the decode GEMV's, operation for operation:
//   PLAIN  out = c (+ bias)                              (llama.c:546-548)
//   RESID  out = out + c                                 (llama.c:578, 589)
//   SWIGLU gate j and up j -> h = (g * (1 / (1 + expf(-g)))) * u  (llama.c:583-587)
//
// Operands are K-contiguous (activation rows [M][kpad], weight rows [N][kpad]).
// Three kernels (launch() chooses):
//  - k_gemm_i8_deep (kpad % 128 == 0): block tiles of 256 x 256, 256 x 128 or 128 x 128
//    (SWIGLU: half the columns are gate rows, half the matching up rows) in K steps
//    of 128 bytes, v_mfma_i32_32x32x32_i8 (the 16x16x64 form runs at half its rate on
//    gfx950).  Both operand tiles are copied straight from global memory into LDS
//    (global_load_lds, no staging registers), two to four K steps in LDS.
//  - k_gemm_i8_pipe (kpad % 64 == 0): 128 x 128 or 256 x 128 tiles, K steps of 64
//    bytes, 8 waves, four or three steps in LDS.
//  - k_gemm_i8 (other K): 128 x 128 tiles staged through registers into
//    double-buffered LDS, 4 waves of 4 x 4 v_mfma_i32_16x16x64_i8; chunks past
//    kpad are zero.
// Fragment layouts (checked on gfx950): 16x16x64: lane l holds row l % 16 and
// bytes 16 * (l / 16) .. +15 of the 64 K values, result element r of lane l is
// C[4 * (l / 16) + r][l % 16]; 32x32x32: lane l holds row l % 32 and bytes
// 16 * (l / 32) .. +15 of 32 K values, result element e of lane l is
// C[8 * (e / 4) + 4 * (l / 32) + e % 4][l % 32].
#include <hip/hip_runtime.h>

#include <type_traits>

#include "qdev_math.h"
#include "qhip.h"
#include "qhip_internal.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

enum { GM_PLAIN = 0, GM_RESID = 1, GM_SWIGLU = 2 };

constexpr int BM = 128, BN = 128, BK = 64;

// Byte offset of 16-byte chunk c of staged row r: rows are 64 bytes, and the
// chunk index is XORed with bits 1-2 of the row, so that the 16-byte accesses of
// 16 consecutive rows (a fragment read) and of 4 consecutive rows x 4 chunks
// (a staging write) fall in distinct bank groups.
__device__ __forceinline__ int stage_off(int r, int c) { return r * BK + ((c ^ ((r >> 1) & 3)) << 4); }

// Block b -> (M tile, N tile): the row tiles of one weight tile run on one XCD
// (workgroups are dealt to the 8 XCDs round-robin by index), so a weight tile
// is fetched from HBM once and then served from that XCD's L2.
__device__ __forceinline__ void gemm_tile(int b, int mt_count, int &mt, int &nt) {
  const int x8 = b & 7, q = b >> 3;
  mt = q % mt_count;
  nt = 8 * (q / mt_count) + x8;
}

template <int MODE>
__global__ __launch_bounds__(256) void k_gemm_i8(const int8_t *A, const float *as, const int8_t *W, const float *ws,
                                                 int M, int N, int kpad, float *out, int ldo, const float *bias,
                                                 int mt_count, int nt_count) {
  __shared__ __attribute__((aligned(16))) int8_t sA[2][BM * BK];
  __shared__ __attribute__((aligned(16))) int8_t sB[2][BN * BK];
  int mtile, ntile;
  gemm_tile(blockIdx.x, mt_count, mtile, ntile);
  if (ntile >= nt_count) return;                                   // uniform for the block
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = mtile * BM;
  constexpr int NOUT = MODE == GM_SWIGLU ? BN / 2 : BN;
  const int n0 = ntile * NOUT;

  // global -> LDS: each operand tile is 512 chunks of 16 bytes; thread tid moves
  // chunks tid and tid + 256 (row = chunk / 4, part = chunk % 4)
  const int8_t *ga[2], *gb[2];
  int soff[2], part[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int c = tid + 256 * i, row = c >> 2;
    part[i] = c & 3;
    soff[i] = stage_off(row, part[i]);
    ga[i] = A + (size_t)min(m0 + row, M - 1) * kpad + part[i] * 16;
    int wrow;
    if (MODE == GM_SWIGLU) wrow = row < 64 ? min(n0 + row, N - 1) : N + min(n0 + row - 64, N - 1);
    else wrow = min(n0 + row, N - 1);
    gb[i] = W + (size_t)wrow * kpad + part[i] * 16;
  }
  const int nk = (kpad + BK - 1) / BK;
  v4i ra[2], rb[2];
  auto gload = [&](int kt) {
    const int k0 = kt * BK;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const bool in = k0 + part[i] * 16 < kpad;
      const v4i z = {0, 0, 0, 0};
      ra[i] = in ? *reinterpret_cast<const v4i *>(ga[i] + k0) : z;
      rb[i] = in ? *reinterpret_cast<const v4i *>(gb[i] + k0) : z;
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      *reinterpret_cast<v4i *>(&sA[buf][soff[i]]) = ra[i];
      *reinterpret_cast<v4i *>(&sB[buf][soff[i]]) = rb[i];
    }
  };

  // this lane's fragment rows inside the staged tiles
  int arow[4], brow[4];
#pragma unroll
  for (int t = 0; t < 4; t++) {
    arow[t] = stage_off(wm * 64 + t * 16 + (lane & 15), lane >> 4);
    const int bl = MODE == GM_SWIGLU ? (t < 2 ? wn * 32 + t * 16 : 64 + wn * 32 + (t - 2) * 16) : wn * 64 + t * 16;
    brow[t] = stage_off(bl + (lane & 15), lane >> 4);
  }

  v4i acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; a++)
#pragma unroll
    for (int b = 0; b < 4; b++) acc[a][b] = (v4i){0, 0, 0, 0};

  gload(0);
  sstore(0);
  __syncthreads();
  for (int kt = 0; kt < nk; kt++) {
    const int buf = kt & 1;
    if (kt + 1 < nk) gload(kt + 1);
    v4i fa[4], fb[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      fa[t] = *reinterpret_cast<const v4i *>(&sA[buf][arow[t]]);
      fb[t] = *reinterpret_cast<const v4i *>(&sB[buf][brow[t]]);
    }
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[a], fb[b], acc[a][b], 0, 0, 0);
    if (kt + 1 < nk) sstore(buf ^ 1);
    __syncthreads();
  }

  // epilogue (the decode GEMV's operations and order)
#pragma unroll
  for (int a = 0; a < 4; a++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = m0 + wm * 64 + a * 16 + 4 * (lane >> 4) + r;
      if (i >= M) continue;
      const float asi = as[i];
      if (MODE == GM_SWIGLU) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
          const int j = n0 + wn * 32 + b * 16 + (lane & 15);
          if (j < N) {
            const float g = (asi * ws[j]) * (float)acc[a][b][r];
            const float up = (asi * ws[N + j]) * (float)acc[a][b + 2][r];
            const float s = 1.0f / (1.0f + qd::expf_glibc(-g));
            out[(size_t)i * ldo + j] = (g * s) * up;
          }
        }
      } else {
#pragma unroll
        for (int b = 0; b < 4; b++) {
          const int j = n0 + wn * 64 + b * 16 + (lane & 15);
          if (j < N) {
            const float c = (asi * ws[j]) * (float)acc[a][b][r];
            float *o = out + (size_t)i * ldo + j;
            if (MODE == GM_RESID) *o = *o + c;
            else *o = bias ? c + bias[j] : c;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Pipelined variant for kpad % 64 == 0: the same tiles, fragments and epilogues,
// but both operand tiles go straight from global memory into LDS
// (global_load_lds, 16 bytes per lane, no staging registers), NSTAGE K steps
// deep.  Wave instruction i of a tile fills LDS slots 64i .. 64i+63 of 16 bytes;
// slot s holds chunk (s % 4) ^ ((r >> 1) % 4) of row r = s / 4, i.e. the lane
// fetches the global chunk that the swizzled layout puts there.  The waits
// before each step's barrier name only the step's own loads (vmcnt of the
// later stages stay in flight); the barrier itself is s_barrier without a
// fence, which would drain every outstanding load.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void *lds_ptr_t;

// Staged layout of the pipelined kernel: 64-byte rows, 16-byte chunk c of row r
// at slot c ^ swz32(r).  The fragment reads of v_mfma_i32_32x32x32_i8 take one
// chunk of 32 consecutive rows per half-wave.  XOR with row bits 2-3 makes those
// 16-byte reads conflict-free on gfx950 (measured with SQ_LDS_BANK_CONFLICT on
// this access pattern: bits 2-3 or 3-4, or 80-byte rows, 0 conflict cycles;
// bits 1-2, or bits 1^3 and 2^4, half of the LDS cycles; bits 0-1 or none,
// three quarters).  The staging writes fill whole 1 KiB runs and never conflict.
__device__ __forceinline__ int swz32(int r) { return (r >> 2) & 3; }
__device__ __forceinline__ int stage_off32(int r, int c) { return r * BK + ((c ^ swz32(r)) << 4); }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

__device__ __forceinline__ void block_sync_lds() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// What a block's epilogue reads besides the sums, requested before its K loop: the
// scales of its TM rows and (SwiGLU) the exp table in LDS, and a lane's column
// scales and biases in registers.  (Read element by element between the stores,
// which the compiler has to keep in order, they cost a memory round trip each: 28 of
// 82 us of the QKV product at 2048 rows, 91 of 300 of gate|up.)
template <int TM>
struct EpiShared {
  __attribute__((aligned(16))) float as[TM];
  uint64_t tab[32];
};

template <int MODE>
struct EpiLane {
  int j[2];            // output columns of the two column blocks (SwiGLU: one, its gate and up scales in w)
  float w[2], b[2];
};

// All threads.  The K loop's barriers are bare (no fence), so the LDS part is readable
// by the block's other waves behind the first barrier that a wave reaches with its LDS
// writes landed: k_gemm_i8_pipe waits for them before its first barrier (epi_publish;
// after a single K step there is no other), k_gemm_i8_deep in the phase between its
// first barrier and the loop's, whose wait is lgkmcnt(0) (a wait before the first one
// as well cost 0.45 of 46.5 us at 1000 x 4096 x 6144).
template <int MODE, int TM, int NT>
__device__ __forceinline__ EpiLane<MODE> epi_begin(EpiShared<TM> &sh, const float *as, const float *ws,
                                                   const float *bias, int M, int N, int m0, int n0, int wn, int lane) {
  for (int r = threadIdx.x; r < TM; r += NT) sh.as[r] = as[min(m0 + r, M - 1)];
  if (MODE == GM_SWIGLU && threadIdx.x < 32) sh.tab[threadIdx.x] = qd::kExp2Tab[threadIdx.x];
  EpiLane<MODE> l;
  if (MODE == GM_SWIGLU) {
    l.j[0] = l.j[1] = n0 + wn * 32 + (lane & 31);
    l.w[0] = ws[min(l.j[0], N - 1)];
    l.w[1] = ws[N + min(l.j[0], N - 1)];
    l.b[0] = l.b[1] = 0.0f;
  } else {
#pragma unroll
    for (int b = 0; b < 2; b++) {
      l.j[b] = n0 + wn * 64 + b * 32 + (lane & 31);
      l.w[b] = ws[min(l.j[b], N - 1)];
      l.b[b] = MODE == GM_PLAIN && bias ? bias[min(l.j[b], N - 1)] : 0.0f;
    }
  }
  return l;
}

__device__ __forceinline__ void epi_publish() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The wave's sums to the output: result element e of row block a is row i0 + 32 a +
// 8 (e / 4) + 4 (lane / 32) + e % 4, i0 = r0 rows into the block's m0.  FULL: every
// row and column of the block exists.  The decode GEMV's operations and order.
template <int MODE, int RB, int TM, bool FULL>
__device__ __forceinline__ void epi_store(const v16i (&acc)[RB][2], const EpiShared<TM> &sh, const EpiLane<MODE> &l,
                                          bool has_bias, int M, int N, float *__restrict__ out, int ldo, int m0,
                                          int r0, int lane) {
  const int rl = r0 + 4 * (lane >> 5);
  auto row = [&](int a, int e) { return 32 * a + 8 * (e >> 2) + (e & 3); };      // from row m0 + rl
  float *o0 = out + (size_t)(m0 + rl) * ldo + l.j[0];
  const int step = l.j[1] - l.j[0];                                              // 32 (SwiGLU: 0)
  float old[2][MODE == GM_RESID ? 16 : 1][2];
  auto fetch = [&](int a) __attribute__((always_inline)) {
    if constexpr (MODE == GM_RESID) {
#pragma unroll
      for (int e = 0; e < 16; e++)
#pragma unroll
        for (int b = 0; b < 2; b++)
          old[a & 1][e][b] = FULL || (m0 + rl + row(a, e) < M && l.j[b] < N) ? o0[(size_t)row(a, e) * ldo + b * step] : 0.0f;
    }
  };
  fetch(0);
#pragma unroll
  for (int a = 0; a < RB; a++) {
    if (a + 1 < RB) fetch(a + 1);                    // requested before this block's stores
    float s[16];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float4 t = *reinterpret_cast<const float4 *>(&sh.as[rl + 32 * a + 8 * q]);
      s[4 * q] = t.x; s[4 * q + 1] = t.y; s[4 * q + 2] = t.z; s[4 * q + 3] = t.w;
    }
    if constexpr (MODE == GM_SWIGLU) {
#pragma unroll
      for (int h = 0; h < 16; h += 8) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = -((s[h + e] * l.w[0]) * (float)acc[a][0][h + e]);
        float g[8];
#pragma unroll
        for (int e = 0; e < 8; e++) g[e] = -x[e];
        qd::expf_glibc_n<8>(x, sh.tab);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float up = (s[h + e] * l.w[1]) * (float)acc[a][1][h + e];
          const float sg = 1.0f / (1.0f + x[e]);
          if (FULL || (m0 + rl + row(a, h + e) < M && l.j[0] < N)) o0[(size_t)row(a, h + e) * ldo] = (g[e] * sg) * up;
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 16; e++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
          const float c = (s[e] * l.w[b]) * (float)acc[a][b][e];
          float v;
          if constexpr (MODE == GM_RESID) v = old[a & 1][e][b] + c;
          else v = has_bias ? c + l.b[b] : c;
          if (FULL || (m0 + rl + row(a, e) < M && l.j[b] < N)) o0[(size_t)row(a, e) * ldo + b * step] = v;
        }
    }
  }
}

// int32 partial sums of K split `split` to part[split][M][N] (SwiGLU: [split][M][2N], up
// columns at N + j).
template <int MODE, int RB>
__device__ __forceinline__ void epi_part(const v16i (&acc)[RB][2], const EpiLane<MODE> &l, int M, int N, int *part,
                                         int split, int i0, int lane) {
  const int ldp = MODE == GM_SWIGLU ? 2 * N : N;
  int *pp = part + (size_t)split * M * ldp;
#pragma unroll
  for (int a = 0; a < RB; a++) {
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int i = i0 + a * 32 + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
      if (i >= M) continue;
#pragma unroll
      for (int b = 0; b < 2; b++)
        if (l.j[b] < N) pp[(size_t)i * ldp + (MODE == GM_SWIGLU && b ? N : 0) + l.j[b]] = acc[a][b][e];
    }
  }
}

template <int MODE, int RB, int TM>
__device__ __forceinline__ void epi_end(const v16i (&acc)[RB][2], const EpiShared<TM> &sh, const EpiLane<MODE> &l,
                                        bool has_bias, int M, int N, float *out, int ldo, int m0, int n0, int nout,
                                        int r0, int lane) {
  if (m0 + TM <= M && n0 + nout <= N) epi_store<MODE, RB, TM, true>(acc, sh, l, has_bias, M, N, out, ldo, m0, r0, lane);
  else epi_store<MODE, RB, TM, false>(acc, sh, l, has_bias, M, N, out, ldo, m0, r0, lane);
}

// Block tile TM x TN, waves WM x WN, each wave (TM/WM) x (TN/WN) from 32 x 32
// v_mfma_i32_32x32x32_i8 blocks: RB row blocks x 2 column blocks (SWIGLU: the
// wave's 32 gate columns and the matching 32 up columns).
//
// Split K (PART): block b of the grid takes tile b % bps and the K steps
// [split * nks, split * nks + nks) of split b / bps, and stores its int32 partial
// sums to part[split][M][N] (SWIGLU: [split][M][2N], up columns at N + j) for
// k_gemm_split_epi.
template <int MODE, int TM, int TN, int WM, int WN, int NSTAGE, bool PART = false>
__global__ __launch_bounds__(64 * WM * WN) void k_gemm_i8_pipe(const int8_t *A, const float *as, const int8_t *W,
                                                              const float *ws, int M, int N, int kpad, float *out,
                                                              int ldo, const float *bias, int mt_count, int nt_count,
                                                              int bps, int nks, int *part) {
  static_assert(NSTAGE == 3 || NSTAGE == 4, "pipeline depth");
  constexpr int NWAVE = WM * WN, RB = TM / WM / 32;
  static_assert(TN == 64 * WN, "two 32-column blocks per wave");
  static_assert(TM % (16 * NWAVE) == 0 && TN % (16 * NWAVE) == 0, "whole wave instructions per tile");
  constexpr int LA = TM / 16 / NWAVE, LB = TN / 16 / NWAVE;        // 1 KiB copies per wave and stage
  constexpr int LPS = LA + LB;                                       // vmcnt per stage
  // one LDS buffer per stage and operand, as distinct variables: the compiler
  // then knows which copies in flight write which buffer
  __shared__ __attribute__((aligned(16))) int8_t sA0[TM * BK], sA1[TM * BK], sA2[TM * BK], sA3[NSTAGE > 3 ? TM * BK : 16];
  __shared__ __attribute__((aligned(16))) int8_t sB0[TN * BK], sB1[TN * BK], sB2[TN * BK], sB3[NSTAGE > 3 ? TN * BK : 16];
  int mtile, ntile;
  const int split = PART ? (int)blockIdx.x / bps : 0;
  gemm_tile(PART ? (int)blockIdx.x % bps : (int)blockIdx.x, mt_count, mtile, ntile);
  if (ntile >= nt_count) return;                                   // uniform for the block
  const int kt0 = split * nks;                                     // first K step of this block
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = mtile * TM;
  constexpr int NOUT = MODE == GM_SWIGLU ? TN / 2 : TN;
  const int n0 = ntile * NOUT;
  __shared__ EpiShared<TM> epi;
  const EpiLane<MODE> el = epi_begin<MODE, TM, 64 * NWAVE>(epi, as, ws, bias, M, N, m0, n0, wn, lane);

  // this lane's global chunks: wave instructions wave*LA + i of the A tile and
  // wave*LB + i of the B tile
  const int8_t *ga[LA], *gb[LB];
#pragma unroll
  for (int i = 0; i < LA; i++) {
    const int slot = (wave * LA + i) * 64 + lane, row = slot >> 2;
    const int c = (slot & 3) ^ swz32(row);
    ga[i] = A + (size_t)min(m0 + row, M - 1) * kpad + c * 16 + (size_t)kt0 * BK;
  }
#pragma unroll
  for (int i = 0; i < LB; i++) {
    const int slot = (wave * LB + i) * 64 + lane, row = slot >> 2;
    const int c = (slot & 3) ^ swz32(row);
    int wrow;
    if (MODE == GM_SWIGLU) wrow = row < TN / 2 ? min(n0 + row, N - 1) : N + min(n0 + row - TN / 2, N - 1);
    else wrow = min(n0 + row, N - 1);
    gb[i] = W + (size_t)wrow * kpad + c * 16 + (size_t)kt0 * BK;
  }
  const int nk = PART ? min(nks, kpad / BK - kt0) : kpad / BK;
  auto bufA = [&](auto st) -> int8_t * {
    if constexpr (decltype(st)::value == 0) return sA0;
    else if constexpr (decltype(st)::value == 1) return sA1;
    else if constexpr (decltype(st)::value == 2) return sA2;
    else return sA3;
  };
  auto bufB = [&](auto st) -> int8_t * {
    if constexpr (decltype(st)::value == 0) return sB0;
    else if constexpr (decltype(st)::value == 1) return sB1;
    else if constexpr (decltype(st)::value == 2) return sB2;
    else return sB3;
  };
  auto issue = [&](auto st, int kt) {
    const int k0 = kt * BK;
    int8_t *da = bufA(st), *db = bufB(st);
#pragma unroll
    for (int i = 0; i < LA; i++)
      __builtin_amdgcn_global_load_lds((const void *)(ga[i] + k0), (lds_ptr_t)(da + (wave * LA + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < LB; i++)
      __builtin_amdgcn_global_load_lds((const void *)(gb[i] + k0), (lds_ptr_t)(db + (wave * LB + i) * 1024), 16, 0, 0);
  };

  // fragments of v_mfma_i32_32x32x32_i8: lane l supplies row l % 32 and bytes
  // 16 * (l / 32) .. +15 of a 32-byte K half, i.e. chunk 2 * kh + l / 32 of the
  // 64-byte staged row; result element e of lane l is
  // C[8 * (e / 4) + 4 * (l / 32) + e % 4][l % 32] (checked on gfx950)
  int arow[RB][2], brow[2][2];
#pragma unroll
  for (int kh = 0; kh < 2; kh++) {
#pragma unroll
    for (int t = 0; t < RB; t++) arow[t][kh] = stage_off32(wm * (TM / WM) + t * 32 + (lane & 31), 2 * kh + (lane >> 5));
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int bl = MODE == GM_SWIGLU ? t * (TN / 2) + wn * 32 : wn * 64 + t * 32;
      brow[t][kh] = stage_off32(bl + (lane & 31), 2 * kh + (lane >> 5));
    }
  }

  v16i acc[RB][2];
#pragma unroll
  for (int a = 0; a < RB; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = (v16i){};

  // step kt from stage ST: wait for its copies, barrier, refill stage ST-1 with
  // step kt + NSTAGE - 1, multiply
  auto step = [&](auto st, int kt) {
    constexpr int ST = decltype(st)::value;
    const int later = min(NSTAGE - 2, nk - 1 - kt);      // steps issued after kt
    if (later >= NSTAGE - 2) wait_vmcnt<LPS * (NSTAGE - 2)>();
    else if (NSTAGE > 3 && later == 1) wait_vmcnt<LPS>();
    else wait_vmcnt<0>();
    block_sync_lds();                   // every wave's copies of step kt have landed; step kt-1 is consumed
    if (kt + NSTAGE - 1 < nk) issue(std::integral_constant<int, (ST + NSTAGE - 1) % NSTAGE>(), kt + NSTAGE - 1);
    // fragment reads in asm, with their own waits: the compiler would otherwise
    // wait for every copy in flight before reading an LDS buffer it cannot
    // tell apart from the ones being filled
    const unsigned la = (unsigned)(uintptr_t)bufA(st), lb = (unsigned)(uintptr_t)bufB(st);
    v4i fa[RB][2], fb[2][2];
#pragma unroll
    for (int kh = 0; kh < 2; kh++) {
#pragma unroll
      for (int t = 0; t < 2; t++) asm volatile("ds_read_b128 %0, %1" : "=v"(fb[t][kh]) : "v"(lb + brow[t][kh]));
#pragma unroll
      for (int t = 0; t < RB; t++) asm volatile("ds_read_b128 %0, %1" : "=v"(fa[t][kh]) : "v"(la + arow[t][kh]));
    }
#pragma unroll
    for (int kh = 0; kh < 2; kh++) {
      // the kh = 0 fragments are the first 2 + RB reads issued
      if (kh == 0) __builtin_amdgcn_s_waitcnt(0xC07F | ((2 + RB) << 8));
      else __builtin_amdgcn_s_waitcnt(0xC07F);
#pragma unroll
      for (int t = 0; t < 2; t++) asm volatile("" : "+v"(fb[t][kh]));
#pragma unroll
      for (int t = 0; t < RB; t++) asm volatile("" : "+v"(fa[t][kh]));
#pragma unroll
      for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
          acc[a][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[a][kh], fb[b][kh], acc[a][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);   // the kh = 0 products go before the wait for the kh = 1 reads
    }
  };

  issue(std::integral_constant<int, 0>(), 0);
  if (1 < nk) issue(std::integral_constant<int, 1>(), 1);
  if (NSTAGE > 3 && 2 < nk) issue(std::integral_constant<int, (NSTAGE > 3 ? 2 : 0)>(), 2);
  epi_publish();
  for (int kt = 0; kt < nk; kt += NSTAGE) {
    step(std::integral_constant<int, 0>(), kt);
    if (kt + 1 < nk) step(std::integral_constant<int, 1>(), kt + 1);
    if (kt + 2 < nk) step(std::integral_constant<int, 2>(), kt + 2);
    if (NSTAGE > 3 && kt + 3 < nk) step(std::integral_constant<int, (NSTAGE > 3 ? 3 : 0)>(), kt + 3);
  }

  if constexpr (PART) epi_part<MODE, RB>(acc, el, M, N, part, split, m0 + wm * (TM / WM), lane);
  else epi_end<MODE, RB, TM>(acc, epi, el, bias != nullptr, M, N, out, ldo, m0, n0, NOUT, wm * (TM / WM), lane);
}

constexpr int kMaxSplits = 16;         // K splits of one GEMM at most

// Split-K epilogue: acc = the sum of the S int32 partials (exact in any order:
// every partial sum of the products is bounded like the whole, |acc| <= 127^2 K),
// then the fused epilogue's operations on it.  Grid (ceil(N / 256), M).
template <int MODE>
__global__ __launch_bounds__(256) void k_gemm_split_epi(const int *part, int S, const float *as, const float *ws,
                                                        int M, int N, float *out, int ldo, const float *bias) {
  const int j = blockIdx.x * 256 + threadIdx.x, i = blockIdx.y;
  if (j >= N) return;
  const int ldp = MODE == GM_SWIGLU ? 2 * N : N;
  const size_t plane = (size_t)M * ldp;
  const int *pp = part + (size_t)i * ldp + j;
  // every partial requested before the first add (S <= kMaxSplits)
  int pv[kMaxSplits], pu[kMaxSplits];
#pragma unroll
  for (int s = 0; s < kMaxSplits; s++) {
    pv[s] = s < S ? pp[s * plane] : 0;
    pu[s] = MODE == GM_SWIGLU && s < S ? pp[s * plane + N] : 0;
  }
  int acc = 0, accu = 0;
#pragma unroll
  for (int s = 0; s < kMaxSplits; s++) {
    acc += pv[s];
    accu += pu[s];
  }
  const float asi = as[i];
  if (MODE == GM_SWIGLU) {
    const float g = (asi * ws[j]) * (float)acc;
    const float up = (asi * ws[N + j]) * (float)accu;
    const float sg = 1.0f / (1.0f + qd::expf_glibc(-g));
    out[(size_t)i * ldo + j] = (g * sg) * up;
  } else {
    const float c = (asi * ws[j]) * (float)acc;
    float *o = out + (size_t)i * ldo + j;
    if (MODE == GM_RESID) *o = *o + c;
    else *o = bias ? c + bias[j] : c;
  }
}

// Tiles that leave CUs idle (a short prompt, a narrow output) split K when the
// caller lends a workspace: S splits of at least 8 K steps, so that tiles x S
// reach one block per CU, with S partial planes of M x N int32 in the workspace.
int g_last_splits = 1;                 // K splits of the last pipelined launch (for the split test)

template <int MODE, int TM, int TN, int WM, int WN, int NS>
int launch_pipe(const int8_t *A, const float *as, const int8_t *W, const float *ws, int M, int N, int kpad, float *out,
                int ldo, const float *bias, int cls, int *work, size_t work_bytes) {
  const int nout = MODE == GM_SWIGLU ? TN / 2 : TN;
  const int mt = (M + TM - 1) / TM, nt = (N + nout - 1) / nout;
  const int blocks = 8 * mt * ((nt + 7) / 8);
  const int nkt = kpad / BK;
  int S = 1;
  if (TM == 128 && work) {               // (the larger tile is taken only where it fills the CUs)
    const int cus = qh::num_cus() > 0 ? qh::num_cus() : 256, active = mt * nt;
    if (active < cus) {
      S = min(min((cus + active - 1) / active, nkt / 8), kMaxSplits);
      const size_t plane = (size_t)M * (MODE == GM_SWIGLU ? 2 * N : N) * 4;
      while (S > 1 && (size_t)S * plane > work_bytes) S--;
    }
  }
  g_last_splits = S < 2 ? 1 : S;
  if (S < 2) {
    QH_LAUNCH(cls, (k_gemm_i8_pipe<MODE, TM, TN, WM, WN, NS>), dim3(blocks), dim3(64 * WM * WN), 0, A, as, W, ws, M,
              N, kpad, out, ldo, bias, mt, nt, blocks, nkt, static_cast<int *>(nullptr));
    return 0;
  }
  if constexpr (TM == 128) {
    const int nks = (nkt + S - 1) / S;
    S = (nkt + nks - 1) / nks;                                     // every split has steps
    g_last_splits = S;
    QH_LAUNCH(cls, (k_gemm_i8_pipe<MODE, TM, TN, WM, WN, NS, true>), dim3(blocks * S), dim3(64 * WM * WN), 0, A, as,
              W, ws, M, N, kpad, out, ldo, bias, mt, nt, blocks, nks, work);
    QH_LAUNCH(cls, k_gemm_split_epi<MODE>, dim3((N + 255) / 256, M), dim3(256), 0, work, S, as, ws, M, N, out, ldo,
              bias);
  }
  return 0;
}

// ---------------------------------------------------------------------------
// Deep variant for kpad % 128 == 0 and many rows: K steps of 128 bytes, so that a
// copy instruction moves eight whole 128-byte lines (64-byte rows cost the cache a
// line each for half its bytes), and a loop whose LDS reads, copies and products
// overlap by construction.  Staged rows are 128 bytes, 16-byte chunk c of row r at
// slot c ^ ((r >> 1) & 7): 16 consecutive rows read at one c fall in distinct banks.
//
// A step is four phases of 32 K bytes.  A phase reads the next phase's fragments
// while it multiplies its own (2 * RB products) and ends when they have arrived:
// one asm block, so that no register holds a load in flight outside it.  The one
// barrier of a step sits before its last phase: every wave has then read all of the
// step's fragments, so its buffer takes the copies of step + NS, and the copies of
// the next step, issued NS - 1 steps ago, have landed for the reads of that phase.
// Limit: the compiler's hazard recognizer does not see the products inside the asm
// blocks.  The blocks read the sums only as accumulators, each last written three or
// more products before, and the s_nops behind the loop cover the last ones; but nothing
// else may read or move the sums between two blocks: no operation on acc there, and no
// spill or copy of it (none in the assembly between the first product and the s_nops,
// in any form; the residual 256 x 256 one spills 24 registers in its epilogue).
// ---------------------------------------------------------------------------
constexpr int DK = 128;

__device__ __forceinline__ int swz_deep(int r) { return (r >> 1) & 7; }

#define DP_RD(dst, base, off) "ds_read_b128 %[" dst "], %[" base "] offset:" off "\n\t"
#define DP_MM(c, a, b) "v_mfma_i32_32x32x32_i8 %[" c "], %[" a "], %[" b "], %[" c "]\n\t"

// acc += fragments (fa, fb); (na, nb) = the fragments at LDS addresses la, lb (row
// blocks 4096 bytes apart, the second column block BOFF bytes on).
template <int BOFF>
__device__ __forceinline__ void gemm_phase(v16i (&acc)[4][2], const v4i (&fa)[4], const v4i (&fb)[2], v4i (&na)[4],
                                           v4i (&nb)[2], unsigned la, unsigned lb) {
  asm volatile(
      DP_RD("nb0", "lb", "0") DP_RD("na0", "la", "0") DP_MM("c00", "a0", "b0")
      DP_RD("nb1", "lb", "%[bo]") DP_MM("c01", "a0", "b1")
      DP_RD("na1", "la", "4096") DP_MM("c10", "a1", "b0")
      DP_RD("na2", "la", "8192") DP_MM("c11", "a1", "b1")
      DP_RD("na3", "la", "12288") DP_MM("c20", "a2", "b0")
      DP_MM("c21", "a2", "b1") DP_MM("c30", "a3", "b0") DP_MM("c31", "a3", "b1")
      "s_waitcnt lgkmcnt(0)"
      : [c00] "+v"(acc[0][0]), [c01] "+v"(acc[0][1]), [c10] "+v"(acc[1][0]), [c11] "+v"(acc[1][1]),
        [c20] "+v"(acc[2][0]), [c21] "+v"(acc[2][1]), [c30] "+v"(acc[3][0]), [c31] "+v"(acc[3][1]),
        [na0] "=&v"(na[0]), [na1] "=&v"(na[1]), [na2] "=&v"(na[2]), [na3] "=&v"(na[3]), [nb0] "=&v"(nb[0]),
        [nb1] "=&v"(nb[1])
      : [a0] "v"(fa[0]), [a1] "v"(fa[1]), [a2] "v"(fa[2]), [a3] "v"(fa[3]), [b0] "v"(fb[0]), [b1] "v"(fb[1]),
        [la] "v"(la), [lb] "v"(lb), [bo] "n"(BOFF)
      : "memory");
}

template <int BOFF>
__device__ __forceinline__ void gemm_phase(v16i (&acc)[2][2], const v4i (&fa)[2], const v4i (&fb)[2], v4i (&na)[2],
                                           v4i (&nb)[2], unsigned la, unsigned lb) {
  asm volatile(
      DP_RD("nb0", "lb", "0") DP_RD("na0", "la", "0") DP_MM("c00", "a0", "b0")
      DP_RD("nb1", "lb", "%[bo]") DP_MM("c01", "a0", "b1")
      DP_RD("na1", "la", "4096") DP_MM("c10", "a1", "b0")
      DP_MM("c11", "a1", "b1")
      "s_waitcnt lgkmcnt(0)"
      : [c00] "+v"(acc[0][0]), [c01] "+v"(acc[0][1]), [c10] "+v"(acc[1][0]), [c11] "+v"(acc[1][1]),
        [na0] "=&v"(na[0]), [na1] "=&v"(na[1]), [nb0] "=&v"(nb[0]), [nb1] "=&v"(nb[1])
      : [a0] "v"(fa[0]), [a1] "v"(fa[1]), [b0] "v"(fb[0]), [b1] "v"(fb[1]), [la] "v"(la), [lb] "v"(lb), [bo] "n"(BOFF)
      : "memory");
}
#undef DP_RD
#undef DP_MM

template <int MODE, int TM, int TN, int WM, int WN, int NS, bool PART = false>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_gemm_i8_deep(
    const int8_t *A, const float *as, const int8_t *W, const float *ws, int M, int N, int kpad, float *out, int ldo,
    const float *bias, int mt_count, int nt_count, int bps, int nks, int *part) {
  constexpr int NWAVE = WM * WN, RB = TM / WM / 32;
  static_assert(TN == 64 * WN, "two 32-column blocks per wave");
  static_assert(TM % (8 * NWAVE) == 0 && TN % (8 * NWAVE) == 0, "whole wave instructions per tile");
  constexpr int LA = TM / 8 / NWAVE, LB = TN / 8 / NWAVE, LPS = LA + LB;     // 1 KiB copies per wave and step
  constexpr int STAGE = (TM + TN) * DK;
  constexpr int BOFF = (MODE == GM_SWIGLU ? TN / 2 : 32) * DK;
  __shared__ __attribute__((aligned(1024))) int8_t lds[NS * STAGE];
  int mtile, ntile;
  const int split = PART ? (int)blockIdx.x / bps : 0;              // as in k_gemm_i8_pipe
  gemm_tile(PART ? (int)blockIdx.x % bps : (int)blockIdx.x, mt_count, mtile, ntile);
  if (ntile >= nt_count) return;                                   // uniform for the block
  const int kt0 = split * nks;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = mtile * TM;
  constexpr int NOUT = MODE == GM_SWIGLU ? TN / 2 : TN;
  const int n0 = ntile * NOUT;
  __shared__ EpiShared<TM> epi;
  const EpiLane<MODE> el = epi_begin<MODE, TM, 64 * NWAVE>(epi, as, ws, bias, M, N, m0, n0, wn, lane);

  // this lane's bytes of copy instruction i of each operand: row 8 * (wave * L + i) + lane / 8 of the
  // tile, the chunk that the swizzle puts at slot lane % 8
  const int8_t *ga[LA], *gb[LB];
#pragma unroll
  for (int i = 0; i < LA; i++) {
    const int row = 8 * (wave * LA + i) + (lane >> 3), c = (lane & 7) ^ swz_deep(row);
    ga[i] = A + (size_t)min(m0 + row, M - 1) * kpad + c * 16 + (size_t)kt0 * DK;
  }
#pragma unroll
  for (int i = 0; i < LB; i++) {
    const int row = 8 * (wave * LB + i) + (lane >> 3), c = (lane & 7) ^ swz_deep(row);
    int wrow;
    if (MODE == GM_SWIGLU) wrow = row < TN / 2 ? min(n0 + row, N - 1) : N + min(n0 + row - TN / 2, N - 1);
    else wrow = min(n0 + row, N - 1);
    gb[i] = W + (size_t)wrow * kpad + c * 16 + (size_t)kt0 * DK;
  }
  const int nk = PART ? min(nks, kpad / DK - kt0) : kpad / DK;
  auto issue = [&](int buf, int kt) __attribute__((always_inline)) {
    int8_t *d = lds + buf * STAGE;
    const int k0 = kt * DK;
#pragma unroll
    for (int i = 0; i < LA; i++)
      __builtin_amdgcn_global_load_lds((const void *)(ga[i] + k0), (lds_ptr_t)(d + (wave * LA + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < LB; i++)
      __builtin_amdgcn_global_load_lds((const void *)(gb[i] + k0), (lds_ptr_t)(d + TM * DK + (wave * LB + i) * 1024), 16,
                                       0, 0);
  };
  // LDS addresses of this lane's fragments of phase p in buffer 0: row lane % 32 of the wave's first row
  // (column) block, chunk 2p + lane / 32
  unsigned la[4], lb[4];
  {
    const int ra = wm * (TM / WM) + (lane & 31), rb = (MODE == GM_SWIGLU ? wn * 32 : wn * 64) + (lane & 31);
#pragma unroll
    for (int p = 0; p < 4; p++) {
      la[p] = (unsigned)(uintptr_t)lds + ra * DK + (((2 * p + (lane >> 5)) ^ swz_deep(ra)) << 4);
      lb[p] = (unsigned)(uintptr_t)lds + (TM + rb) * DK + (((2 * p + (lane >> 5)) ^ swz_deep(rb)) << 4);
    }
  }

  v16i acc[RB][2];
#pragma unroll
  for (int a = 0; a < RB; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = (v16i){};
  v4i xa[RB], xb[2], ya[RB], yb[2];

#pragma unroll
  for (int i = 0; i < NS; i++)
    if (i < nk) issue(i, i);
  if (nk >= NS) wait_vmcnt<LPS * (NS - 1)>();
  else wait_vmcnt<0>();
  block_sync_lds();
  // the first fragments: read and waited for in one block (the sums they go into are still zero, and so
  // are the fragments multiplied meanwhile)
#pragma unroll
  for (int a = 0; a < RB; a++) ya[a] = (v4i){};
#pragma unroll
  for (int b = 0; b < 2; b++) yb[b] = (v4i){};
  gemm_phase<BOFF>(acc, ya, yb, xa, xb, la[0], lb[0]);   // its wait also covers epi_begin's LDS writes
  int buf = 0;
  for (int kt = 0; kt < nk; kt++) {
    const unsigned o = buf * STAGE;
    gemm_phase<BOFF>(acc, xa, xb, ya, yb, la[1] + o, lb[1] + o);
    gemm_phase<BOFF>(acc, ya, yb, xa, xb, la[2] + o, lb[2] + o);
    gemm_phase<BOFF>(acc, xa, xb, ya, yb, la[3] + o, lb[3] + o);
    if (kt + NS <= nk) wait_vmcnt<LPS * (NS - 2)>();   // the copies of step kt + 1 (later ones stay in flight)
    else wait_vmcnt<0>();
    block_sync_lds();
    if (kt + NS < nk) issue(buf, kt + NS);
    buf = buf + 1 < NS ? buf + 1 : 0;
    const unsigned n = buf * STAGE;
    gemm_phase<BOFF>(acc, ya, yb, xa, xb, la[0] + n, lb[0] + n);   // after the last step: read, not used
  }
  // the compiler does not see the products' latency inside the asm blocks
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int a = 0; a < RB; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) asm volatile("" : "+v"(acc[a][b]));
  if constexpr (PART) epi_part<MODE, RB>(acc, el, M, N, part, split, m0 + wm * (TM / WM), lane);
  else epi_end<MODE, RB, TM>(acc, epi, el, bias != nullptr, M, N, out, ldo, m0, n0, NOUT, wm * (TM / WM), lane);
}

template <int MODE, int TM, int TN, int WM, int WN, int NS>
int launch_deep(const int8_t *A, const float *as, const int8_t *W, const float *ws, int M, int N, int kpad, float *out,
                int ldo, const float *bias, int cls, int S, int *work) {
  const int nout = MODE == GM_SWIGLU ? TN / 2 : TN;
  const int mt = (M + TM - 1) / TM, nt = (N + nout - 1) / nout, blocks = 8 * mt * ((nt + 7) / 8), nkt = kpad / DK;
  const dim3 block(64 * WM * WN);
  g_last_splits = S;
  if (S < 2) {
    QH_LAUNCH(cls, (k_gemm_i8_deep<MODE, TM, TN, WM, WN, NS>), dim3(blocks), block, 0, A, as, W, ws, M, N, kpad, out,
              ldo, bias, mt, nt, blocks, nkt, static_cast<int *>(nullptr));
    return 0;
  }
  if constexpr (NS == 4) {
    const int nks = (nkt + S - 1) / S;
    QH_LAUNCH(cls, (k_gemm_i8_deep<MODE, TM, TN, WM, WN, NS, true>), dim3(blocks * S), block, 0, A, as, W, ws, M, N,
              kpad, out, ldo, bias, mt, nt, blocks, nks, work);
    QH_LAUNCH(cls, k_gemm_split_epi<MODE>, dim3((N + 255) / 256, M), dim3(256), 0, work, S, as, ws, M, N, out, ldo, bias);
    return 0;
  }
  return qh::fail_msg("gemm_i8: this tile does not split K");
}

// Tile choice for kpad % 128 == 0, by the time of each in hundredths of a microsecond
// (measured on 2048, 1500, 1000, 512, 333, 200, 100 and 40 rows of the 8B and 1B
// layers' products): a round of blocks takes a fixed part (first copies, epilogue)
// and a part a step of 128 bytes of K,
//   256 x 256, 8 waves, one block a CU                18.0 + 1.35 us a step and round
//   256 x 128, 8 waves, three steps in LDS            15.0 + 0.96
//   128 x 128, 4 waves, two steps in LDS, two a CU     6.0 + 0.50 us a block on its CU
//   128 x 128, four steps in LDS, one a CU             8.0 + 0.49
// the last with K split S ways where the caller lends a workspace (the S partial
// planes written and read at 3 TB/s).  At 2048 rows, us: 8B gate|up 276 317 313
// (256 x 256, 256 x 128, 128 x 128), QKV 61 71 65, Wo 86 52 46, down 189 126 131; 1B
// down at 333 rows unsplit 43, split 5 ways 22.
// kpad % 128 == 64 (steps of 64 bytes): 128 x 128, 8 waves, or for residual and
// SwiGLU, where its tiles fill the CUs and the rounds cost less, 256 x 128,
//   128 x 128, four steps in LDS                       1.65 + 0.35 us a step and round
//   256 x 128, three steps in LDS                      5.60 + 0.54
// us, 128 x 128 and 256 x 128: SwiGLU 2048 x 11008, K 4160 257 234; 800 x 11008, K 4160
// 117 123; 2048 x 4224, K 1600 51 56; 2048 x 5632, K 2112 78 72; residual 2048 x 4096,
// K 8256 105 90; 1500 x 6144, K 8256 138 147.
template <int MODE>
int launch(const int8_t *A, const float *as, const int8_t *W, const float *ws, int M, int N, int kpad, float *out,
           int ldo, const float *bias, int cls, int *work, size_t work_bytes) {
  if (kpad % DK == 0) {
    const int cus = qh::num_cus() > 0 ? qh::num_cus() : 256, st = kpad / DK;
    auto rounds = [&](int tm, int tn) {
      const int nout = MODE == GM_SWIGLU ? tn / 2 : tn;
      const long long tiles = (long long)((M + tm - 1) / tm) * ((N + nout - 1) / nout);
      return (tiles + cus - 1) / cus;
    };
    long long cost = rounds(256, 256) * (1800 + 135 * st);       // hundredths
    int best = 0, S = 1;
    if (const long long c = rounds(256, 128) * (1500 + 96 * st); c < cost) { cost = c; best = 1; }
    const long long n = rounds(128, 128);
    if (n > 1) {
      if (const long long c = n * (600 + 50 * st); c < cost) { cost = c; best = 2; }
    } else {
      const int nout = MODE == GM_SWIGLU ? 64 : 128, tiles = ((M + 127) / 128) * ((N + nout - 1) / nout);
      if (const long long c = 800 + 49 * st; c < cost) { cost = c; best = 3; }
      const size_t plane = (size_t)M * (MODE == GM_SWIGLU ? 2 * N : N) * 4;
      for (int q = 2; work && q <= min(kMaxSplits, st / 4) && tiles * q <= cus && (size_t)q * plane <= work_bytes; q++) {
        const int nks = (st + q - 1) / q;
        if ((st + nks - 1) / nks != q) continue;                 // every split has steps
        const long long c = 800 + 49 * nks + 150 + (long long)((2 * q + 2) * plane / 30000);
        if (c < cost) { cost = c; best = 3; S = q; }
      }
    }
    switch (best) {
      case 0: return launch_deep<MODE, 256, 256, 2, 4, 2>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, 1, nullptr);
      case 1: return launch_deep<MODE, 256, 128, 4, 2, 3>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, 1, nullptr);
      case 2: return launch_deep<MODE, 128, 128, 2, 2, 2>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, 1, nullptr);
      default: return launch_deep<MODE, 128, 128, 2, 2, 4>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, S, work);
    }
  }
  if (kpad % BK == 0) {
    if constexpr (MODE != GM_PLAIN) {
      const int cus = qh::num_cus() > 0 ? qh::num_cus() : 256, st = kpad / BK;
      const long long nt = (N + (MODE == GM_SWIGLU ? 63 : 127)) / (MODE == GM_SWIGLU ? 64 : 128);
      const long long t1 = (M + 127) / 128 * nt, t2 = (M + 255) / 256 * nt;
      if (t2 >= cus && (t2 + cus - 1) / cus * (560 + 54 * st) < (t1 + cus - 1) / cus * (165 + 35 * st))
        return launch_pipe<MODE, 256, 128, 4, 2, 3>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, work, work_bytes);
    }
    return launch_pipe<MODE, 128, 128, 4, 2, 4>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, work, work_bytes);
  }
  const int nout = MODE == GM_SWIGLU ? BN / 2 : BN;
  const int mt = (M + BM - 1) / BM, nt = (N + nout - 1) / nout;
  const int blocks = 8 * mt * ((nt + 7) / 8);
  QH_LAUNCH(cls, k_gemm_i8<MODE>, dim3(blocks), dim3(256), 0, A, as, W, ws, M, N, kpad, out, ldo, bias, mt, nt);
  return 0;
}

}  // namespace

extern "C" int qhip_gemm_i8_ws(int mode, int cls, const int8_t *A, const float *as, const int8_t *W, const float *ws,
                               int M, int N, int kpad, float *out, int ldo, const float *bias, int *work,
                               size_t work_bytes) {
  if (M <= 0 || N <= 0 || kpad <= 0 || kpad % 16) return qh::fail_msg("gemm_i8: bad shape");
  switch (mode) {
    case GM_PLAIN: return launch<GM_PLAIN>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, work, work_bytes);
    case GM_RESID: return launch<GM_RESID>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, work, work_bytes);
    case GM_SWIGLU: return launch<GM_SWIGLU>(A, as, W, ws, M, N, kpad, out, ldo, bias, cls, work, work_bytes);
    default: return qh::fail_msg("gemm_i8: bad mode");
  }
}

extern "C" int qhip_gemm_i8(int mode, int cls, const int8_t *A, const float *as, const int8_t *W, const float *ws,
                            int M, int N, int kpad, float *out, int ldo, const float *bias) {
  return qhip_gemm_i8_ws(mode, cls, A, as, W, ws, M, N, kpad, out, ldo, bias, nullptr, 0);
}

// Test entry: one GEMM (mode 0 plain + bias, 1 residual, 2 SwiGLU) from host
// operands, run whole and with a 64 MB split-K workspace; out_plain and
// out_split hold the residual's initial values on entry (mode 1) and the two
// results on return; *splits = the K splits the second run used.
extern "C" int qllama_test_gemm_split(int mode, const int8_t *A, const float *as, const int8_t *W, const float *ws,
                                      int M, int N, int kpad, const float *bias, float *out_plain, float *out_split,
                                      int *splits) {
  if (qhip_init()) return 1;
  if (mode < 0 || mode > 2 || M <= 0 || N <= 0 || kpad <= 0 || kpad % 16) return qh::fail_msg("test_gemm_split: bad shape");
  const size_t wrows = mode == GM_SWIGLU ? 2 * (size_t)N : (size_t)N, nout = (size_t)M * N;
  const size_t work_bytes = (size_t)64 << 20;
  int8_t *dA = (int8_t *)qhip_malloc((size_t)M * kpad), *dW = (int8_t *)qhip_malloc(wrows * kpad);
  float *das = (float *)qhip_malloc((size_t)M * 4), *dws = (float *)qhip_malloc(wrows * 4);
  float *db = bias ? (float *)qhip_malloc((size_t)N * 4) : nullptr;
  float *o1 = (float *)qhip_malloc(nout * 4), *o2 = (float *)qhip_malloc(nout * 4);
  int *work = (int *)qhip_malloc(work_bytes);
  int rc = (!dA || !dW || !das || !dws || (bias && !db) || !o1 || !o2 || !work) ? 1 : 0;
  if (!rc)
    rc = qhip_h2d(dA, A, (size_t)M * kpad) || qhip_h2d(dW, W, wrows * kpad) || qhip_h2d(das, as, (size_t)M * 4) ||
         qhip_h2d(dws, ws, wrows * 4) || (bias && qhip_h2d(db, bias, (size_t)N * 4)) ||
         qhip_h2d(o1, out_plain, nout * 4) || qhip_h2d(o2, out_split, nout * 4);
  if (!rc) rc = qhip_gemm_i8(mode, QK_OTHER, dA, das, dW, dws, M, N, kpad, o1, N, db);
  if (!rc) rc = qhip_gemm_i8_ws(mode, QK_OTHER, dA, das, dW, dws, M, N, kpad, o2, N, db, work, work_bytes);
  if (!rc) *splits = g_last_splits;
  if (!rc) rc = qhip_device_sync() || qhip_d2h(out_plain, o1, nout * 4) || qhip_d2h(out_split, o2, nout * 4);
  qhip_free(dA); qhip_free(dW); qhip_free(das); qhip_free(dws); qhip_free(db); qhip_free(o1); qhip_free(o2);
  qhip_free(work);
  return rc;
}
