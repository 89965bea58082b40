// k_sample.hip - token sampling on the device: greedy (sampler.c:8-21) and
// temperature + top-k + top-p (sampler.c:54-143), with the reference's results
// bit for bit.
//
// Order of work for one logits row of V values (temperature > 0):
//   k_smp_bmax, k_smp_exp   blockwise: max, e_j = expf((l_j - max) / T)
//   k_smp_steps, k_smp_walk   the sequential float sum of the e_j evaluated
//                 exactly (qdev_seqsum.h): one wave classifies each 1024 steps,
//                 one block walks the hard steps of all of them; p_j = e_j / sum (a
//                 true division, sampler.c:79) is formed where it is used.
//   top-k <= 64   k_smp_walk also finds a bound that at least k of the p_j reach (the
//                 k-th largest of the maxima of groups of 256); k_smp_gather
//                 collects the p_j that reach it, k_smp_top sorts them.
//   otherwise     a stable radix sort of all (p, index) pairs by p descending
//                 (k_rs_*: four passes of 8 bits over the bits of p).  Both
//                 orders are p descending, then index ascending: the order the
//                 reference's qsort (glibc's merge sort, stable) leaves them in.
//   k_smp_pick (k_smp_top's last step)  one wave: keep = top-k, then the top-p cut over the running
//                 sum, the kept mass z, u = uniform * z from the xorshift64
//                 state held in device memory, and the first kept entry whose
//                 running sum reaches u.  Every running sum is the reference's
//                 left-to-right float sum.
#include <hip/hip_runtime.h>

#include <climits>

#include "qdev_math.h"
#include "qdev_seqsum.h"
#include "qhip.h"
#include "qhip_internal.h"

namespace {

constexpr int kNT = 1024;      // threads of the one-block kernels
constexpr int kCM = 32;        // terms per thread in one chunk of the one-block exact sum

__device__ float block_max(float v, float *red) {
  v = qd::wave_max_f32(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float m = red[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = fmaxf(m, red[w]);
  return m;
}

constexpr int kSlice = 1024;   // logits per block in the blockwise kernels (256 threads x 4)
constexpr int kTopC = 64;      // candidates each block passes to the top-k merge
constexpr int kMergeCap = 16384;
constexpr int kUnits = kMergeCap / kTopC;   // slices the top-k path and the split exact sum serve
constexpr int kUnitHard = 256; // hard steps recorded per slice
constexpr int kWalkHard = 1024;             // and over all slices

// What k_smp_walk reads of one slice's steps (see seq_sum_nonneg).
struct SmpUnit {
  unsigned wk;      // total of its k
  int wh;           // hard steps
  int wg, wgi;      // grid of the run continuing past its last step; of its first step if easy, else -1
};

// Per-block maximum of the logits; block 0 clears the counters of the later kernels.
__global__ __launch_bounds__(256) void k_smp_bmax(const float *l, int V, float *bm, int *ctr) {
  __shared__ float red[4];
  const int j0 = blockIdx.x * kSlice + threadIdx.x;
  if (blockIdx.x == 0 && threadIdx.x < 2) ctr[threadIdx.x] = 0;
  float mx = -INFINITY;
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (j0 + 256 * r < V) mx = fmaxf(mx, l[j0 + 256 * r]);
  mx = block_max(mx, red);
  if (threadIdx.x == 0) bm[blockIdx.x] = mx;
}

// e[j] = expf((l[j] - max_l) / temperature)  (sampler.c:68-76); max_l from the
// per-block maxima (a maximum does not depend on the order it is taken in).
// gm[4 b + w]: the largest e of the 256 terms wave w of slice b forms; tot[b]: a float
// total of slice b in any order.
__global__ __launch_bounds__(256) void k_smp_exp(const float *l, int V, float temperature, const float *bm, int nb,
                                                 float *e, float *gm, float *tot) {
  __shared__ float red[4];
  float mx = -INFINITY;
  for (int i = threadIdx.x; i < nb; i += 256) mx = fmaxf(mx, bm[i]);
  mx = block_max(mx, red);
  const int j0 = blockIdx.x * kSlice + threadIdx.x;
  float big = 0.0f, sum = 0.0f;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int j = j0 + 256 * r;
    if (j < V) {
      const float x = qd::expf_glibc((l[j] - mx) / temperature);
      e[j] = x;
      big = fmaxf(big, x);
      sum += x;
    }
  }
  big = qd::wave_max_f32(big);
  sum = qd::wave_sum_f32(sum);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) gm[4 * blockIdx.x + w] = big;
  __syncthreads();                              // red is read above
  if ((threadIdx.x & 63) == 0) red[w] = sum;
  __syncthreads();
  if (threadIdx.x == 0) tot[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// The steps of slice u = blockIdx.x of the sum, classified by one wave (16 a lane):
// its hard steps in order to rec[u * kUnitHard ..], the rest to unit[u].  *bad is
// set where two lanes do not agree on the grid between them.
__global__ __launch_bounds__(64) void k_smp_steps(const float *e, int V, const float *tot, const float *gm,
                                                  SmpUnit *unit, int4 *rec, int *bad) {
  constexpr int CM = kSlice / 64;
  const int u = blockIdx.x, lane = threadIdx.x, j0 = u * kSlice + lane * CM;
  float a[CM];
  if ((u + 1) * kSlice <= V) {
#pragma unroll
    for (int c = 0; c < CM; c += 4) {
      const float4 t = *reinterpret_cast<const float4 *>(e + j0 + c);
      a[c] = t.x; a[c + 1] = t.y; a[c + 2] = t.z; a[c + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int c = 0; c < CM; c++) a[c] = j0 + c < V ? e[j0 + c] : 0.0f;
  }
  // predicted sum before the slice and the largest term before it
  float pre = 0.0f, pm = 0.0f;
  for (int i = lane; i < u; i += 64) {
    const float4 m = *reinterpret_cast<const float4 *>(gm + 4 * i);
    pre += tot[i];
    pm = fmaxf(pm, fmaxf(fmaxf(m.x, m.y), fmaxf(m.z, m.w)));
  }
  pre = qd::wave_sum_f32(pre);
  pm = qd::wave_max_f32(pm);
  float loc = 0.0f;
  unsigned cmx = 0u;
#pragma unroll
  for (int c = 0; c < CM; c++) {
    loc += a[c];
    cmx = max(cmx, __float_as_uint(a[c]));
  }
  const float xin = qd::seq_wave_scan(loc);
  const unsigned mex = qd::seq_wave_scan_umax(qd::seq_shr1(cmx));
  const float rho = 0x1p-20f * __builtin_amdgcn_sqrtf((float)(j0 + CM + 2)) + 0x1p-17f;
  qd::SeqSteps<CM> st;
  qd::seq_classify<CM>(a, pre + (xin - loc), loc, max(mex, __float_as_uint(pm)), rho, false, st);
  const unsigned kin = qd::seq_wave_scan(st.ks);
  const int hin = qd::seq_wave_scan(st.nh);
  const int gprev = (int)qd::seq_shr1((unsigned)st.gout);
  if (lane > 0 && st.gin >= 0 && st.gin != gprev) *bad = 1;
  if (st.nh && hin <= kUnitHard) {
    const unsigned kb = kin - st.ks;
    int m = u * kUnitHard + hin - st.nh;
#pragma unroll
    for (int c = 0; c < CM; c++) {
      const bool h = (st.hardmask >> c) & 1u;
      if (h) rec[m] = make_int4((int)(kb + st.kp[c]), j0 + c, __float_as_int(a[c]), st.gh[c]);
      m += h ? 1 : 0;
    }
  }
  const int gin0 = __builtin_amdgcn_readfirstlane(st.gin);
  if (lane == 63) unit[u] = SmpUnit{kin, hin, st.gout, gin0};
}

// *S = ((0 + e_0) + e_1) + ... + e_{V-1} in float (sampler.c:76), evaluated exactly
// in chunks of kSumNT*kCM terms; after the first chunk, term 0 of a chunk is the
// partial sum so far ((0 + s) = s exactly).  Eight waves: each wave may record
// up to 64 hard steps (the first chunk's partial sums cross many binades early
// on) before the exact-sum walk has to fall back to the loop; sixteen waves
// (32 each) fell back on real logits.
constexpr int kSumNT = 512;
__device__ float chunked_sum(const float *e, int V, qd::SeqScratch &S) {
  const int tid = threadIdx.x;
  float s = 0.0f;
  for (int base = 0, off = 0; base < V; off = 1) {
    const int nnew = min(V - base, kSumNT * kCM - off), n = nnew + off;
    const float s0 = s;
    const int b0 = base, o0 = off;
    float a[kCM];
#pragma unroll
    for (int c = 0; c < kCM; c++) {
      const int q = tid * kCM + c;
      a[c] = q < n ? (q < o0 ? s0 : e[b0 + q - o0]) : 0.0f;
    }
    s = qd::seq_sum_nonneg<kSumNT, kCM>(a, n, S, [=](int i) { return i < o0 ? s0 : e[b0 + i - o0]; });
    base += nnew;
  }
  return s;
}

__global__ __launch_bounds__(kSumNT) void k_smp_sum(const float *e, int V, float *S_out) {
  __shared__ qd::SeqScratch S;
  const float s = chunked_sum(e, V, S);
  if (threadIdx.x == 0) S_out[0] = s;
}

// The same sum from the classified slices: the slices' offsets by a block scan, every
// hard step into LDS in order, and the walk with its proofs by wave 0; where a proof
// fails (or a slice has more hard steps than it could record) the chunked form.
// Meanwhile the other waves find the want-th largest of the group maxima (want >
// 0): at least want terms are as large, so their p is at least S_out[1] = that
// term / S.  S_out[1] = 0 (every p reaches it) where there are fewer groups or S
// is not a positive number.
// Latency of one block: 128256 terms 94 -> 3.5 (k_smp_steps) + 7 us (the chunks of
// 16384 terms ran one after the other, eight meetings and walks in a row).
__global__ __launch_bounds__(kSumNT) void k_smp_walk(const float *e, int V, const SmpUnit *unit, int nu,
                                                     const int4 *rec, const int *bad, const float *gm, int want,
                                                     float *S_out) {
  __shared__ qd::SeqScratch S;
  __shared__ int4 hs[kWalkHard];
  __shared__ __attribute__((aligned(16))) float g[4 * kUnits];
  __shared__ unsigned koff[kUnits];
  __shared__ int hoff[kUnits + 1], wg[kUnits], wsum[kSumNT / 64][2], fail;
  __shared__ float bound;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  static_assert(kUnits <= kSumNT, "one slice a thread");
  if (tid == 0) { fail = *bad; bound = 0.0f; }
  const SmpUnit q = tid < nu ? unit[tid] : SmpUnit{0u, 0, 0, -1};
  const unsigned kin = qd::seq_wave_scan(q.wk);
  const int hin = qd::seq_wave_scan(q.wh);
  if (lane == 63) { wsum[wave][0] = (int)kin; wsum[wave][1] = hin; }
  if (tid < nu) wg[tid] = q.wg;
  // groups: the slices (padded to whole float4s), or their quarters where the slices are few
  const int ng = nu >= 2 * want ? nu : 4 * nu;
  if (ng == nu) {
    if (tid < ((nu + 3) & ~3)) {
      const float4 m = tid < nu ? *reinterpret_cast<const float4 *>(gm + 4 * tid) : make_float4(0.f, 0.f, 0.f, 0.f);
      g[tid] = fmaxf(fmaxf(m.x, m.y), fmaxf(m.z, m.w));
    }
  } else {
    for (int i = tid; i < 4 * nu; i += kSumNT) g[i] = gm[i];
  }
  __syncthreads();
  unsigned kb = kin - q.wk;
  int hb = hin - q.wh, htot = 0;
  unsigned ktot = 0;
#pragma unroll
  for (int w = 0; w < kSumNT / 64; w++) {
    if (w < wave) { kb += (unsigned)wsum[w][0]; hb += wsum[w][1]; }
    ktot += (unsigned)wsum[w][0];
    htot += wsum[w][1];
  }
  if (tid < nu) {
    koff[tid] = kb;
    hoff[tid] = hb;
    if (q.wh > kUnitHard || (tid > 0 && q.wgi >= 0 && q.wgi != wg[tid - 1])) fail = 1;
  }
  if (tid == 0) hoff[nu] = htot;
  __syncthreads();
  bool ok = fail == 0 && htot <= kWalkHard;
  if (ok) {
    for (int i = tid; i < htot; i += kSumNT) {
      int lo = 0, hi = nu;                       // the slice of hard step i: the last whose steps begin at or before i
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (hoff[mid] <= i) lo = mid; else hi = mid;
      }
      int4 r = rec[lo * kUnitHard + i - hoff[lo]];
      r.x = (int)((unsigned)r.x + koff[lo]);
      hs[i] = r;
    }
  }
  __syncthreads();
  if (wave == 0) {
    if (ok) {
      float s = 0.0f;
      int cx = 0, cy = -1, cw = 0;
      for (int base = 0; ok && base <= htot; base += 64) {
        const int m = base + lane;
        const int4 cur = m < htot ? hs[m] : make_int4((int)ktot, INT_MAX, 0, 0);     // the tail
        ok = qd::seq_walk_batch(S, cur, m, base, htot, s, cx, cy, cw) && ok;
      }
      if (lane == 0) S.result = s;
      if (!ok && lane == 0) fail = 1;
    } else if (lane == 0) {
      fail = 1;
    }
  } else if (want > 0 && want <= ng) {
    for (int i = tid - 64; i < ng; i += kSumNT - 64) {
      const float x = g[i];
      int above = 0;                             // maxima before this one in (value descending, index) order
      for (int k = 0; k < ng; k += 4) {
        const float4 y = *reinterpret_cast<const float4 *>(g + k);
        above += (y.x > x || (y.x == x && k < i)) + (y.y > x || (y.y == x && k + 1 < i)) +
                 (y.z > x || (y.z == x && k + 2 < i)) + (y.w > x || (y.w == x && k + 3 < i));
      }
      if (above == want - 1) bound = x;
    }
  }
  __syncthreads();
  float s = S.result;
  if (fail) {                                    // uniform for the block
    __syncthreads();
    s = chunked_sum(e, V, S);
  }
  if (tid == 0) {
    S_out[0] = s;
    S_out[1] = s > 0.0f && s < INFINITY ? bound / s : 0.0f;
  }
}

// p[j] = e[j] / S  (sampler.c:79)
__global__ __launch_bounds__(256) void k_smp_div(const float *e, int V, const float *S, float *p) {
  const float s = S[0];
  const int j0 = blockIdx.x * kSlice + threadIdx.x;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int j = j0 + 256 * r;
    if (j < V) p[j] = e[j] / s;
  }
}

// Sort key of (p, j): probability descending, then index ascending (the order
// of a stable sort by probability, sampler.c:82).  p >= 0, so its bits order
// like its values; 0 never is a real key (j < 2^31).
__device__ __forceinline__ unsigned long long prob_key(float p, int j) {
  return ((unsigned long long)__float_as_uint(p) << 32) | (unsigned)(0xffffffffu - (unsigned)j);
}

// Sum of one int per thread over the block; red holds 2 * (NT / 64) ints and
// alternates halves between calls (parity), so one barrier per call suffices.
template <int NT>
__device__ __forceinline__ int block_count(int n, int *red, int parity) {
  n = qd::wave_sum_i32(n);
  int *r = red + parity * (NT / 64);
  if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = n;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; w++) t += r[w];
  return t;
}

// The K largest of the block's keys (NK per thread; nonzero keys are distinct, 0
// is an empty slot), written unordered to out[0 .. K-1] with K = min(want, number
// of nonzero keys): the K-th largest key is found bit by bit from the top (the
// largest T with at least K keys >= T), then the keys >= T are gathered.
template <int NT, int NK>
__device__ int block_top(const unsigned long long (&k)[NK], int want, unsigned long long *out, int *red, int *cnt) {
  int nz = 0;
#pragma unroll
  for (int i = 0; i < NK; i++) nz += k[i] != 0ull;
  const int K = min(want, block_count<NT>(nz, red, 0));
  unsigned long long T = 0;
  if (K > 0) {
    for (int b = 63; b >= 0; b--) {
      const unsigned long long c = T | (1ull << b);
      int n = 0;
#pragma unroll
      for (int i = 0; i < NK; i++) n += k[i] >= c;
      if (block_count<NT>(n, red, b & 1) >= K) T = c;
    }
  }
  if (threadIdx.x == 0) *cnt = 0;
  __syncthreads();
  if (K > 0) {
#pragma unroll
    for (int i = 0; i < NK; i++)
      if (k[i] >= T) out[atomicAdd(cnt, 1)] = k[i];
  }
  __syncthreads();
  return K;
}

// The keys of the p = e / S that reach S[1], appended to cand in any order (*cnt of
// them): of a slice that holds more than kTopC the kTopC largest, which hold what
// the slice can contribute to the top kTopC of all.
__global__ __launch_bounds__(256) void k_smp_gather(const float *e, int V, const float *S, unsigned long long *cand,
                                                    int *cnt) {
  __shared__ unsigned long long top[kTopC];
  __shared__ int red[8], n, base;
  const float sum = S[0];
  const unsigned least = __float_as_uint(S[1]);
  const int j0 = blockIdx.x * kSlice + threadIdx.x;
  if (threadIdx.x == 0) n = 0;
  __syncthreads();
  unsigned long long k[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int j = j0 + 256 * r;
    const float p = j < V ? e[j] / sum : 0.0f;
    k[r] = j < V && __float_as_uint(p) >= least ? prob_key(p, j) : 0ull;
    if (k[r]) {
      const int at = atomicAdd(&n, 1);
      if (at < kTopC) top[at] = k[r];
    }
  }
  __syncthreads();
  int K = n;
  if (K == 0) return;                            // uniform for the block
  if (K > kTopC) K = block_top<256, 4>(k, kTopC, top, red, &n);
  if (threadIdx.x == 0) base = atomicAdd(cnt, K);
  __syncthreads();
  if ((int)threadIdx.x < K) cand[base + threadIdx.x] = top[threadIdx.x];
}

// First index of the maximum (sampler.c:8-21).  Optional decode-state update as
// k_smp_pick's.
__global__ __launch_bounds__(kNT) void k_smp_argmax(const float *l, int V, int *tok, int *d_in, const int *d_state,
                                                     int *d_out, int max_seq) {
  __shared__ float sv[kNT / 64];
  __shared__ int si[kNT / 64];
  float best = -INFINITY;
  int idx = INT_MAX;
  for (int j = threadIdx.x; j < V; j += kNT) {
    const float v = l[j];
    if (idx == INT_MAX || v > best) { best = v; idx = j; }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (oi != INT_MAX && (idx == INT_MAX || ob > best || (ob == best && oi < idx))) { best = ob; idx = oi; }
  }
  if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = best; si[threadIdx.x >> 6] = idx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float b = sv[0];
    int i0 = si[0];
    for (int w = 1; w < kNT / 64; w++)
      if (si[w] != INT_MAX && (i0 == INT_MAX || sv[w] > b || (sv[w] == b && si[w] < i0))) { b = sv[w]; i0 = si[w]; }
    tok[0] = i0;
    if (d_state) {
      const int P = d_state[0];
      if (P >= 1 && P - 1 < max_seq) d_out[P - 1] = i0;
      if (P >= d_state[1] && P <= max_seq) d_in[P] = i0;
    }
  }
}

__global__ void k_smp_iota(int *idx, int V) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j < V) idx[j] = j;
}

// Lane l's running sum ((s + v_0) + v_1) + ... + v_l over the lanes' values v >= 0
// in lane order: each lane adds the terms up to its own (a +0 otherwise, which
// changes no sum >= +0).  Three instructions a term.
__device__ __forceinline__ float wave_running_sum(float v, float s) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 64; i++) {
    const float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i));
    s += lane >= i ? t : 0.0f;
  }
  return s;
}

// sampler.c:81-139 over the sorted (ps, is) pairs; the xorshift64 step and
// uniform of sampler.c:31-45 on the device state *rng.  When d_state is given
// (decode loop) the token also becomes the next input: position P = d_state[0]
// (already advanced past the row's position) gets d_in[P] = token when P is past
// the prompt, and d_out[P - 1] records it, as k_argmax_final does for greedy.
// The cut, the kept mass and the choice read the same left-to-right running sums,
// which are formed once, 64 at a time, and kept in run (keep floats, where keep may
// exceed 64); they never decrease, so the choice is a search.
// Kept lists of thousands (no top-k): 848 -> 171 us at 128256 logits, top-p 0.95,
// against three serial passes of a read, an add and a branch a term.
__device__ __forceinline__ void smp_pick(const float *ps, const int *is, int V, int top_k, float top_p, float *run,
                                         unsigned long long *rng, int *tok, int *d_in, const int *d_state, int *d_out,
                                         int max_seq) {
  const int lane = threadIdx.x & 63;
  int keep = V;
  if (top_k > 0 && top_k < keep) keep = top_k;
  const bool cut = top_p > 0.0f && top_p < 1.0f;
  float z = 0.0f, r = 0.0f;
  float v = lane < keep ? ps[lane] : 0.0f;
  for (int b = 0; b < keep; b += 64) {
    const float nv = b + 64 + lane < keep ? ps[b + 64 + lane] : 0.0f;      // in flight during the sums
    r = wave_running_sum(v, z);
    if (keep > 64 && b + lane < keep) run[b + lane] = r;
    const int last = min(63, keep - 1 - b);
    const unsigned long long m = cut ? __ballot(lane <= last && r >= top_p) : 0ull;
    const int at = m ? __ffsll((long long)m) - 1 : last;
    z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r), at));
    if (m) {
      keep = b + at + 1;                        // ends the loop
    }
    v = nv;
  }
  unsigned long long x = *rng;
  x ^= x << 13;
  x ^= x >> 7;
  x ^= x << 17;
  const float u = (float)((double)(x >> 11) * (1.0 / 9007199254740992.0)) * z;
  // the first kept entry whose running sum reaches u, else the last
  int c = keep - 1;
  if (keep <= 64) {
    const unsigned long long m = __ballot(lane < keep && u <= r);
    if (m) c = __ffsll((long long)m) - 1;
  } else if (u <= z) {                          // run[keep - 1] = z reaches it (no NaN among them)
    __threadfence_block();
    int lo = 0, hi = keep - 1;                  // the answer lies in [lo, hi]
    while (hi > lo) {
      const int step = (hi - lo + 64) >> 6, i = min(lo + step * (lane + 1) - 1, hi);
      const unsigned long long m = __ballot(u <= run[i]);
      const int l = __ffsll((long long)m) - 1;  // lane 63 covers hi, so m is not empty
      const int nlo = lo + step * l;
      hi = min(nlo + step - 1, hi);
      lo = nlo;
    }
    c = lo;
  }
  const int t = is[c];
  if (lane == 0) {
    *rng = x;
    tok[0] = t;
    if (d_state) {
      const int P = d_state[0];
      if (P >= 1 && P - 1 < max_seq) d_out[P - 1] = t;
      if (P >= d_state[1] && P <= max_seq) d_in[P] = t;
    }
  }
}

__global__ __launch_bounds__(64) void k_smp_pick(const float *ps, const int *is, int V, int top_k, float top_p,
                                                  float *run, unsigned long long *rng, int *tok, int *d_in, const int *d_state,
                                                  int *d_out, int max_seq) {
  smp_pick(ps, is, V, top_k, top_p, run, rng, tok, d_in, d_state, d_out, max_seq);
}

// The kTopC largest of the gathered keys in order, and the pick over them.  Keys are
// distinct, so a key's place is the number of larger ones; more than kNT keys (many
// equal logits) are first cut to the kTopC largest.
// Typically 50-100 keys: 30 + 16 us of bitwise searches over 64 keys a slice -> 6 us.
__global__ __launch_bounds__(kNT) void k_smp_top(const unsigned long long *cand, const int *cnt, int V, int top_k,
                                                 float top_p, unsigned long long *rng, int *tok, int *d_in,
                                                 const int *d_state, int *d_out, int max_seq) {
  constexpr int NK = kMergeCap / kNT;
  __shared__ __attribute__((aligned(16))) unsigned long long keys[kNT];
  __shared__ int red[2 * (kNT / 64)], c2;
  __shared__ float ps[kTopC];
  __shared__ int is[kTopC];
  const int tid = threadIdx.x;
  int n = *cnt;
  if (n > kNT) {                                 // uniform for the block
    unsigned long long k[NK];
#pragma unroll
    for (int i = 0; i < NK; i++) {
      const int c = tid + kNT * i;
      k[i] = c < n ? cand[c] : 0ull;
    }
    n = block_top<kNT, NK>(k, kTopC, keys, red, &c2);
  } else if (tid < n) {
    keys[tid] = cand[tid];
  }
  if (tid >= n) keys[tid] = 0ull;
  __syncthreads();
  if (tid < n) {
    const unsigned long long x = keys[tid];
    int above = 0;
    for (int i = 0; i < n; i += 2) {             // keys past n are 0
      const ulonglong2 y = *reinterpret_cast<const ulonglong2 *>(&keys[i]);
      above += (y.x > x) + (y.y > x);
    }
    if (above < kTopC) {
      ps[above] = __uint_as_float((unsigned)(x >> 32));
      is[above] = (int)(0xffffffffu - (unsigned)x);
    }
  }
  __syncthreads();
  if (tid < 64) smp_pick(ps, is, V, top_k, top_p, nullptr, rng, tok, d_in, d_state, d_out, max_seq);
}

size_t al256(size_t n) { return (n + 255) & ~(size_t)255; }

// ---- stable LSD radix sort of (p, index) by p descending ----
// p >= 0, so the bits of p order like its values; a pass sorts by one byte of
// them, digit = 255 - byte (ascending digits = descending p), keeping the order
// of equal digits, so four passes from the low byte leave p descending with
// equal p in their input (index) order.  A block owns a tile of kRsTile items
// taken in kRsRounds rounds of 256 (item = tile start + 256 * round + thread),
// which is their input order.
constexpr int kRsNT = 256, kRsRounds = 16, kRsTile = kRsNT * kRsRounds;

int rs_blocks(int V) { return (V + kRsTile - 1) / kRsTile; }

__device__ __forceinline__ int rs_digit(float p, int shift) {
  return 255 - (int)((__float_as_uint(p) >> shift) & 255u);
}

// counts[256 b + d]: items of tile b with digit d
__global__ __launch_bounds__(kRsNT) void k_rs_hist(const float *keys, int V, int shift, int *counts, int nbs) {
  __shared__ int h[256];
  const int tid = threadIdx.x;
  h[tid] = 0;
  __syncthreads();
  const int j0 = blockIdx.x * kRsTile + tid;
  for (int r = 0; r < kRsRounds; r++) {
    const int j = j0 + kRsNT * r;
    if (j < V) atomicAdd(&h[rs_digit(keys[j], shift)], 1);
  }
  __syncthreads();
  counts[blockIdx.x * 256 + tid] = h[tid];
}

// In place: counts[256 b + d] becomes the output position of the first item of
// tile b with digit d (an exclusive scan in (digit, tile) order).  One block,
// thread d; the tiles' counts eight at a time in flight.
__global__ __launch_bounds__(kRsNT) void k_rs_scan(int *counts, int nbs) {
  __shared__ int wt[kRsNT / 64];
  const int d = threadIdx.x;
  int t = 0;
#pragma unroll 8
  for (int b = 0; b < nbs; b++) t += counts[b * 256 + d];
  const int in = qd::seq_wave_scan(t);
  if ((d & 63) == 63) wt[d >> 6] = in;
  __syncthreads();
  int base = in - t;                              // exclusive prefix over the digits below d
  for (int w = 0; w < (d >> 6); w++) base += wt[w];
  for (int b0 = 0; b0 < nbs; b0 += 8) {
    int c[8];
#pragma unroll
    for (int i = 0; i < 8; i++) c[i] = b0 + i < nbs ? counts[(b0 + i) * 256 + d] : 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (b0 + i < nbs) counts[(b0 + i) * 256 + d] = base;
      base += c[i];
    }
  }
}

// Each item to offs[digit, tile] + the number of earlier items of its tile with
// the same digit: in a round, the lanes of a wave with the same digit are found
// by ballots over the digit's bits, and the waves' counts per digit are added in
// wave order.
__global__ __launch_bounds__(kRsNT) void k_rs_scatter(const float *kin, const int *vin, float *kout, int *vout, int V,
                                                      int shift, const int *offs, int nbs) {
  constexpr int NW = kRsNT / 64;
  __shared__ int base[256];
  __shared__ int wc[NW][256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  base[tid] = offs[blockIdx.x * 256 + tid];
  const unsigned long long lt = (1ull << lane) - 1ull;
  const int j0 = blockIdx.x * kRsTile + tid;
  for (int r = 0; r < kRsRounds; r++) {
#pragma unroll
    for (int w = 0; w < NW; w++) wc[w][tid] = 0;
    __syncthreads();
    const int j = j0 + kRsNT * r;
    const bool ok = j < V;
    const float key = ok ? kin[j] : 0.0f;
    const int val = ok ? vin[j] : 0;
    const int d = ok ? rs_digit(key, shift) : 256;    // 256: no item (9 bits tell it apart)
    unsigned long long peers = __ballot(1);
#pragma unroll
    for (int bit = 0; bit < 9; bit++) {
      const bool set = (d >> bit) & 1;
      const unsigned long long m = __ballot(set);
      peers &= set ? m : ~m;
    }
    const int rank = __popcll(peers & lt);
    if (ok && rank == 0) wc[wave][d] = __popcll(peers);
    __syncthreads();
    {                                             // thread tid = digit tid: offsets of the waves
      int acc = base[tid];
#pragma unroll
      for (int w = 0; w < NW; w++) {
        const int c = wc[w][tid];
        wc[w][tid] = acc;
        acc += c;
      }
      base[tid] = acc;
    }
    __syncthreads();
    if (ok) {
      const int pos = wc[wave][d] + rank;
      kout[pos] = key;
      vout[pos] = val;
    }
    __syncthreads();
  }
}

int nblocks(int V) { return (V + kSlice - 1) / kSlice; }

// Scratch layout: e, p, sorted p, indices, sorted indices (V each), block maxima,
// the sum and the top-k bound, counters, top-k candidates, the slices' totals, group
// maxima and classified steps, then the radix sort's digit counts per tile.
struct Layout {
  float *e, *p, *ps, *bm, *S, *gm, *tot;
  int *idx, *is, *counts, *ctr;
  SmpUnit *unit;
  int4 *rec;
  unsigned long long *cand;
  size_t total;
};

Layout layout(void *base, int V) {
  Layout L{};
  uint8_t *b = static_cast<uint8_t *>(base);
  const size_t slot = al256((size_t)V * 4), nb = (size_t)nblocks(V);
  size_t o = 0;
  L.e = reinterpret_cast<float *>(b + o); o += slot;
  L.p = reinterpret_cast<float *>(b + o); o += slot;
  L.ps = reinterpret_cast<float *>(b + o); o += slot;
  L.idx = reinterpret_cast<int *>(b + o); o += slot;
  L.is = reinterpret_cast<int *>(b + o); o += slot;
  L.bm = reinterpret_cast<float *>(b + o); o += al256(nb * 4);
  L.S = reinterpret_cast<float *>(b + o); o += 256;
  L.ctr = reinterpret_cast<int *>(b + o); o += 256;      // [0] grids that do not meet, [1] candidates
  const size_t nu = nb <= (size_t)kUnits ? nb : 0;       // larger vocabularies sum in one block and sort
  L.cand = reinterpret_cast<unsigned long long *>(b + o); o += al256(nu * kTopC * 8);
  L.gm = reinterpret_cast<float *>(b + o); o += al256(nb * 16);
  L.tot = reinterpret_cast<float *>(b + o); o += al256(nb * 4);
  L.unit = reinterpret_cast<SmpUnit *>(b + o); o += al256(nu * sizeof(SmpUnit));
  L.rec = reinterpret_cast<int4 *>(b + o); o += al256(nu * kUnitHard * sizeof(int4));
  L.counts = reinterpret_cast<int *>(b + o); o += al256((size_t)256 * rs_blocks(V) * 4);
  L.total = o;
  return L;
}

}  // namespace

// Scratch of qhip_sample for rows of V logits.
extern "C" size_t qhip_sample_scratch(int V) {
  if (V <= 0) return 0;
  return layout(nullptr, V).total;
}

// Whether qhip_sample takes the top-k path (top_k <= 64) for these arguments
// rather than the full radix sort.
extern "C" int qhip_sample_topk_path(int V, int top_k) {
  return top_k >= 1 && top_k <= kTopC && V > 0 && nblocks(V) <= kUnits;
}

extern "C" int qhip_sample(const float *logits, int V, float temperature, int top_k, float top_p, void *scratch,
                           size_t scratch_bytes, unsigned long long *rng, int *tok, int *d_in, const int *d_state,
                           int *d_out, int max_seq) {
  if (V <= 0 || !(temperature > 0.0f)) return qh::fail_msg("sample: needs V > 0 and temperature > 0");
  if (scratch_bytes < qhip_sample_scratch(V)) return qh::fail_msg("sample: scratch too small");
  const Layout L = layout(scratch, V);
  const int nb = nblocks(V);
  const int topk = qhip_sample_topk_path(V, top_k);
  QH_LAUNCH(QK_OTHER, k_smp_bmax, dim3(nb), dim3(256), 0, logits, V, L.bm, L.ctr);
  QH_LAUNCH(QK_OTHER, k_smp_exp, dim3(nb), dim3(256), 0, logits, V, temperature, L.bm, nb, L.e, L.gm, L.tot);
  if (nb <= kUnits) {
    QH_LAUNCH(QK_OTHER, k_smp_steps, dim3(nb), dim3(64), 0, L.e, V, L.tot, L.gm, L.unit, L.rec, L.ctr);
    QH_LAUNCH(QK_OTHER, k_smp_walk, dim3(1), dim3(kSumNT), 0, L.e, V, L.unit, nb, L.rec, L.ctr, L.gm,
              topk ? min(top_k, V) : 0, L.S);
  } else {
    QH_LAUNCH(QK_OTHER, k_smp_sum, dim3(1), dim3(kSumNT), 0, L.e, V, L.S);
  }
  if (topk) {
    QH_LAUNCH(QK_OTHER, k_smp_gather, dim3(nb), dim3(256), 0, L.e, V, L.S, L.cand, L.ctr + 1);
    QH_LAUNCH(QK_OTHER, k_smp_top, dim3(1), dim3(kNT), 0, L.cand, L.ctr + 1, V, top_k, top_p, rng, tok, d_in, d_state,
              d_out, max_seq);
    return 0;
  } else {
    // p and the indices start in (ps, is); four passes, ping-ponging through
    // (p, idx), leave them sorted in (ps, is)
    QH_LAUNCH(QK_OTHER, k_smp_div, dim3(nb), dim3(256), 0, L.e, V, L.S, L.ps);
    QH_LAUNCH(QK_OTHER, k_smp_iota, dim3((V + 255) / 256), dim3(256), 0, L.is, V);
    const int nbs = rs_blocks(V);
    for (int pass = 0; pass < 4; pass++) {
      const int shift = 8 * pass;
      const float *ki = pass & 1 ? L.p : L.ps;
      const int *vi = pass & 1 ? L.idx : L.is;
      float *ko = pass & 1 ? L.ps : L.p;
      int *vo = pass & 1 ? L.is : L.idx;
      QH_LAUNCH(QK_OTHER, k_rs_hist, dim3(nbs), dim3(kRsNT), 0, ki, V, shift, L.counts, nbs);
      QH_LAUNCH(QK_OTHER, k_rs_scan, dim3(1), dim3(kRsNT), 0, L.counts, nbs);
      QH_LAUNCH(QK_OTHER, k_rs_scatter, dim3(nbs), dim3(kRsNT), 0, ki, vi, ko, vo, V, shift, L.counts, nbs);
    }
  }
  QH_LAUNCH(QK_OTHER, k_smp_pick, dim3(1), dim3(64), 0, L.ps, L.is, V, top_k, top_p, L.e, rng, tok, d_in, d_state,
            d_out, max_seq);
  return 0;
}

extern "C" int qhip_argmax_row(const float *logits, int V, int *tok, int *d_in, const int *d_state, int *d_out,
                               int max_seq) {
  if (V <= 0) return qh::fail_msg("argmax: needs V > 0");
  QH_LAUNCH(QK_OTHER, k_smp_argmax, dim3(1), dim3(kNT), 0, logits, V, tok, d_in, d_state, d_out, max_seq);
  return 0;
}
