// Shared parts of the sampling kernels: torch's argmax order, the race's best
// key with its bounds, the decision's error band and the commit cut of a round
// (engine/spec_scheduler.py:46-88, 274-303; specdec/sampler.py:59-92).
#pragma once

#include <math.h>

#include "spv_common.h"

namespace spv {

constexpr float kLog2e = 1.4426950408889634f;
constexpr double kEps = 1e-12;     // specdec/sampler.py:16
// Relative rounding of the race's fast keys against the same key formed with
// torch's arithmetic on the same p and q (hardware reciprocal of E, x / T as a
// product, r / E against (r / t) / E): a few ulp, well inside 1e-6.
constexpr float kTieRel = 1e-6f;
// Error of p (and q) in logits mode against torch's softmax, relative: the
// normaliser (another summation order of fast-exp2 terms) and the per-element
// exp. The race's fused exponent fma(x, log2 e, -m log2 e) adds |m| 2^-22
// (kMRel: the rounding of m log2 e, and with T != 1 the product x * (1/T)
// against torch's x / T) and a part proportional to |x - m|, at most
// 6 2^-24 |x - m|; since p = e^(x - m) / s and y e^-y <= 1/e, that part is an
// absolute error below kDAbs / s (kDAbs = 2^-21 / e).
constexpr float kProbRel = 4e-6f;
constexpr float kMRel = 2.384185791015625e-07f;  // 2^-22
constexpr float kDAbs = 1.7542e-07f;             // 2^-21 / e, rounded up
// Band of a decision: the relative error of p / q (twice kProbRel, plus the
// rounding of the quotient).
constexpr double kDecideRel = 2.0 * 4e-6 + 2.384185791015625e-07;
// Exact re-races: keys formed with torch's arithmetic on this kernel's p, q and
// normalisers differ from torch's own by a few roundings (exp, the divisions):
// 8 ulp covers them.
constexpr float kExactRel = 9.5367431640625e-07f;  // 2^-20

// torch.argmax order: NaN beats numbers (first NaN wins), else larger value,
// ties to the lower index.
__device__ __forceinline__ bool better(float va, int ia, float vb, int ib) {
  const bool na = isnan(va), nb = isnan(vb);
  if (na || nb) return na && (!nb || ia < ib);
  return va > vb || (va == vb && ia < ib);
}

__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float v2 = __shfl_xor(v, o, 64);
    const int i2 = __shfl_xor(i, o, 64);
    if (better(v2, i2, v, i)) {
      v = v2;
      i = i2;
    }
  }
}

// Argmax over the workgroup; every thread gets the result.
__device__ __forceinline__ void block_argmax(float& v, int& i) {
  __shared__ float sv[16];
  __shared__ int si[16];
  wave_argmax(v, i);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sv[w] = v;
    si[w] = i;
  }
  __syncthreads();
  v = sv[0];
  i = si[0];
  for (int k = 1; k < nw; ++k)
    if (better(sv[k], si[k], v, i)) {
      v = sv[k];
      i = si[k];
    }
  __syncthreads();
}

// The best key (torch.argmax order) with an upper bound u of its true value,
// and uo, the largest upper bound over every other key seen. The best key is
// certain when its lower bound v - (u - v) clears uo: no other key can be
// above it, whatever its rounding. With exact keys (u = v) uo is the
// runner-up's value.
struct Top1 {
  float v, u, uo;
  int i;
  __device__ __forceinline__ void init() {
    v = u = uo = -INFINITY;
    i = 0x7fffffff;
  }
  // A key of a higher index than every key pushed before (a thread's keys come
  // in rising index order, so an equal key never takes the lead). NaN keys are
  // tracked apart by the caller (lead_nan).
  __device__ __forceinline__ void push(float key, float ub, int idx) {
    const bool c1 = key > v;
    uo = fmaxf(uo, c1 ? u : ub);
    u = c1 ? ub : u;
    v = c1 ? key : v;
    i = c1 ? idx : i;
  }
  __device__ __forceinline__ void merge(float w, float wu, float wuo, int j) {
    if (better(w, j, v, i)) {
      uo = fmaxf(fmaxf(uo, u), wuo);
      v = w;
      u = wu;
      i = j;
    } else {
      uo = fmaxf(fmaxf(uo, wu), wuo);
    }
  }
  __device__ __forceinline__ void wave_reduce() {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
      merge(__shfl_xor(v, o, 64), __shfl_xor(u, o, 64), __shfl_xor(uo, o, 64), __shfl_xor(i, o, 64));
  }
  // The first NaN key of the thread (index nan_i) leads its list, as in torch.argmax.
  __device__ __forceinline__ void lead_nan(int nan_i) {
    if (nan_i == 0x7fffffff) return;
    uo = fmaxf(uo, u);
    v = u = __uint_as_float(0x7fc00000u);
    i = nan_i;
  }
  // The best key is above every other by more than the bounds and `slack`
  // (a NaN key is certain: it wins outright).
  __device__ __forceinline__ bool certain(float slack) const {
    return isnan(v) || (v - (u - v)) - uo > slack;
  }
};

// Top1 over the workgroup; every thread gets the result.
__device__ __forceinline__ void block_top1(Top1& t) {
  __shared__ float sv[16], su[16], suo[16];
  __shared__ int si[16];
  t.wave_reduce();
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sv[w] = t.v;
    su[w] = t.u;
    suo[w] = t.uo;
    si[w] = t.i;
  }
  __syncthreads();
  t.v = sv[0];
  t.u = su[0];
  t.uo = suo[0];
  t.i = si[0];
  for (int k = 1; k < nw; ++k) t.merge(sv[k], su[k], suo[k], si[k]);
  __syncthreads();
}

__device__ __forceinline__ double block_sum_f64(double x) {
  __shared__ double sd[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) sd[w] = x;
  __syncthreads();
  double t = 0.0;
  for (int k = 0; k < nw; ++k) t += sd[k];
  __syncthreads();
  return t;
}

// ------------------------------------------------------------ arguments
struct DecideArgs {
  const float* target;
  const float* draft;
  const float* dstats;  // (B, gamma) float2 statistics of the draft rows, or null
  const int32_t* proposals;
  const float* u;
  double* accept_prob;
  int32_t* accept_len;
  int32_t* out_tokens;
  int32_t* flags;
  int B, gamma, V, is_probs, greedy, decide_only;
  int split;  // pieces per statistics row
  float tf;
};

struct CommitArgs {
  const int32_t* start;
  const int32_t* remaining;
  const float* noise;
  int eos;
  int32_t* n_commit;
  int32_t* finished;
  int32_t* new_len;
};

// p[x] of a softmax row, float32 as torch.softmax forms it: exp(x - max) / sum.
__device__ __forceinline__ float softmax_at(float z, float m, float s, float tf) {
  const float x = tf == 1.0f ? z : z / tf;
  return expf(x - m) / s;
}

// Commit cut of one sequence (spec_scheduler.py:274-303): the budget with
// Python slice semantics, then the first eos (not kept). `xs` holds the
// proposals; `rem` and `st` are remaining[b] and start[b] (loaded early).
__device__ __forceinline__ void commit_cut(const DecideArgs& a, const CommitArgs& cm, int b, int k, int token, const int* xs,
                           int rem, int st) {
  int n = k + 1;
  bool fin = false;
  if (cm.remaining && n > rem) n = rem >= 0 ? rem : max(0, n + rem);
  if (cm.eos >= 0) {
    for (int i = 0; i < n; ++i) {
      const int tok = i < k ? xs[i] : token;
      if (tok == cm.eos) {
        n = i;
        fin = true;
        break;
      }
    }
  }
  if (n == 0) fin = true;
  if (cm.remaining && n >= rem) fin = true;
  if (cm.n_commit) cm.n_commit[b] = n;
  if (cm.finished) cm.finished[b] = fin ? 1 : 0;
  if (cm.new_len) cm.new_len[b] = n > 0 ? st + n : -1;
}

// Whether the reference's decision `u < min(1, p/q)` (both 1e-12 branches) can
// differ from this one when its p and q may each lie a relative `beta`/2 away
// from pd and qd (beta: the band of the quotient).
__device__ __forceinline__ bool decision_in_band(double pd, double qd, double u, double beta) {
  const double lo_eps = kEps / (1.0 + beta), hi_eps = kEps * (1.0 + beta);
  if (qd >= lo_eps && qd <= hi_eps) return true;  // the q <= 1e-12 branch itself
  if (qd < lo_eps) return pd >= lo_eps && pd <= hi_eps;  // a = 1 or 0 by p > 1e-12
  const double rho = pd / qd;
  const double lo = rho * (1.0 - beta);
  if (lo >= 1.0) return false;  // a = 1 for both, and u < 1
  return u >= lo && u < fmin(1.0, rho * (1.0 + beta));
}

// float(max(T, 1e-12)) as the fp32 scalar torch divides by.
inline float temperature_divisor(float T) { return (float)((double)T > kEps ? (double)T : kEps); }

// ------------------------------------------------------- top-k / top-p filters
// Half width of the window around the nucleus edge p W (relative to W) where
// the reference's fp32 softmax and cumulative sum can keep or drop a value
// differently from the exact masses: torch's normalisation of a 151,936-entry
// row is off by up to ~1e-5, and the cumulative sum rounds each entry.
constexpr double kTopPWindow = 5e-5;

// Larger x, larger key; NaN above everything (torch.topk ranks NaN first).
__device__ __forceinline__ uint32_t order_key(float x) {
  const uint32_t u = __float_as_uint(x);
  if (x != x) return 0xffffffffu;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// A top-k bound: +0.0 ranks above -0.0, which the filter's float comparison does
// not drop either. (One key for both zeros in order_key itself cost 2-3 us a call
// at top_k 512, and 1% of the general filter.)
__device__ __forceinline__ uint32_t with_both_zeros(uint32_t key) { return key == 0x80000000u ? 0x7fffffffu : key; }

__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// The mass exp(x - max) of a value, as fp64 sums take it. (x - max first: max
// log2 e overflows in a row whose largest value is a mask's, the type's lowest.)
__device__ __forceinline__ double mass_of(float x, float mx) {
  return (double)__builtin_amdgcn_exp2f((x - mx) * kLog2e);
}
__device__ __forceinline__ double key_mass(uint32_t k, float mx) { return mass_of(key_value(k), mx); }

// Block-wide exclusive scan of one double per thread (bins in descending order).
__device__ __forceinline__ double block_exclusive_scan_f64(double v, double* lds, double* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  double incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  double off = 0.0, sum = 0.0;
  for (int w = 0; w < nw; ++w) {
    const double x = lds[w];
    if (w < wave) off += x;
    sum += x;
  }
  __syncthreads();
  *total = sum;
  return off + incl - v;
}

// spv_verify_sample with rows filtered beforehand (verify_sample.hip): `need`
// (B, may be null): only the sequences with need[b] != 0 take part;
// `amb_t` (B, gamma + 1) and `amb_d` (B, gamma), may be null: a sequence with
// a nonzero count gets SPV_FLAG_TOP_P_BAND.
int verify_sample_impl(const float* target, const float* draft, int is_probs, float temperature,
                       const int32_t* proposals, const float* u_accept, const float* exp_noise,
                       const float* draft_stats, const int32_t* start_pos, const int32_t* remaining, int32_t eos_id,
                       int32_t B, int32_t gamma, int32_t V, int32_t* accept_len, int32_t* out_tokens,
                       int32_t* n_commit, int32_t* finished, int32_t* new_len, double* accept_prob, int32_t* flags,
                       int32_t decide_only, const int32_t* need, const int32_t* amb_t, const int32_t* amb_d,
                       void* workspace, size_t workspace_bytes, void* stream);

// The filters of a verify step's rows (filter_logits.hip), target and draft in
// one launch: (B, gamma + 1, V) and (B, gamma, V), contiguous; counts and
// `need` as above (counts null: not taken).
int filter_verify_rows(const float* target, float* target_out, int32_t* amb_t, const float* draft, float* draft_out,
                       int32_t* amb_d, const int32_t* need, int32_t B, int32_t gamma, int32_t V, float temperature,
                       int32_t top_k, float top_p, void* stream);

}  // namespace spv
