// Verify sampling with top-k / top-p filters on gfx950: logits_to_probs with
// filters (specdec/sampler.py:19-56) on every target and draft row, then
// batch_accept and the commit cut (engine/spec_scheduler.py:46-88, 274-303).
//
// With top-k on, at most a few hundred values of a 151,936-entry row survive,
// so the filtered rows are never written: one launch reads every row once and
// keeps its survivors.
//   1. A workgroup per row piece holds the piece in registers (64 values per
//      thread for most calls, all loads in flight). The k-th largest of 1,024 group maxima
//      bounds the piece's k-th largest value from below, so every value at or
//      above it (a few more than k) is a candidate and the rest cannot survive.
//   2. The last piece of a row takes the candidates of all pieces, selects the
//      exact k-th largest scaled value (ties stay), sorts what is kept, cuts
//      the nucleus by fp64 masses in sorted order, and publishes the row's
//      softmax statistics, the kept value at the proposal, and the kept list.
//   3. The last row of a sequence decides, races the raced row's kept list with
//      torch's arithmetic (every other token's key is exactly 0) and commits.
// The rows are read once and nothing else of their size moves: the launch is
// bound by HBM. B = 32, gamma = 5, V = 151,936, T = 0.8, top_k 50, top_p 0.9
// (233 MB): 75 us per call against 662 for filtering all rows into memory
// (five passes a row), their statistics and the race, 900 when a draw was re-raced.
// Of the 75 the reading takes 38; the rest is the tail of the last rows -- bound,
// publication, row, sequence, each a chain of barriers and uncached round trips
// -- and three empty launches of the general kernels. With searches that halved
// the key space (14 and 19 barriers) and a row's lists read one dependent load
// at a time the call took 98.
//
// Whatever the short form does not cover -- a NaN or infinite logit, more ties
// or candidates than the lists hold, a row with nothing finite, a race noise
// entry that is not above zero -- marks its sequence in `need`, and the general
// kernels (filter_logits.hip, verify_sample.hip), launched after it on the
// marked sequences alone, make its result.
#include <algorithm>

#include "sample_common.h"

using namespace spv;

namespace {

constexpr int kTThreads = 256;
constexpr int kTWaves = kTThreads / 64;
// Largest top_k of the short form (and the temperatures it takes: those whose
// quotients stay far from overflow and underflow). B = 32, gamma = 5,
// V = 151,936, T = 0.8, top_p 0.9, us per call: top_k 20 72, 50 76, 200 106,
// 400 153, 512 193 (the lists grow with it), against 605 for the general path;
// B = 1: 33 to 67 against 256.
constexpr int kTopkMax = 512;
constexpr float kTempMin = 0x1p-10f, kTempMax = 0x1p10f;
constexpr int kPieceCap = 1024;  // candidates of a piece
constexpr int kRowCap = 4096;    // candidates of a row
constexpr int kRowCapMid = 2048; // the same where kVecMid pieces are held
constexpr int kKeepCap = 1024;   // kept values of a row
constexpr int kMaxPieces = 16;
// float4 per thread of a piece: 16 (16,384 values) when the batch's rows fill
// the CUs, 10 for a few rows, and 40 where the lists of 16 would not hold a
// large top_k's candidates. 16 take 128 registers, so four workgroups of a CU
// overlap one's loads with the others' selection (B = 32, top_k 50, us per call:
// 77 with 16, 79 with 20, 87 with 40 and two workgroups per CU).
constexpr int kVecBig = 40, kVecMid = 16, kVecSmall = 10;
constexpr int row_cap(int nvec) { return nvec == kVecMid ? kRowCapMid : kRowCap; }
constexpr size_t kMaxListBytes = (size_t)256 << 20;
constexpr int kMaxRows = 65536;  // row counters

// What a row publishes: softmax statistics of the kept values, the kept scaled
// value at the row's proposal (-inf: dropped), the kept count, the window
// count, and the last kept value (key, index): a value is kept when it sorts
// at or before it.
struct RowDesc {
  float M, S, zx;
  int n, amb;
  uint32_t last_key;
  int last_idx, bad;
};  // 32 bytes: two coherent 16-byte accesses

struct TkArgs {
  DecideArgs d;
  CommitArgs c;
  int pieces, top_k;
  float top_p;
  int32_t* need;
  int* cnt_row;   // [B (2 gamma + 1)] pieces of a row that have finished
  int* cnt_seq;   // [B] rows and noise pieces of a sequence that have finished
  int2* counts;   // [B (2 gamma + 2)][pieces]: a piece's candidates (-1: too many), or a noise piece's verdict
  uint2* lists;   // [B (2 gamma + 1)][pieces][kPieceCap]: (logit bits, index); then the row's kept list (x bits, index)
  RowDesc* desc;  // [B (2 gamma + 1)]
};

__device__ __forceinline__ unsigned long long pack_entry(uint32_t key, int idx) {
  return (unsigned long long)key << 32 | (0xffffffffu - (uint32_t)idx);  // larger: larger value, then lower index
}
__device__ __forceinline__ uint32_t entry_key(unsigned long long e) { return (uint32_t)(e >> 32); }
__device__ __forceinline__ int entry_idx(unsigned long long e) { return (int)(0xffffffffu - (uint32_t)e); }

// The first key above -inf's.
constexpr uint32_t kFirstKey = 0x00800000u;

// A bracket of the want-th largest of the workgroup's keys: at least `want`
// (c of them) are >= lo, fewer are >= hi; lo = 0 when fewer than `want` are
// finite. One histogram of the keys over 256 equal bins of their range and its
// suffix sums, three barriers: halving the key space took 14 (a piece's bound) to
// 19 (a row's threshold) of them, about 0.4 us each.
struct Bracket {
  uint32_t lo, hi;
  int c;
};
struct BracketLds {
  int hist[256];
  uint32_t lo[kTWaves], hi[kTWaves];
};
template <int N>
__device__ __forceinline__ Bracket block_bracket(const uint32_t (&key)[N], int want, BracketLds& s) {
  const int t = threadIdx.x, lane = t & 63;
  uint32_t kmin = 0xffffffffu, kmax = 0;
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (key[i] >= kFirstKey) {
      kmin = min(kmin, key[i]);
      kmax = max(kmax, key[i]);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, o, 64));
    kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o, 64));
  }
  s.hist[t] = 0;
  if (lane == 0) {
    s.lo[t >> 6] = kmin;
    s.hi[t >> 6] = kmax;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kTWaves; ++w) {
    kmin = min(kmin, s.lo[w]);
    kmax = max(kmax, s.hi[w]);
  }
  // bins of 2^sh keys: the range's top 8 bits
  const int sh = kmax > kmin ? max(0, 24 - __clz((int)(kmax - kmin))) : 0;
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (key[i] >= kFirstKey) atomicAdd(&s.hist[(key[i] - kmin) >> sh], 1);
  __syncthreads();
  // lane l: bins 255 - 4 l down to 252 - 4 l, the largest keys in lane 0
  int n[4], sum = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    n[j] = s.hist[255 - 4 * lane - j];
    sum += n[j];
  }
  int incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o, 64);
    if (lane >= o) incl += y;
  }
  const unsigned long long enough = __ballot(incl >= want);
  __syncthreads();  // the buffers are free again
  if (!enough) return Bracket{0u, kFirstKey, 0};
  int c = incl - sum, bin = 255 - 4 * lane;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (c < want) {
      c += n[j];
      bin = 255 - 4 * lane - j;
    }
  const int from = __ffsll(enough) - 1;
  c = __shfl(c, from, 64);
  bin = __shfl(bin, from, 64);
  const unsigned long long hi = (unsigned long long)kmin + ((unsigned long long)(bin + 1) << sh);
  return Bracket{kmin + ((uint32_t)bin << sh), hi > 0xffffffffull ? 0xffffffffu : (uint32_t)hi, c};
}

// A bound t such that at least `want` and at most about `most` of the
// workgroup's keys are >= t (exactly the want-th largest key when most ==
// want, unless ties make more), or 0 when fewer than `want` are finite: the
// bracket, halved (a count of the workgroup per step) while it holds more.
template <int N>
__device__ __forceinline__ uint32_t block_bound(const uint32_t (&key)[N], int want, int most, BracketLds& s_br,
                                                int (*s_cnt)[kTWaves]) {
  Bracket br = block_bracket<N>(key, want, s_br);
  int par = 0;
  while (br.c > most && br.hi - br.lo > 1) {
    const uint32_t mid = br.lo + (br.hi - br.lo) / 2;
    int c = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) c += __popcll(__ballot(key[i] >= mid));
    if ((threadIdx.x & 63) == 0) s_cnt[par][threadIdx.x >> 6] = c;
    __syncthreads();
    int n = 0;
#pragma unroll
    for (int w = 0; w < kTWaves; ++w) n += s_cnt[par][w];
    par ^= 1;  // the next count writes the other buffer: one barrier per step
    if (n >= want) br.lo = mid, br.c = n;
    else br.hi = mid;
  }
  __syncthreads();  // the buffers are free again
  return br.lo;
}

// The decision, the race over the raced row's kept list and the commit of one
// sequence (decide_seq and finalize_seq of verify_sample.hip on the short
// form), in the workgroup that completed its rows.
template <bool UNIT>
__device__ void finish_sequence(const TkArgs& a, int b) {
  const int gamma = a.d.gamma, C = gamma + 1, nr = 2 * gamma + 1, V = a.d.V, t = threadIdx.x;
  __shared__ RowDesc s_d[2 * 32 + 1];
  __shared__ float s_u[32];
  __shared__ int s_x[32];
  __shared__ int s_k, s_flag;
  int bad = 0, amb = 0;
  if (t < gamma) {
    s_x[t] = a.d.proposals[(size_t)b * gamma + t];
    s_u[t] = a.d.u[(size_t)b * gamma + t];
  }
  int rem = 0, st = 0;
  if (t == 0) {
    if (a.c.remaining) rem = a.c.remaining[b];
    if (a.c.start) st = a.c.start[b];
  }
  if (t < nr) {
    const __amdgpu_buffer_rsrc_t rd = coherent_rsrc(a.desc);
    const size_t o = ((size_t)b * nr + t) * sizeof(RowDesc);
    const u32x4_t lo = load_coherent_b128(rd, o), hi = load_coherent_b128(rd, o + 16);
    s_d[t] = RowDesc{__uint_as_float(lo.x), __uint_as_float(lo.y), __uint_as_float(lo.z), (int)lo.w,
                     (int)hi.x,             hi.y,                  (int)hi.z,             (int)hi.w};
    bad = (int)hi.w;
    amb = (int)hi.x;
  }
  if (t >= kTThreads - a.pieces) {  // the noise row's pieces
    const size_t o = (((size_t)b * (nr + 1) + nr) * a.pieces + (t - (kTThreads - a.pieces))) * sizeof(int2);
    bad |= (int)load_coherent_b64(coherent_rsrc(a.counts), o).x;
  }
  bad = __syncthreads_or(bad);
  amb = __syncthreads_or(amb);
  if (bad) {
    if (t == 0) a.need[b] = 1;
    return;
  }
  if (t == 0) {
    int k = gamma, flag = 0;
    for (int j = 0; j < gamma; ++j) {
      const RowDesc &p = s_d[j], &q = s_d[C + j];
      float pp = 0.f, qq = 0.f;
      const bool in = (unsigned)s_x[j] < (unsigned)V;
      if (in) {
        pp = softmax_at(p.zx, p.M, p.S, 1.f);
        qq = softmax_at(q.zx, q.M, q.S, 1.f);
      }
      const double qd = (double)qq, pd = (double)pp, u = (double)s_u[j];
      const double acc = qd <= kEps ? (pd > kEps ? 1.0 : 0.0) : fmin(1.0, pd / qd);
      if (in && decision_in_band(pd, qd, u, kDecideRel)) flag |= SPV_FLAG_ACCEPT_BAND;
      if (!(u < acc)) {
        k = j;
        break;
      }
    }
    s_k = k;
    s_flag = flag;
  }
  __syncthreads();
  const int k = s_k;
  const bool resid = k < gamma;
  const RowDesc pd = s_d[k], qd = s_d[resid ? C + k : k];
  // p, q and the residual of the kept tokens: p is 0 everywhere else, so the
  // residual and its key are too.
  constexpr int kItems = kKeepCap / kTThreads;
  const float* qrow = resid ? a.d.draft + ((size_t)b * gamma + k) * V : nullptr;
  const float* noise = a.c.noise + (size_t)b * V;
  const __amdgpu_buffer_rsrc_t rl = coherent_rsrc(a.lists);
  const size_t lbase = ((size_t)b * nr + k) * a.pieces * kPieceCap * sizeof(uint2);
  float p[kItems], q[kItems], e[kItems];
  int idx[kItems];
  u32x2_t ent[kItems];
#pragma unroll
  for (int i = 0; i < kItems; ++i)
    if (t + i * kTThreads < pd.n) ent[i] = load_coherent_b64(rl, lbase + (size_t)(t + i * kTThreads) * sizeof(uint2));
  double rs = 0.0, ps = 0.0;
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    p[i] = q[i] = 0.f;
    e[i] = 1.f;
    idx[i] = 0x7fffffff;
    if (t + i * kTThreads >= pd.n) continue;
    idx[i] = (int)ent[i].y;
    e[i] = noise[idx[i]];
    p[i] = softmax_at(__uint_as_float(ent[i].x), pd.M, pd.S, 1.f);
    if (resid) {
      const float xq = UNIT ? qrow[idx[i]] : qrow[idx[i]] / a.d.tf;
      const uint32_t key = order_key(xq);
      if (key > qd.last_key || (key == qd.last_key && idx[i] <= qd.last_idx)) q[i] = softmax_at(xq, qd.M, qd.S, 1.f);
    }
    const float d = p[i] - q[i];
    rs += (double)(d < 0.f ? 0.f : d);
    ps += (double)p[i];
  }
  rs = block_sum_f64(rs);
  ps = block_sum_f64(ps);
  const float tot = (float)rs, psum = fmaxf((float)ps, 1e-12f);
  // the residual's normaliser, p's where the residual is empty; the bonus row
  // is raced as it is (specdec/sampler.py:72-83)
  const bool empty = resid && (double)tot <= kEps;
  const float div = !resid ? 1.f : empty ? psum : tot;
  Top1 t1;
  t1.init();
#pragma unroll
  for (int i = 0; i < kItems; ++i) {
    if (t + i * kTThreads >= pd.n) continue;
    const float d = resid && !empty ? p[i] - q[i] : p[i];
    const float rhat = resid ? (d < 0.f ? 0.f : d) / div : d;
    const float key = rhat / e[i];
    const float err = fmaf(kProbRel, p[i], resid && !empty ? kProbRel * q[i] : 0.f);
    const float hi = fmaxf(d + err, 0.f) / (div * e[i]);
    t1.merge(key, fmaxf(fmaf(key, kExactRel, key), fmaf(hi, kExactRel, hi)), -INFINITY, idx[i]);
  }
  block_top1(t1);
  if (!(t1.v > 0.f)) {  // no kept token's key stands out from the others' zeros
    if (t == 0) a.need[b] = 1;
    return;
  }
  if (t < C) a.d.out_tokens[(size_t)b * C + t] = t < k ? s_x[t] : t == k ? t1.i : -1;
  if (t == 0) {
    a.need[b] = 0;
    a.d.accept_len[b] = k;
    if (a.d.flags)
      a.d.flags[b] = s_flag | (t1.certain(0.f) ? 0 : SPV_FLAG_DRAW_BAND) | (amb ? SPV_FLAG_TOP_P_BAND : 0);
    commit_cut(a.d, a.c, b, k, t1.i, s_x, rem, st);
  }
}

// Sum of one int per thread over the workgroup.
__device__ __forceinline__ int block_sum(int v, int (*s_cnt)[kTWaves]) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) s_cnt[0][threadIdx.x >> 6] = v;
  __syncthreads();
  int n = 0;
#pragma unroll
  for (int w = 0; w < kTWaves; ++w) n += s_cnt[0][w];
  __syncthreads();
  return n;
}

// grid: per sequence (2 gamma + 1) rows and the noise row, `pieces` workgroups
// each; sequences one after another.
template <int NVEC, bool VEC, bool UNIT>
__global__ __launch_bounds__(kTThreads, NVEC == kVecMid ? 4 : 2) void topk_sample_kernel(TkArgs a) {
  constexpr int kCap = row_cap(NVEC);
  constexpr int kGroups = NVEC != kVecSmall ? 4 : 5, kPer = NVEC / kGroups;  // group maxima per thread
  static_assert(NVEC % kGroups == 0 && kGroups * kTThreads >= 2 * kTopkMax, "enough group maxima for any top_k");
  const int gamma = a.d.gamma, C = gamma + 1, nr = 2 * gamma + 1, V = a.d.V, P = a.pieces, t = threadIdx.x;
  const int b = blockIdx.x / ((nr + 1) * P), rem = blockIdx.x - b * (nr + 1) * P, r = rem / P, pc = rem - r * P;
  __shared__ unsigned long long s_row[kCap];  // the piece's candidates, then the row's
  __shared__ unsigned long long s_keep[kKeepCap];
  __shared__ int s_cnt[2][kTWaves];
  __shared__ BracketLds s_br;
  __shared__ double s_scan[kTWaves];
  __shared__ float s_zx;
  __shared__ int s_n, s_last;
  const float* src = r < C ? a.d.target + ((size_t)b * C + r) * V
                     : r < nr ? a.d.draft + ((size_t)b * gamma + (r - C)) * V : a.c.noise + (size_t)b * V;
  // this piece: n values from i0 on, n4 whole float4 when rows are made of them
  int i0, n;
  if (VEC) {
    const int nv = V >> 2, j0 = (int)((long long)nv * pc / P);
    i0 = 4 * j0;
    n = 4 * ((int)((long long)nv * (pc + 1) / P) - j0);
  } else {
    i0 = (int)((long long)V * pc / P);
    n = (int)((long long)V * (pc + 1) / P) - i0;
  }
  // Loads past the piece return zero without a memory access; those values
  // are made -inf (noise: 1). Element (k, e) of a thread is value 4 (t + 256 k)
  // + e of the piece, or t + 256 (4 k + e) when rows are not whole float4.
  const __amdgpu_buffer_rsrc_t rs = span_rsrc(src + i0, (uint32_t)n * 4u);
  u32x4_t v[NVEC];
#pragma unroll
  for (int k = 0; k < NVEC; ++k) {
    if (VEC) {
      v[k] = load_b128(rs, t * 16u, (uint32_t)k * kTThreads * 16u);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[k][e] = load_b32(rs, t * 4u, (uint32_t)(4 * k + e) * kTThreads * 4u);
    }
  }
  auto index = [&](int k, int e) { return VEC ? 4 * (t + kTThreads * k) + e : t + kTThreads * (4 * k + e); };
  const uint32_t pad = __float_as_uint(r < nr ? -INFINITY : 1.f);
#pragma unroll
  for (int k = 0; k < NVEC; ++k)
    if (4 * kTThreads * (k + 1) > n) {  // uniform: this step reaches past the piece
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (index(k, e) >= n) v[k][e] = pad;
    }
  const __amdgpu_buffer_rsrc_t rc = coherent_rsrc(a.counts), rl = coherent_rsrc(a.lists);
  const size_t crow = ((size_t)b * (nr + 1) + r) * P;

  if (r == nr) {
    // the noise row: whether every entry is above zero, as Exp(1) noise is
    bool bad = false;
#pragma unroll
    for (int k = 0; k < NVEC; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= !(__uint_as_float(v[k][e]) > 0.f);
    const int any = __syncthreads_or(bad);
    if (t == 0) store_coherent_b64(rc, (crow + pc) * sizeof(int2), u32x2_t{(unsigned)any, 0u});
  } else {
    // 1. the piece's candidates
    uint32_t gk[kGroups];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      float m = -INFINITY;
#pragma unroll
      for (int k = g * kPer; k < (g + 1) * kPer; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, __uint_as_float(v[k][e]));
      gk[g] = order_key(m);
    }
    if (t == 0) s_n = 0;
    const uint32_t bound = block_bound<kGroups>(gk, a.top_k, a.top_k + a.top_k / 16 + 16, s_br, s_cnt);
    // On the raw logits: lowered so that no logit whose quotient by T rounds to
    // the bound's is left out (2 ulp of the quotient; the constant covers
    // quotients that underflow).
    float z0 = bound ? key_value(bound) : -INFINITY;
    if (!UNIT) z0 = z0 - fabsf(z0) * 0x1p-20f - 1e-30f;
    z0 = fmaxf(z0, -3.402823466e38f);  // -inf is no candidate
#pragma unroll
    for (int k = 0; k < NVEC; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float z = __uint_as_float(v[k][e]);
        if (!(z < z0)) {  // a NaN is a candidate
          const int at = atomicAdd(&s_n, 1);
          if (at < kPieceCap) s_row[at] = (unsigned long long)(uint32_t)(i0 + index(k, e)) << 32 | v[k][e];
        }
      }
    __syncthreads();
    const int nc = s_n;
    const size_t lrow = ((size_t)b * nr + r) * P * kPieceCap;  // the row's lists
    if (nc <= kPieceCap)
      for (int i = t; i < nc; i += kTThreads) {
        const unsigned long long c = s_row[i];
        store_coherent_b64(rl, (lrow + (size_t)pc * kPieceCap + i) * sizeof(uint2),
                           u32x2_t{(unsigned)c, (unsigned)(c >> 32)});
      }
    if (t == 0) store_coherent_b64(rc, (crow + pc) * sizeof(int2), u32x2_t{(unsigned)(nc <= kPieceCap ? nc : -1), 0u});
    if (!arrive_last(a.cnt_row + (size_t)b * nr + r, P, &s_last)) return;

    // 2. the row: every piece's candidates, scaled. 256 / P threads take a piece;
    // its count and their first kAhead entries come in one round trip (what lies
    // past the count is dropped).
    constexpr int kAhead = 4;
    const int tp = kTThreads / P, q = t / tp, sub = t - q * tp;
    const size_t lpiece = lrow + (size_t)min(q, P - 1) * kPieceCap;
    int pn = (int)load_coherent_b64(rc, (crow + min(q, P - 1)) * sizeof(int2)).x;
    u32x2_t ahead[kAhead];
#pragma unroll
    for (int e = 0; e < kAhead; ++e) ahead[e] = load_coherent_b64(rl, (lpiece + sub + e * tp) * sizeof(uint2));
    const int j = r < gamma ? r : r >= C ? r - C : -1;  // the row's proposal
    const int xj = j >= 0 ? a.d.proposals[(size_t)b * gamma + j] : -1;
    if (t == 0) {
      s_n = 0;
      s_zx = -INFINITY;
    }
    __syncthreads();
    bool odd = false;
    auto take = [&](const u32x2_t& c) {
      const float z = __uint_as_float(c.x), x = UNIT ? z : z / a.d.tf;
      odd |= !(fabsf(x) < INFINITY);  // NaN, or infinite
      const int at = atomicAdd(&s_n, 1);
      if (at < kCap) s_row[at] = pack_entry(order_key(x), (int)c.y);
    };
    if (q < P) {
      odd |= pn < 0;
#pragma unroll
      for (int e = 0; e < kAhead; ++e)
        if (sub + e * tp < pn) take(ahead[e]);
      for (int i = sub + kAhead * tp; i < pn; i += tp) take(load_coherent_b64(rl, (lpiece + i) * sizeof(uint2)));
    }
    bool bad = __syncthreads_or(odd);
    const int total = s_n;
    bad |= total < 1 || total > kCap;
    RowDesc out{};
    if (!bad) {
      // What is at or above the k-th largest. The entries from the bracket's
      // lower end on (a few more than k) are sorted, and the k-th of them is
      // the threshold; where the lists do not hold them the exact bound is
      // searched first.
      uint32_t thr = 0;
      int held;  // entries >= thr
      auto bracket = [&](auto& key, bool exact) {
        constexpr int N = sizeof(key) / sizeof(key[0]);
#pragma unroll
        for (int i = 0; i < N; ++i) key[i] = t + i * kTThreads < total ? entry_key(s_row[t + i * kTThreads]) : 0u;
        if (exact) {
          thr = block_bound<N>(key, a.top_k, a.top_k, s_br, s_cnt);
          return;
        }
        const Bracket br = block_bracket<N>(key, a.top_k, s_br);
        thr = br.lo;
        held = br.lo ? br.c : total;
      };
      auto find = [&](bool exact) {
        if (total <= 4 * kTThreads) {
          uint32_t key[4];
          bracket(key, exact);
        } else {
          uint32_t key[kCap / kTThreads];
          bracket(key, exact);
        }
      };
      find(false);
      if (held > kKeepCap) find(true);
      thr = with_both_zeros(thr);
      if (t == 0) s_n = 0;
      __syncthreads();
      for (int i = t; i < total; i += kTThreads) {
        const unsigned long long c = s_row[i];
        if (entry_key(c) >= thr) {
          const int at = atomicAdd(&s_n, 1);
          if (at < kKeepCap) s_keep[at] = c;
        }
      }
      __syncthreads();
      int nk = s_n;
      bad = nk > kKeepCap;
      if (!bad) {
        // sorted by value, equal values by index: every entry's rank
        for (int i = t; i < nk; i += kTThreads) {
          const unsigned long long c = s_keep[i];
          int rank = 0;
          for (int q = 0; q < nk; ++q) rank += s_keep[q] > c;
          s_row[rank] = c;
        }
        __syncthreads();
        if (thr && nk > a.top_k) {  // cut at the k-th value; its ties stay
          const uint32_t kth = with_both_zeros(entry_key(s_row[a.top_k - 1]));
          int ties = 0;
          for (int i = a.top_k + t; i < nk; i += kTThreads) ties += entry_key(s_row[i]) >= kth;
          nk = a.top_k + block_sum(ties, s_cnt);
        }
        const float M = key_value(entry_key(s_row[0]));
        int keep = nk, amb = 0;
        const int per = (nk + kTThreads - 1) / kTThreads, q0 = min(nk, t * per), q1 = min(nk, q0 + per);
        if (a.top_p > 0.f && a.top_p < 1.f) {
          // the nucleus: a value stays while the mass before it is below p W
          double mine = 0.0, W;
          for (int q = q0; q < q1; ++q) mine += key_mass(entry_key(s_row[q]), M);
          double before = block_exclusive_scan_f64(mine, s_scan, &W);
          const double tgt = (double)a.top_p * W, lo = tgt - kTopPWindow * W, hi = tgt + kTopPWindow * W;
          int kept = 0, near = 0;
          for (int q = q0; q < q1; ++q) {
            kept += before < tgt;
            near += before >= lo && before < hi;
            before += key_mass(entry_key(s_row[q]), M);
          }
          // the masses before them rise with the rank: the kept values come first
          keep = max(1, block_sum(kept, s_cnt));
          amb = block_sum(near, s_cnt);
        }
        // the kept values' softmax normaliser; the kept list; the value at the proposal
        double S = 0.0;
        for (int i = t; i < keep; i += kTThreads) {
          const unsigned long long c = s_row[i];
          const float x = key_value(entry_key(c));
          S += (double)exp2f((x - M) * kLog2e);
          if (r < C)
            store_coherent_b64(rl, (lrow + i) * sizeof(uint2), u32x2_t{__float_as_uint(x), (unsigned)entry_idx(c)});
          if (entry_idx(c) == xj) s_zx = x;
        }
        S = block_sum_f64(S);  // (its barriers publish s_zx)
        const unsigned long long last = s_row[keep - 1];
        out = RowDesc{M, (float)S, s_zx, keep, amb, entry_key(last), entry_idx(last), 0};
      }
    }
    if (t == 0) {
      out.bad = bad;
      const __amdgpu_buffer_rsrc_t rd = coherent_rsrc(a.desc);
      const size_t o = ((size_t)b * nr + r) * sizeof(RowDesc);
      store_coherent_b128(rd, o, u32x4_t{__float_as_uint(out.M), __float_as_uint(out.S), __float_as_uint(out.zx),
                                         (unsigned)out.n});
      store_coherent_b128(rd, o + 16, u32x4_t{(unsigned)out.amb, out.last_key, (unsigned)out.last_idx,
                                              (unsigned)out.bad});
    }
  }
  // 3. rows and noise pieces that are done; the last one finishes the sequence
  if (arrive_last(a.cnt_seq + b, nr + P, &s_last)) finish_sequence<UNIT>(a, b);
}

// ------------------------------------------------------------------ host side
int ceil_of(int a, int b) { return (a + b - 1) / b; }

// The short form's split of a row, or 0 when it does not take the call.
struct TkPlan {
  int pieces, nvec;
};
TkPlan tk_plan(int B, int gamma, int V, float temperature, int top_k) {
  const long long rows = (long long)B * (2 * gamma + 1);
  if (top_k < 1 || top_k > kTopkMax || top_k >= V || rows > kMaxRows || !(temperature >= kTempMin) ||
      !(temperature <= kTempMax))
    return {0, 0};
  // candidates of a row over n pieces, with a third to spare
  auto fits = [&](int n, int nvec) {
    return n <= kMaxPieces && (long long)n * (top_k + top_k / 16 + 16) * 4 / 3 <= row_cap(nvec) &&
           rows * n * kPieceCap * sizeof(uint2) <= kMaxListBytes;
  };
  // One float4 less than the registers hold per thread, so that an uneven cut fits.
  auto pieces = [&](int nvec) { return ceil_of(V, 4 * kTThreads * nvec - 4); };
  const int small = pieces(kVecSmall), mid = pieces(kVecMid), big = pieces(kVecBig);
  if (fits(small, kVecSmall) && rows * small <= 1024) return {small, kVecSmall};
  if (fits(mid, kVecMid)) return {mid, kVecMid};
  if (fits(big, kVecBig)) return {big, kVecBig};
  return {0, 0};
}

constexpr size_t kTkCounterBytes = ((size_t)kMaxRows + 65536) * sizeof(int);

// Workspace: the short form's counters and spv_verify_sample's (both at fixed
// offsets, zero between calls, whatever the shape), then the rest.
struct TkLayout {
  size_t sample, need, amb, counts, desc, lists, total;
};
TkLayout tk_layout(int B, int gamma, int V, const TkPlan& pl) {
  TkLayout l{};
  size_t off = kTkCounterBytes;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off += (bytes + 255) & ~(size_t)255;
    return o;
  };
  const size_t rows = (size_t)B * (2 * gamma + 1);
  l.sample = take(spv_verify_sample_workspace_bytes(B, gamma, V));
  l.need = take((size_t)B * sizeof(int32_t));
  l.amb = take(rows * sizeof(int32_t));
  l.counts = take((rows + B) * pl.pieces * sizeof(int2));
  l.desc = take(rows * sizeof(RowDesc));
  l.lists = take(rows * pl.pieces * kPieceCap * sizeof(uint2));
  l.total = off;
  return l;
}

template <int NVEC>
void launch_tk(const TkArgs& a, int grid, hipStream_t s) {
  const bool unit = a.d.tf == 1.0f;
  if (a.d.V & 3) {
    if (unit) hipLaunchKernelGGL((topk_sample_kernel<NVEC, false, true>), dim3(grid), dim3(kTThreads), 0, s, a);
    else hipLaunchKernelGGL((topk_sample_kernel<NVEC, false, false>), dim3(grid), dim3(kTThreads), 0, s, a);
  } else {
    if (unit) hipLaunchKernelGGL((topk_sample_kernel<NVEC, true, true>), dim3(grid), dim3(kTThreads), 0, s, a);
    else hipLaunchKernelGGL((topk_sample_kernel<NVEC, true, false>), dim3(grid), dim3(kTThreads), 0, s, a);
  }
}

}  // namespace

extern "C" {

size_t spv_verify_sample_filtered_workspace_bytes(int32_t B, int32_t gamma, int32_t V, float temperature,
                                                  int32_t top_k) {
  if (spv_verify_sample_workspace_bytes(B, gamma, V) == 0) return 0;
  return tk_layout(B, gamma, V, tk_plan(B, gamma, V, temperature, top_k)).total;
}

int spv_verify_sample_filtered(const float* target, const float* draft, float temperature, int32_t top_k, float top_p,
                               const int32_t* proposals, const float* u_accept, const float* exp_noise,
                               const int32_t* start_pos, const int32_t* remaining, int32_t eos_id, int32_t B,
                               int32_t gamma, int32_t V, int32_t* accept_len, int32_t* out_tokens, int32_t* n_commit,
                               int32_t* finished, int32_t* new_len, int32_t* flags, float* target_scratch,
                               float* draft_scratch, void* workspace, size_t workspace_bytes, void* stream) {
  if (!target || !draft || !proposals || !u_accept || !exp_noise || !accept_len || !out_tokens || !target_scratch ||
      !draft_scratch || B < 0 || B > 65535 || gamma < 1 || gamma > 32 || V < 1 || !(temperature > 0.f) ||
      (size_t)V * 4 > 0x7fffffffu || (long long)B * (2 * gamma + 1) > 0x7fffffffLL)
    return SPV_ERR_ARG;
  if (B == 0) return SPV_OK;
  const TkPlan pl = tk_plan(B, gamma, V, temperature, top_k);
  const TkLayout l = tk_layout(B, gamma, V, pl);
  if (!workspace || workspace_bytes < l.total) return SPV_ERR_WORKSPACE;
  char* ws = static_cast<char*>(workspace);
  const int rows = B * (2 * gamma + 1);
  int32_t* amb_t = top_p > 0.f && top_p < 1.f ? reinterpret_cast<int32_t*>(ws + l.amb) : nullptr;
  int32_t* amb_d = amb_t ? amb_t + (size_t)B * (gamma + 1) : nullptr;
  int32_t* need = nullptr;
  if (pl.pieces) {
    TkArgs a{};
    a.d.target = target;
    a.d.draft = draft;
    a.d.proposals = proposals;
    a.d.u = u_accept;
    a.d.accept_len = accept_len;
    a.d.out_tokens = out_tokens;
    a.d.flags = flags;
    a.d.B = B;
    a.d.gamma = gamma;
    a.d.V = V;
    a.d.tf = temperature_divisor(temperature);
    a.c = CommitArgs{start_pos, remaining, exp_noise, eos_id, n_commit, finished, new_len};
    a.pieces = pl.pieces;
    a.top_k = top_k;
    a.top_p = top_p;
    need = a.need = reinterpret_cast<int32_t*>(ws + l.need);
    a.cnt_row = reinterpret_cast<int*>(ws);
    a.cnt_seq = a.cnt_row + kMaxRows;
    a.counts = reinterpret_cast<int2*>(ws + l.counts);
    a.lists = reinterpret_cast<uint2*>(ws + l.lists);
    a.desc = reinterpret_cast<RowDesc*>(ws + l.desc);
    const int grid = (rows + B) * pl.pieces;
    if (pl.nvec == kVecBig) launch_tk<kVecBig>(a, grid, (hipStream_t)stream);
    else if (pl.nvec == kVecMid) launch_tk<kVecMid>(a, grid, (hipStream_t)stream);
    else launch_tk<kVecSmall>(a, grid, (hipStream_t)stream);
    SPV_CHECK_LAUNCH();
  }
  // the general path: every sequence, or those the short form left
  int rc = filter_verify_rows(target, target_scratch, amb_t, draft, draft_scratch, amb_d, need, B, gamma, V,
                              temperature, top_k, top_p, stream);
  if (rc != SPV_OK) return rc;
  return verify_sample_impl(target_scratch, draft_scratch, 0, 1.f, proposals, u_accept, exp_noise, nullptr, start_pos,
                            remaining, eos_id, B, gamma, V, accept_len, out_tokens, n_commit, finished, new_len,
                            nullptr, flags, 0, need, amb_t, amb_d, ws + l.sample, workspace_bytes - l.sample, stream);
}

}  // extern "C"
