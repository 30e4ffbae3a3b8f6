// nls_rowsplit.hip -- softmaxInPlace (sampler.nim:51-57), logProb's and
// perplexity's per-position terms and the sum of topTokens, with every row
// split over slices of 4096 logits, one 256-thread workgroup each.
//
// The one-launch kernels (nls_softmax.hip, nls_kernels.hip) give a row one
// workgroup on one CU.  Its passes then run one after the other (the maximum:
// bound by the requests one CU keeps in flight; the exponentials: by float64
// issue; the sum: by the latency of its windows), and fewer rows than CUs
// leave the rest of the chip idle.  Here the launches are:
//   A. split_max_kernel: the maximum m of each 1024 logits (a wave's) and an
//      estimate a of their sum exp(l - m) (v_exp_f32), one read of the row.
//   B. split_terms_kernel: mx = the largest m.  The reference's index-order
//      fp32 sum s of exp(l - mx) is a scan of parity maps (nls_seqsum.h) once
//      the running sum's binade is known, so each group of 256 terms takes
//      the binade of its estimated running sum (the a of the waves' logits
//      below, this wave's own terms) and stores its map for that binade.
//      A term's part of a map is round(e / u), u the binade's spacing.  An
//      fp32 estimate y of e (|y - e| <= kSplitErr e) settles it unless y / u
//      lies within kSplitErr y / u of a half; only those terms (about 1 in
//      16,000) take the correctly rounded exponential, whose float64
//      arithmetic bounded the one-launch kernels' sum.
//   C. split_walk_kernel: a workgroup per row walks the maps with the exact
//      sum.  A group's map is used when its binade is the sum's and the sum
//      stays in it; any other group (it crosses a binade, or the estimate was
//      off) is replayed from its exact terms.  An estimate therefore only
//      costs time, never a bit.  logProb ends here.
//   D. softmax: exp(l - mx) / s for every element (split_out_kernel).
//      topTokens: the entries B listed, in order (top_tokens_kernel<true>).
//      perplexity: B sums float64 exponentials as row_nll_kernel's waves do, C
//      adds the waves' sums.
// The launches hand over through memory: an arrival count per row with the
// walk in its last slice (agent-scope fences, or write-through stores and a
// wait) cost 30 us of 256 x 128256's 95 us in launch B.
// Measured, one pass, one launch -> split: topTokens, n = 5, 32 x 128256 146 -> 40 us;
// softmax 256 x 128256 187 -> 152, 1 x 128256 151 -> 27; logProb 201 x 50001 66 -> 44,
// 1 x 50001 61 -> 27; perplexity's term 8 x 128256 36 -> 12.  Of softmax's 152 us (traced):
// A 21, B 59 (about 500 vector instructions a wave, 28 us at full issue), C 21
// (latency of one wave), D 43 (262 MB at 6.1 TB/s).
#include "nls_device.h"
#include "nls_exp64.h"
#include "nls_rowsplit.h"
#include "nls_seqsum.h"

namespace nls {

namespace {

constexpr int kNT = kSplitNT;
constexpr int kPer = kSplitSlice / kNT;          // logits per thread
constexpr int kGpw = kPer / 4;                   // groups of 256 per wave
constexpr int kGroup = 4 * kWave;                // 256 consecutive logits, four per lane
constexpr int kWpb = kNT / kWave;
constexpr int kHeadGroups = 1;                   // the row's first group is added one term at a time
constexpr int kWalkNT = 1024;                    // groups per round of the walk, one per thread
constexpr int kSlots = kWalkNT / kWave - 1;      // crossing groups prepared per round, one per wave
                                                 // (the last wave adds the row's first group)
constexpr int kManyLanes = 24;                   // topTokens: lanes with a logit to list, of a wave that looks for
                                                 // a bound of its own
constexpr float kLog2e = 1.44269502162933349609375f;

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

// four consecutive logits; absent ones read as -inf (terms of exactly zero).
// Rows may start off 16 bytes: the load is 4-byte aligned then.
__device__ __forceinline__ f32x4 load4(const float* x, int i, int n) {
  f32x4 v;
  if (i + 4 <= n) {
    __builtin_memcpy(&v, x + i, 16);
  } else {
    const float none = -__builtin_inff();
    v.x = i < n ? x[i] : none;
    v.y = i + 1 < n ? x[i + 1] : none;
    v.z = i + 2 < n ? x[i + 2] : none;
    v.w = none;
  }
  return v;
}

// This wave's groups: g * 256 + 4 * lane .. of each from element i0 on.
__device__ __forceinline__ void load_groups(const float* x, int i0, int n, f32x4 (&v)[kGpw]) {
  const int i = i0 + 4 * lane_id();
  if (i0 + kGpw * kGroup <= n) {  // wave-uniform: all but a row's last wave
#pragma unroll
    for (int g = 0; g < kGpw; ++g) __builtin_memcpy(&v[g], x + i + g * kGroup, 16);
  } else {
#pragma unroll
    for (int g = 0; g < kGpw; ++g) v[g] = load4(x, i + g * kGroup, n);
  }
}

template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_or(float v, float none) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(none), __float_as_int(v), CTRL, ROWS, 0xf, false));
}
// the wave's sum / maximum, in every lane
__device__ __forceinline__ float wave_sum_f(float v) {
  v += dpp_or<0x111, 0xf>(v, 0.0f);  // row_shr 1, 2, 4, 8
  v += dpp_or<0x112, 0xf>(v, 0.0f);
  v += dpp_or<0x114, 0xf>(v, 0.0f);
  v += dpp_or<0x118, 0xf>(v, 0.0f);
  v += dpp_or<0x142, 0xa>(v, 0.0f);  // row_bcast 15, 31
  v += dpp_or<0x143, 0xc>(v, 0.0f);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// (lane 15 of each row of 16 holds the row's maximum in `row`)
__device__ __forceinline__ float wave_max_f(float v, float& row) {
  const float none = -__builtin_inff();
  v = __builtin_fmaxf(v, dpp_or<0x111, 0xf>(v, none));
  v = __builtin_fmaxf(v, dpp_or<0x112, 0xf>(v, none));
  v = __builtin_fmaxf(v, dpp_or<0x114, 0xf>(v, none));
  v = __builtin_fmaxf(v, dpp_or<0x118, 0xf>(v, none));
  row = v;
  v = __builtin_fmaxf(v, dpp_or<0x142, 0xa>(v, none));
  v = __builtin_fmaxf(v, dpp_or<0x143, 0xc>(v, none));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// Four sums over the wave at once, each in every lane: lanes of a quad keep
// one value each after two exchanges, so one chain of four steps serves all.
__device__ __forceinline__ void wave_sum4(float (&v)[4]) {
  const int lane = lane_id();
  const bool odd = lane & 1, hi = (lane & 2) != 0;
  const float a0 = (odd ? v[1] : v[0]) + dpp_or<0xB1, 0xf>(odd ? v[0] : v[1], 0.0f);  // quad_perm 1,0,3,2
  const float a1 = (odd ? v[3] : v[2]) + dpp_or<0xB1, 0xf>(odd ? v[2] : v[3], 0.0f);
  float t = (hi ? a1 : a0) + dpp_or<0x4E, 0xf>(hi ? a0 : a1, 0.0f);                   // quad_perm 2,3,0,1
  t += dpp_or<0x114, 0xf>(t, 0.0f);  // row_shr 4, 8: lanes 12..15 of each row hold its sums
  t += dpp_or<0x118, 0xf>(t, 0.0f);
  const int b = __float_as_int(t);
#pragma unroll
  for (int k = 0; k < 4; ++k)
    v[k] = (__int_as_float(__builtin_amdgcn_readlane(b, 12 + k)) + __int_as_float(__builtin_amdgcn_readlane(b, 28 + k))) +
           (__int_as_float(__builtin_amdgcn_readlane(b, 44 + k)) + __int_as_float(__builtin_amdgcn_readlane(b, 60 + k)));
}

// A group's map in 64 bits: a and c with increments clamped at 2^24 (any such
// increment leaves the binade), the binade's code, and whether the estimates
// say the group crosses into another binade.
constexpr int kCodeAny = 254;   // no term but zeros: the map of every binade
constexpr int kCodeBias = 126;  // code = E + 126
__device__ __forceinline__ uint64_t pack_map(SeqMap m, int code, bool cross) {
  const uint32_t a = ((uint32_t)min(m.a >> 1, 1 << 24) << 1) | (m.a & 1);
  const uint32_t c = ((uint32_t)min(m.c >> 1, 1 << 24) << 1) | (m.c & 1);
  return (uint64_t)a | ((uint64_t)c << 26) | ((uint64_t)(uint32_t)code << 52) | ((uint64_t)cross << 60);
}
__device__ __forceinline__ SeqMap unpack_map(uint64_t u) {
  return SeqMap{(int)(u & 0x3ffffffu), (int)((u >> 26) & 0x3ffffffu)};
}
__device__ __forceinline__ int unpack_code(uint64_t u) { return (int)((u >> 52) & 0xff); }

struct RowWork {  // one row's part of the workspace
  uint64_t* maps;   // [ns * 16] (nll: 16 float64 sums)
  float2* part;     // [np]: m and a of each wave's 1024 logits
  int np;
  SplitRowInfo* info;
  float* gmax;      // [ns * 16], topTokens: maxima of 256 logits each
  uint64_t* list;   // [kSplitList], topTokens: key << 32 | index
};
__device__ __forceinline__ RowWork row_work(const SplitArgs& a, int row) {
  RowWork w;
  w.maps = a.maps + (int64_t)row * a.ns * kSplitGroups;
  w.np = a.ns * kWpb;
  w.part = a.part + (int64_t)row * w.np;
  w.info = a.info + row;
  w.gmax = a.gmax + (int64_t)row * a.ns * kSplitGroups;
  w.list = a.list + (int64_t)row * kSplitList;
  return w;
}

// The correctly rounded exponentials of four differences l - mx (<= 0, or NaN).
__device__ __forceinline__ void exact_terms(const float (&d)[4], const double* pow2, float (&e)[4]) {
  bool all = true;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    bool ok;
    e[j] = expf_cr_quick(d[j], pow2, ok);
    all = all && ok;
  }
  if (!all) {
#pragma unroll 1
    for (int j = 0; j < 4; ++j) {
      const float t = expf_cr_t(j == 0 ? d[0] : j == 1 ? d[1] : j == 2 ? d[2] : d[3], pow2);
      e[0] = j == 0 ? t : e[0];
      e[1] = j == 1 ? t : e[1];
      e[2] = j == 2 ? t : e[2];
      e[3] = j == 3 ? t : e[3];
    }
  }
}

// This lane's four exact terms of group g.
__device__ __forceinline__ void group_terms(const float* x, int n, int g, float mx, const double* pow2,
                                            float (&e)[4]) {
  const f32x4 v = load4(x, g * kGroup + 4 * lane_id(), n);
  const float d[4] = {v.x - mx, v.y - mx, v.z - mx, v.w - mx};
  exact_terms(d, pow2, e);
}

// Inclusive scan of the wave's maps, each lane's map taken before those of the
// lanes below it.
__device__ __forceinline__ SeqMap sm_wave_scan_rev(SeqMap m) {
  m = sm_then(m, sm_dpp<0x111, 0xf>(m));
  m = sm_then(m, sm_dpp<0x112, 0xf>(m));
  m = sm_then(m, sm_dpp<0x114, 0xf>(m));
  m = sm_then(m, sm_dpp<0x118, 0xf>(m));
  m = sm_then(m, sm_dpp<0x142, 0xa>(m));
  m = sm_then(m, sm_dpp<0x143, 0xc>(m));
  return m;
}

// The map of a lane's four terms (those at or past place p0 of the group) in
// the binade of exponent E: the plain increment A, and m when a lane of the
// wave holds a tie or a term too large (`wodd`).
__device__ __forceinline__ void lane_run(const float (&e)[4], int p0, int E, int& A, bool& wodd, SeqMap& m) {
  const int i0 = 4 * lane_id();
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = i0 + j >= p0 ? e[j] : 0.0f;
  int a = 0;
  bool odd = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float q = seq_ldexp(v[j], 23 - E);
    const bool ok = q < 16777216.0f;
    const float qc = ok ? q : 0.0f;
    const float fr = seq_fract(qc);
    a += (int)qc + (fr > 0.5f ? 1 : 0);
    odd = odd || !ok || fr == 0.5f;
  }
  A = min(a, 1 << 24);
  wodd = __ballot(odd) != 0ull;
  if (wodd) {
    SeqRun run;
#pragma unroll
    for (int j = 0; j < 4; ++j) run.add(v[j], E);
    m = run.map();
  }
}

// s + the group's terms from place p0 on, one fp32 add at a time: maps while the sum stays in
// its binade, the four terms of the lane that leaves it as plain adds.
__device__ __forceinline__ float replay_group(float s, const float (&e)[4], int p0) {
  while (p0 < kGroup && s == s) {  // uniform
    const int E = seq_binade(s);
    const int S = (int)seq_ldexp(s, 23 - E);
    int A = 0;
    bool wodd = false;
    SeqMap m = sm_identity();
    lane_run(e, p0, E, A, wodd, m);
    int Sin, Sout;
    if (!wodd) {
      Sout = S + wave_incl_scan(A);  // <= 2^24 + 2^30
      Sin = Sout - A;
    } else {
      const SeqMap inc = sm_wave_scan(m);
      Sin = S + sm_inc(sm_dpp<0x138, 0xf>(inc), S);  // wave_shr:1 -- the lanes below
      Sout = Sin < (1 << 24) ? Sin + sm_inc(m, Sin) : Sin;
    }
    const uint64_t cross = __ballot(Sout >= (1 << 24));
    if (!cross) return seq_ldexp((float)__builtin_amdgcn_readlane(Sout, 63), E - 23);
    const int L = __ffsll((unsigned long long)cross) - 1;
    s = seq_ldexp((float)__builtin_amdgcn_readlane(Sin, L), E - 23);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e[j]), L));
      if (4 * L + j >= p0) s = s + t;
    }
    p0 = 4 * L + 4;
  }
  return s;
}

}  // namespace

// ---------------------------------------------------------------- launch A

template <int KIND>
__global__ __launch_bounds__(kNT) void split_max_kernel(SplitArgs a) {
  const int row = (int)(blockIdx.x / (unsigned)a.ns), sl = (int)(blockIdx.x % (unsigned)a.ns);
  const int tid = (int)threadIdx.x, lane = lane_id(), wv = wave_id();
  const float* x = a.logits + (int64_t)row * a.V;
  const int n = (int)a.V;
  const RowWork w = row_work(a, row);
  f32x4 v[kGpw];
  load_groups(x, sl * kSplitSlice + wv * kGpw * kGroup, n, v);
  if (sl == 0 && tid == 0) {
    w.info->count = 0;
    w.info->bound = 0u;
  }
  float m = -__builtin_inff(), rowm;
#pragma unroll
  for (int g = 0; g < kGpw; ++g)
    m = __builtin_fmaxf(m, __builtin_fmaxf(__builtin_fmaxf(v[g].x, v[g].y), __builtin_fmaxf(v[g].z, v[g].w)));
  m = wave_max_f(m, rowm);
  if (KIND == kSplitTop && (lane & 15) == 15) w.gmax[sl * kSplitGroups + wv * 4 + (lane >> 4)] = rowm;
  float t = 0.0f;
  if (KIND != kSplitNll) {
#pragma unroll
    for (int g = 0; g < kGpw; ++g)
      t += (__builtin_amdgcn_exp2f((v[g].x - m) * kLog2e) + __builtin_amdgcn_exp2f((v[g].y - m) * kLog2e)) +
           (__builtin_amdgcn_exp2f((v[g].z - m) * kLog2e) + __builtin_amdgcn_exp2f((v[g].w - m) * kLog2e));
    t = wave_sum_f(t);
    if (!(m > -__builtin_inff())) {  // only -inf (no part of the sum), or NaN among them
      bool nan = false;
#pragma unroll
      for (int g = 0; g < kGpw; ++g)
        nan = nan || v[g].x != v[g].x || v[g].y != v[g].y || v[g].z != v[g].z || v[g].w != v[g].w;
      t = __ballot(nan) ? __builtin_nanf("") : 0.0f;
    }
  }
  // (a NaN or +inf logit leaves a NaN in t)
  if (lane == 0) w.part[sl * kWpb + wv] = make_float2(m, t);
}

// ---------------------------------------------------------------- launch B

// (Rows whose a holds a NaN, or without a finite logit, have a NaN sum; what
// this kernel stores for them is not read.)
template <int KIND>
__global__ __launch_bounds__(kNT, 8) void split_terms_kernel(SplitArgs a) {
  __shared__ double s_pow2[kExpfPow2Count];
  const int row = (int)(blockIdx.x / (unsigned)a.ns), sl = (int)(blockIdx.x % (unsigned)a.ns);
  const int lane = lane_id(), wv = wave_id();
  const float* x = a.logits + (int64_t)row * a.V;
  const int n = (int)a.V;
  const RowWork w = row_work(a, row);
  const int g0 = sl * kSplitGroups + wv * kGpw;  // this wave's first group
  f32x4 v[kGpw];
  load_groups(x, g0 * kGroup, n, v);
  // (every wave writes the whole table, the same values: no barrier, so the
  // workgroup's waves run on their own)
  s_pow2[lane] = kExpfPow2J64[lane];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  // the row's maximum, and the estimated sum of the waves' logits below this one's
  const int me = sl * kWpb + wv;
  float mx = -__builtin_inff(), P = 0.0f, unused;
  if (w.np <= 2 * kWave) {
    const float2 none = make_float2(mx, 0.0f);
    const float2 p0 = lane < w.np ? w.part[lane] : none;
    const float2 p1 = lane + kWave < w.np ? w.part[lane + kWave] : none;
    mx = wave_max_f(__builtin_fmaxf(p0.x, p1.x), unused);
    if (lane < me) P = p0.y * __builtin_amdgcn_exp2f((p0.x - mx) * kLog2e);
    if (lane + kWave < me) P += p1.y * __builtin_amdgcn_exp2f((p1.x - mx) * kLog2e);
  } else {
    for (int i = lane; i < w.np; i += kWave) mx = __builtin_fmaxf(mx, w.part[i].x);
    mx = wave_max_f(mx, unused);
    for (int i = lane; i < me; i += kWave) P += w.part[i].y * __builtin_amdgcn_exp2f((w.part[i].x - mx) * kLog2e);
  }
  P = wave_sum_f(P);
  if (KIND == kSplitTop) {
    // The list's bound.  The row's 256-element maxima, merged to 64: the m-th
    // largest of those is a logit that m distinct elements reach.  Bounds are
    // lowered by more than the spacing at which l - mx, the exponential and
    // the division can round unlike logits to one probability.
    uint32_t key = 0u;
    for (int i = lane; i < a.ns * kSplitGroups; i += kWave) key = max(key, f2key(w.gmax[i]));
    auto lowered = [&](uint32_t k) {
      const float t = key2f(k);
      return t - 0x1p-18f * __builtin_fmaxf(1.0f, __builtin_fmaxf(__builtin_fabsf(mx), __builtin_fabsf(t)));
    };
    float th = lowered(wave_kth_largest(key, a.m));
    if (me == 0 && lane == 0) atomicMax(&w.info->bound, f2key(th));
    float lm = -__builtin_inff();
#pragma unroll
    for (int g = 0; g < kGpw; ++g)
      lm = __builtin_fmaxf(lm, __builtin_fmaxf(__builtin_fmaxf(v[g].x, v[g].y), __builtin_fmaxf(v[g].z, v[g].w)));
    const int lanes = (int)__popcll(__ballot(lm >= th));
    if (lanes > kManyLanes) {  // uniform
      // A wave that holds many of the row's largest logits side by side (rows that
      // rise or fall) has bounds of its own: the m-th largest of its lanes' maxima,
      // and the value that the four neighbours of m / 4 lanes reach.  Without them the
      // list overflows and the last launch reads the row several times (falling
      // rows of 128256, n = 20: one row 194 us, 31 here; 256 rows 300, 120; one launch
      // 131 and 138).
      float four = -__builtin_inff();
#pragma unroll
      for (int g = 0; g < kGpw; ++g)
        four = __builtin_fmaxf(four, __builtin_fminf(__builtin_fminf(v[g].x, v[g].y), __builtin_fminf(v[g].z, v[g].w)));
      const uint32_t own = max(wave_kth_largest(f2key(lm), a.m), wave_kth_largest(f2key(four), (a.m + 3) / 4));
      const float tw = lowered(own);
      if (tw > th) {
        th = tw;
        if (lane == 0) atomicMax(&w.info->bound, f2key(th));
      }
      int total = 0;
#pragma unroll
      for (int g = 0; g < kGpw; ++g) {
        const float l[4] = {v[g].x, v[g].y, v[g].z, v[g].w};
        const int i0 = (g0 + g) * kGroup + 4 * lane;
#pragma unroll
        for (int j = 0; j < 4; ++j) total += (int)__popcll(__ballot(l[j] >= th && i0 + j < n));
      }
      int base = 0;
      if (lane == 0) base = atomicAdd(&w.info->count, total);
      base = __builtin_amdgcn_readfirstlane(base);
      if (base < kSplitList) {
#pragma unroll
        for (int g = 0; g < kGpw; ++g) {
          const float l[4] = {v[g].x, v[g].y, v[g].z, v[g].w};
          const int i0 = (g0 + g) * kGroup + 4 * lane;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const bool in = l[j] >= th && i0 + j < n;
            const uint64_t at = __ballot(in);
            const int slot = base + (int)__popcll(at & lanes_below());
            if (in && slot < kSplitList) w.list[slot] = ((uint64_t)f2key(l[j]) << 32) | (uint32_t)(i0 + j);
            base += (int)__popcll(at);
          }
        }
      }
    } else if (lanes > 0) {
#pragma unroll
      for (int g = 0; g < kGpw; ++g) {
        const float l[4] = {v[g].x, v[g].y, v[g].z, v[g].w};
        const int i0 = (g0 + g) * kGroup + 4 * lane;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (l[j] >= th && i0 + j < n) {
            const int slot = atomicAdd(&w.info->count, 1);
            if (slot < kSplitList) w.list[slot] = ((uint64_t)f2key(l[j]) << 32) | (uint32_t)(i0 + j);
          }
      }
    }
  }

  // l - mx as the reference forms it, and the estimates of the terms
  float d[kGpw][4], y[kGpw][4], gsum[kGpw];
#pragma unroll
  for (int g = 0; g < kGpw; ++g) {
    d[g][0] = v[g].x - mx;
    d[g][1] = v[g].y - mx;
    d[g][2] = v[g].z - mx;
    d[g][3] = v[g].w - mx;
#pragma unroll
    for (int j = 0; j < 4; ++j) y[g][j] = expf_estimate(d[g][j]);
    gsum[g] = (y[g][0] + y[g][1]) + (y[g][2] + y[g][3]);
  }
  wave_sum4(gsum);
  const int ng = (n + kGroup - 1) / kGroup;
  int E[kGpw];
  float inc[kGpw];        // the group's increment, as far as it is settled
  uint32_t late = 0u;     // groups with unsettled terms
  uint32_t cross = 0u;    // groups the estimates take into another binade
#pragma unroll
  for (int g = 0; g < kGpw; ++g) {
    E[g] = seq_binade(P);
    P += gsum[g];
    if (seq_binade(P) != E[g]) cross |= 1u << g;
    const float up = seq_ldexp(1.0f, min(23 - E[g], 127));
    float open = 0.0f, t = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float q = y[g][j] * up;
      const float r = __builtin_rintf(q);
      open = __builtin_fmaxf(open, __builtin_fmaf(q, kSplitErr, __builtin_fabsf(q - r)));
      t += r;  // exact where settled: each r <= 2^21, four of them below 2^24
    }
    inc[g] = t;
    // (from 2^-80 on, a term whose estimate was flushed is far below u / 2)
    if (__ballot(!(open < 0.5f)) || gsum[g] == 0.0f || E[g] < -80) late |= 1u << g;
  }
  // sums of integers up to 2^29: exact below 2^24, and rounding keeps any other at
  // 2^24 or more (it is monotone), where the group leaves the binade
  wave_sum4(inc);
  {
    // lane g stores group g's map
    float t = inc[0];
    int Eg = E[0];
#pragma unroll
    for (int k = 1; k < kGpw; ++k) {
      t = lane == k ? inc[k] : t;
      Eg = lane == k ? E[k] : Eg;
    }
    const int ti = (int)__builtin_fminf(t, 16777216.0f);
    if (lane < kGpw && g0 + lane < ng && !((late >> lane) & 1u))
      w.maps[g0 + lane] = pack_map(sm_make(ti, ti & 1, ti, (ti + 1) & 1), Eg + kCodeBias,
                                   ((cross >> lane) & 1u) != 0u || ti >= (1 << 24));
  }
  // the groups with unsettled terms, from the exact ones
#pragma unroll 1
  for (; late; late &= late - 1) {  // uniform
    const int g = __ffs(late) - 1;
    if (g0 + g >= ng) break;
    int Eg = E[0];
    float dg[4] = {d[0][0], d[0][1], d[0][2], d[0][3]}, e[4];
#pragma unroll
    for (int k = 1; k < kGpw; ++k) {
      Eg = g == k ? E[k] : Eg;
#pragma unroll
      for (int j = 0; j < 4; ++j) dg[j] = g == k ? d[k][j] : dg[j];
    }
    exact_terms(dg, s_pow2, e);
    SeqMap m = sm_identity();
    int code = Eg + kCodeBias;
    if (__ballot(e[0] != 0.0f || e[1] != 0.0f || e[2] != 0.0f || e[3] != 0.0f) == 0ull) {
      code = kCodeAny;
    } else {
      int A;
      bool wodd;
      lane_run(e, 0, Eg, A, wodd, m);
      if (!wodd) {
        const int t = wave_incl_scan(A);  // <= 2^30
        m = sm_make(t, t & 1, t, (t + 1) & 1);
      } else {
        m = sm_wave_scan(m);
      }
      m = sm_readlane(m, 63);
    }
    const bool cr = ((cross >> g) & 1u) != 0u || (m.a >> 1) >= (1 << 24) || (m.c >> 1) >= (1 << 24);
    if (lane == 0) w.maps[g0 + g] = pack_map(m, code, cr);
  }
}

// perplexity's term (model.nim:578-583).  row_nll_kernel's 1024 threads each add
// their own float64 exponentials in index order (a thread's are 1024 float4 groups
// apart, or 1024 logits in rows off 16 bytes), then the waves' lanes in a tree, then
// the 16 waves.  The same sum here, so that a position's term does not depend on
// how many are scored together: a workgroup per row and one of those waves, whose
// exponentials the workgroup's waves share out (64 slots of the 64 lanes per chunk,
// through LDS) and its first wave adds in their order.  Bound by float64 issue
// and, for few rows, by the chunks' barriers: 8 x 50001 9.6 us, 8 x 128256 11.6 (row_nll_kernel
// 19.5 and 36.3; slices of 4096 logits with a tree of their own 9.9 and 9.9).  (Sixteen
// waves, the last one adding a chunk behind the others: 10.2 and 12.3.)
constexpr int kNllNT = 512;
constexpr int kNllWaves = kNllNT / kWave;
constexpr int kNllParts = 16;                      // row_nll_kernel's waves
constexpr int kNllThreads = kNllParts * kWave;     // and threads
constexpr int kNllSlots = 64;                      // of a chunk
constexpr int kNllPer = kNllSlots / kNllWaves;     // a wave's slots
__global__ __launch_bounds__(kNllNT) void split_nll_kernel(SplitArgs a) {
  __shared__ double s_t[kExp64Table];
  __shared__ double s_e[kNllSlots][kWave];
  const int row = (int)(blockIdx.x / kNllParts), part = (int)(blockIdx.x % kNllParts);
  const int tid = (int)threadIdx.x, lane = lane_id(), wv = wave_id();
  const float* x = a.logits + (int64_t)row * a.V;
  const int n = (int)a.V;
  const RowWork w = row_work(a, row);
  const int t = part * kWave + lane;  // the thread of row_nll_kernel
  const bool vec = n % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
  const int slots = vec ? (n / 4 + kNllThreads - 1) / kNllThreads * 4 : (n + kNllThreads - 1) / kNllThreads;
  float v[kNllPer];
  auto first = [&](int s0) { return s0 + wv * kNllPer; };  // this wave's first slot of the chunk
  // element of slot s (past the row: none)
  auto elem = [&](int s) { return vec ? 4 * (t + (s >> 2) * kNllThreads) + (s & 3) : t + s * kNllThreads; };
  auto load = [&](int s0) __attribute__((always_inline)) {
    if (vec) {
#pragma unroll
      for (int k = 0; k < kNllPer; k += 4) {
        const int i = elem(first(s0) + k);
        f32x4 q{};
        if (i < n) q = *reinterpret_cast<const f32x4*>(x + i);
        v[k] = q.x;
        v[k + 1] = q.y;
        v[k + 2] = q.z;
        v[k + 3] = q.w;
      }
    } else {
#pragma unroll
      for (int k = 0; k < kNllPer; ++k) {
        const int i = elem(first(s0) + k);
        v[k] = i < n ? x[i] : 0.0f;
      }
    }
  };
  load(0);
  if (tid < kExp64Table) s_t[tid] = exp64_table_entry(tid);
  float mx = -__builtin_inff(), unused;
  for (int i = lane; i < w.np; i += kWave) mx = __builtin_fmaxf(mx, w.part[i].x);
  mx = wave_max_f(mx, unused);
  __syncthreads();
  double ps = 0.0;
  for (int s0 = 0; s0 < slots; s0 += kNllSlots) {
#pragma unroll
    for (int k = 0; k < kNllPer; ++k)
      // (+0 past the row: no exponential is -0, so the sum keeps its bits)
      s_e[wv * kNllPer + k][lane] = elem(first(s0) + k) < n ? exp64((double)(v[k] - mx), s_t) : 0.0;
    if (s0 + kNllSlots < slots) load(s0 + kNllSlots);
    __syncthreads();
    if (wv == 0) {
#pragma unroll 16
      for (int k = 0; k < kNllSlots; ++k) ps += s_e[k][lane];
    }
    __syncthreads();
  }
  if (wv != 0) return;
  for (int o = kWave / 2; o > 0; o >>= 1) ps += __shfl_xor(ps, o);
  if (lane == 0) w.maps[part] = (uint64_t)__double_as_longlong(ps);
}

// ---------------------------------------------------------------- launch C

// The waves' sums in row_nll_kernel's order, and the row's term.
__global__ __launch_bounds__(kWave) void split_nll_sum_kernel(SplitArgs a) {
  const int row = (int)blockIdx.x, lane = lane_id();
  const RowWork w = row_work(a, row);
  const int t = a.targets[row];
  const bool in = t >= 0 && t < a.V;
  const float lt = in ? a.logits[(int64_t)row * a.V + t] : 0.0f;
  const double p = lane < kNllParts ? __longlong_as_double((long long)w.maps[lane]) : 0.0;
  float mx = -__builtin_inff(), unused;
  for (int i = lane; i < w.np; i += kWave) mx = __builtin_fmaxf(mx, w.part[i].x);
  mx = wave_max_f(mx, unused);
  double s = __shfl(p, 0);
  for (int k = 1; k < kNllParts; ++k) s += __shfl(p, k);
  if (lane == 0) a.logp[row] = in ? -((double)(lt - mx) - log(s)) : __builtin_nan("");
}

// The walk: rounds of 1024 groups, one map per thread, 64 groups per wave.  All
// waves prepare: the prefix sums of their 64 increments; the list of events,
// the groups that are more than an increment in the binade of the group
// before them; and, one wave each, the groups expected to cross a binade
// (their terms, the maps of every lane's predecessors in the binade the group
// starts in and of its successors in the next).  Then one wave goes from event
// to event with the sum as an integer S in units of its binade E, every step a
// few scalar instructions; what no preparation foresaw takes walk_rest's
// general steps.  (Scanning the maps after each event instead, the one wave
// took 31,000 cycles for 500 groups; from event to event of 64 groups with
// their maps in LDS, 22,000; now 12,700.)
struct WalkShared {
  double pow2[kExpfPow2Count];
  uint64_t map[kWalkNT];
  int ps[kWalkNT];               // increments up to and with this group, within its 64
  signed char slot[kWalkNT];     // where the group's terms are, or -1
  short event[kWalkNT + 1];      // the events' places in the round, ascending, then the round's end
  uint64_t events[kWalkNT / kWave];
  int nslot;
  int slotg[kSlots];
  int2 below[kSlots][kWave];     // map of the lanes up to this one, starting binade
  int2 above[kSlots][kWave];     // map of the lanes past this one, next binade
  float e[kSlots * kGroup];
  float head[kHeadGroups * kGroup];
  float head_sum;
};

// s over groups pos .. 63 of the 64 at `first`, any maps.
__device__ __forceinline__ float walk_rest(float s, int pos, uint64_t uq, int slots, int first, const float* x, int n, float mx,
                           const WalkShared& sh) {
  const int lane = lane_id();
  const int code = unpack_code(uq);
  const SeqMap mq = unpack_map(uq);
  while (pos < kWave) {  // uniform
    const int E = seq_binade(s);
    const int S = (int)seq_ldexp(s, 23 - E);
    const bool ok = code == kCodeAny || code == E + kCodeBias;
    const int Sa = S + sm_inc(sm_wave_scan(ok && lane >= pos ? mq : sm_identity()), S);
    const uint64_t stop = __ballot(lane >= pos && (!ok || Sa >= (1 << 24)));
    if (!stop) return seq_ldexp((float)__builtin_amdgcn_readlane(Sa, 63), E - 23);
    const int f = __ffsll((unsigned long long)stop) - 1;
    const int Sb = f > 0 ? __builtin_amdgcn_readlane(Sa, f - 1) : S;
    s = seq_ldexp((float)Sb, E - 23);
    const int sf = __builtin_amdgcn_readlane(slots, f);
    float e[4];
    if (sf >= 0) {
      const float4 t = *reinterpret_cast<const float4*>(sh.e + sf * kGroup + 4 * lane);
      e[0] = t.x;
      e[1] = t.y;
      e[2] = t.z;
      e[3] = t.w;
    } else {
      group_terms(x, n, first + f, mx, sh.pow2, e);
    }
    s = replay_group(s, e, 0);
    pos = f + 1;
  }
  return s;
}

// One wave: s over the round's groups, nev events before its end.
__device__ __forceinline__ float walk_round(float s, int c0, int nev, const float* x, int n, float mx, const WalkShared& sh) {
  const int lane = lane_id();
  int E = __builtin_amdgcn_readfirstlane(seq_binade(s));
  int S = __builtin_amdgcn_readfirstlane((int)seq_ldexp(s, 23 - E));
  auto set = [&](float t) __attribute__((always_inline)) {
    E = __builtin_amdgcn_readfirstlane(seq_binade(t));
    S = __builtin_amdgcn_readfirstlane((int)seq_ldexp(t, 23 - E));
  };
  bool resumed = false;  // S is the sum up to the next event already
  for (int k0 = 0; k0 <= nev; k0 += kWave) {
    // lane k: event k0 + k.  (The first group of every 64 is an event, so the
    // increments between two events are those of one wave's prefix sums.)
    const int k = min(k0 + lane, nev);
    const int ge = sh.event[k];
    const int gp = k > 0 ? sh.event[k - 1] : -1;
    const int between = gp >= 0 ? sh.ps[ge - 1] - sh.ps[gp] : 0;  // <= 2^30
    const bool end = k == nev;
    const uint64_t um = end ? pack_map(sm_identity(), kCodeAny, false) : sh.map[ge];
    const int slot = end ? -1 : (int)sh.slot[ge];
    const int ma = (int)(um & 0x3ffffffu), mc = (int)((um >> 26) & 0x3ffffffu), top = (int)(um >> 52);
    int i = 0;
    const int cnt = min(kWave, nev + 1 - k0);
    while (i < cnt) {  // uniform
      const int g = __builtin_amdgcn_readlane(ge, i);
      const int code = __builtin_amdgcn_readlane(top, i);  // (the crossing mark in bit 8)
      const int sf = __builtin_amdgcn_readlane(slot, i);
      const int S2 = S + (resumed ? 0 : __builtin_amdgcn_readlane(between, i));
      resumed = false;
      int rest = -1;  // >= 0: groups rest .. up to the end of its 64 take the general steps
      if (S2 >= (1 << 24)) {
        rest = __builtin_amdgcn_readlane(gp, i) + 1;
      } else {
        S = S2;
        if (code == kCodeAny) {
        } else if ((code & 0xff) != E + kCodeBias) {
          rest = g;
        } else if (sf >= 0) {
          const int2 b = sh.below[sf][lane], t = sh.above[sf][lane];
          const float4 e4 = *reinterpret_cast<const float4*>(sh.e + sf * kGroup + 4 * lane);
          const int Sl = S + sm_inc(SeqMap{b.x, b.y}, S);
          const uint64_t over = __ballot(Sl >= (1 << 24));
          if (!over) {
            S = __builtin_amdgcn_readlane(Sl, 63);
            rest = g + 1;  // (the groups after it are mapped for the next binade)
          } else {
            // the first lane to leave the binade adds its four terms as they
            // are; the lanes past it are in the next binade
            const int L = __ffsll((unsigned long long)over) - 1;
            float e[4] = {e4.x, e4.y, e4.z, e4.w};
            s = seq_ldexp((float)(L > 0 ? __builtin_amdgcn_readlane(Sl, L - 1) : S), E - 23);
#pragma unroll
            for (int j = 0; j < 4; ++j) s = s + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e[j]), L));
            const int S1 = __builtin_amdgcn_readfirstlane((int)seq_ldexp(s, 22 - E));
            const int Sn =
                S1 + sm_inc(SeqMap{__builtin_amdgcn_readlane(t.x, L), __builtin_amdgcn_readlane(t.y, L)}, S1);
            if (S1 >= (1 << 23) && S1 < (1 << 24) && Sn < (1 << 24)) {
              E = E + 1;
              S = Sn;
            } else {
              const int before = E;
              set(replay_group(s, e, 4 * L + 4));
              if (E != before + 1) rest = g + 1;
            }
          }
        } else {
          const int Sn = S + sm_inc(SeqMap{__builtin_amdgcn_readlane(ma, i), __builtin_amdgcn_readlane(mc, i)}, S);
          if ((code >> 8) || Sn >= (1 << 24))
            rest = g;  // (or a crossing past the last slot)
          else
            S = Sn;
        }
      }
      ++i;
      if (rest >= 0) {
        const int first = (rest > g ? g : rest) & ~(kWave - 1);
        s = walk_rest(seq_ldexp((float)S, E - 23), rest - first, sh.map[first + lane], sh.slot[first + lane],
                      c0 + first, x, n, mx, sh);
        set(s);
        // on to the first event past those 64 (the next 64's first group)
        resumed = true;
        const uint64_t past = __ballot(ge >= first + kWave && lane < cnt);
        i = past ? __ffsll((unsigned long long)past) - 1 : cnt;
        if (!past && k0 + kWave <= nev) {
          // (more than 64 events: the next 64 may still lie in those groups)
          int kn = k0 + kWave;
          while (kn < nev && sh.event[kn] < first + kWave) ++kn;
          k0 = kn - kWave;
        }
      }
    }
  }
  return seq_ldexp((float)S, E - 23);
}

// The sum of a row with a NaN term (one wave): the reference's adds leave the first
// NaN term as it is from there on, sign and payload included.  topTokens orders
// the quotients by them: with another NaN than the row's own as the sum, the
// entries that are NaN themselves would leave their places among the others.
__device__ __forceinline__ float first_nan_term(const RowWork& w, const float* x, int n, float mx) {
  const int lane = lane_id();
  int i0 = 0;  // (no finite logit: -inf - -inf is the first term)
  if (mx > -__builtin_inff()) {
    for (int k = 0; k < w.np; k += kWave) {  // the first 1024 logits whose estimate is a NaN
      const float y = k + lane < w.np ? w.part[k + lane].y : 0.0f;
      const uint64_t hit = __ballot(y != y);
      if (hit) {
        i0 = (k + __ffsll((unsigned long long)hit) - 1) * kGpw * kGroup;
        break;
      }
    }
  }
  for (int i = i0; i < n; i += kWave) {
    const float d = i + lane < n ? x[i + lane] - mx : 0.0f;
    const uint64_t hit = __ballot(d != d);
    if (hit) {
      const int l = __ffsll((unsigned long long)hit) - 1;
      const float t = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d), l));
      return t + t;  // (the exponential's NaN)
    }
  }
  return __builtin_nanf("");
}

template <bool LOGP>
__global__ __launch_bounds__(kWalkNT) void split_walk_kernel(SplitArgs a) {
  __shared__ __align__(16) WalkShared sh;
  const int row = (int)blockIdx.x, tid = (int)threadIdx.x, lane = lane_id(), wv = wave_id();
  const float* x = a.logits + (int64_t)row * a.V;
  const int n = (int)a.V;
  const int ng = (n + kGroup - 1) / kGroup;
  const RowWork w = row_work(a, row);
  uint64_t u = kHeadGroups + tid < ng ? w.maps[kHeadGroups + tid] : 0ull;
  float s = 0.0f;
  if (tid < kExpfPow2Count) sh.pow2[tid] = kExpfPow2J64[tid];
  float mx = -__builtin_inff(), bad = 0.0f, unused;
  for (int i = lane; i < w.np; i += kWave) {
    mx = __builtin_fmaxf(mx, w.part[i].x);
    bad += w.part[i].y;  // (a sum of finite estimates is no NaN)
  }
  mx = wave_max_f(mx, unused);
  bad = wave_sum_f(bad);
  if (bad == bad && mx > -__builtin_inff()) {  // uniform
    for (int c0 = kHeadGroups; c0 < ng; c0 += kWalkNT) {
      const int g = c0 + tid;
      if (c0 > kHeadGroups) u = g < ng ? w.maps[g] : 0ull;
      if (g >= ng) u = pack_map(sm_identity(), kCodeAny, false);
      if (tid == 0) sh.nslot = 0;
      __syncthreads();
      const bool cross = (u >> 60) & 1;
      const SeqMap mu = unpack_map(u);
      // the group before it in its 64, and the binade that leaves
      const uint64_t up = (uint64_t)(uint32_t)__shfl_up((int)(u >> 32), 1) << 32;
      const int after = unpack_code(up) == kCodeAny ? -1 : unpack_code(up) + (int)((up >> 60) & 1);
      const int code = unpack_code(u);
      const bool event =
          g < ng && (lane == 0 || cross || !sm_is_plain(mu) || (code != kCodeAny && code != after));
      sh.map[tid] = u;
      sh.ps[tid] = wave_incl_scan(event ? 0 : mu.a >> 1);  // <= 2^30
      const uint64_t ev = __ballot(event);
      if (lane == 0) sh.events[wv] = ev;
      int slot = -1;
      if (cross) {
        slot = atomicAdd(&sh.nslot, 1);
        if (slot < kSlots)
          sh.slotg[slot] = g;
        else
          slot = -1;
      }
      sh.slot[tid] = (signed char)slot;
      __syncthreads();
      int nev = 0, before = 0;
      for (int k = 0; k < kWalkNT / kWave; ++k) {
        const int c = __popcll(sh.events[k]);
        before += k < wv ? c : 0;
        nev += c;
      }
      if (event) sh.event[before + __popcll(ev & lanes_below())] = (short)tid;
      if (tid == 0) sh.event[nev] = (short)min(kWalkNT, (ng - c0 + kWave - 1) / kWave * kWave);
      if (c0 == kHeadGroups && wv == kWalkNT / kWave - 1) {
        // the row's first terms, one at a time: while the sum is a few terms
        // large it changes binade every few terms
        float e[4];
        group_terms(x, n, 0, mx, sh.pow2, e);
        *reinterpret_cast<float4*>(sh.head + 4 * lane) = make_float4(e[0], e[1], e[2], e[3]);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        float t = 0.0f;
#pragma unroll 8
        for (int i = 0; i < kGroup; i += 4) {
          const float4 h = *reinterpret_cast<const float4*>(sh.head + i);
          t = t + h.x;
          t = t + h.y;
          t = t + h.z;
          t = t + h.w;
        }
        if (lane == 0) sh.head_sum = t;
      } else if (wv < min(sh.nslot, kSlots)) {
        float e[4];
        const int sg = sh.slotg[wv];
        group_terms(x, n, sg, mx, sh.pow2, e);
        *reinterpret_cast<float4*>(sh.e + wv * kGroup + 4 * lane) = make_float4(e[0], e[1], e[2], e[3]);
        const int E = unpack_code(sh.map[sg - c0]) - kCodeBias;
        int A;
        bool odd;
        SeqMap m = sm_identity();
        lane_run(e, 0, E, A, odd, m);
        m = sm_wave_scan(odd ? m : sm_make(A, A & 1, A, (A + 1) & 1));
        sh.below[wv][lane] = make_int2(m.a, m.c);
        lane_run(e, 0, E + 1, A, odd, m);
        if (!odd) m = sm_make(A, A & 1, A, (A + 1) & 1);
        // the lanes past this one: the scan over the lanes in reverse
        m = sm_wave_scan_rev(SeqMap{__shfl(m.a, kWave - 1 - lane), __shfl(m.c, kWave - 1 - lane)});
        m = sm_dpp<0x138, 0xf>(m);  // wave_shr:1
        sh.above[wv][lane] = make_int2(__shfl(m.a, kWave - 1 - lane), __shfl(m.c, kWave - 1 - lane));
      }
      __syncthreads();
      if (wv == 0) s = walk_round(c0 == kHeadGroups ? sh.head_sum : s, c0, nev, x, n, mx, sh);
      __syncthreads();  // (the round's LDS is free again)
    }
  } else if (wv == 0) {
    s = first_nan_term(w, x, n, mx);
  }
  if (tid == 0) {
    if (LOGP) {
      // p[t] (:57) and ln(float64(p[t]))
      const int t = a.targets[row];
      float p = __builtin_nanf("");
      if (t >= 0 && t < n) p = expf_cr_t(x[t] - mx, sh.pow2) / s;
      a.prob[row] = p;
      a.logp[row] = log((double)p);
    } else {
      w.info->mx = mx;
      w.info->sum = s;
    }
  }
}

// ---------------------------------------------------------------- launch D

__global__ __launch_bounds__(kNT, 8) void split_out_kernel(SplitArgs a) {
  __shared__ double s_pow2[kExpfPow2Count];
  const int row = (int)(blockIdx.x / (unsigned)a.ns), sl = (int)(blockIdx.x % (unsigned)a.ns);
  const int tid = (int)threadIdx.x, lane = lane_id(), wv = wave_id();
  const float* x = a.logits + (int64_t)row * a.V;  // (may be a.out's row: a thread reads, then writes, its own)
  float* o = a.out + (int64_t)row * a.V;
  const int n = (int)a.V;
  const int i0 = sl * kSplitSlice + wv * kGpw * kGroup + 4 * lane;
  f32x4 v[kGpw];
  load_groups(x, i0 - 4 * lane, n, v);
  if (tid < kExpfPow2Count) s_pow2[tid] = kExpfPow2J64[tid];
  const float mx = a.info[row].mx, s = a.info[row].sum;
  // e / s = e (1 / s) in float64: the quotient of two 24-bit numbers that is no
  // float lies at least 2^-49 of itself from the middle of two, and the product is within
  // 2^-52 of it, so its rounding is the quotient's (results below 2^-126, with
  // fewer bits, are divided)
  const double inv = 1.0 / (double)s;
  __syncthreads();
#pragma unroll
  for (int g = 0; g < kGpw; ++g) {
    const int i = i0 + g * kGroup;
    float d[4] = {v[g].x - mx, v[g].y - mx, v[g].z - mx, v[g].w - mx}, r[4];
    bool all = true;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      bool ok;
      r[j] = (float)((double)expf_cr_quick(d[j], s_pow2, ok) * inv);
      // (masked logits: their exponential is 0 from -104 on, with no exact path to take;
      // 256 x 128256 with 1 logit of 97 unmasked 174 us without this, 145 with it)
      const bool zero = d[j] <= -104.0f && s == s;
      r[j] = zero ? 0.0f : r[j];
      all = all && (zero || (ok && r[j] >= 0x1p-126f));
    }
    if (!all) {
      float e[4];
      exact_terms(d, s_pow2, e);
#pragma unroll
      for (int j = 0; j < 4; ++j) r[j] = e[j] / s;
    }
    if (i + 4 <= n) {
      __builtin_memcpy(o + i, r, 16);
    } else {
      if (i < n) o[i] = r[0];
      if (i + 1 < n) o[i + 1] = r[1];
      if (i + 2 < n) o[i + 2] = r[2];
    }
  }
}

// ---------------------------------------------------------------- host side

size_t split_workspace(int kind, int64_t rows, int64_t V, int m) {
  // One slice gains nothing from the split; the slices' records fit one
  // wave's registers up to kSplitMaxSlices; the grid stays below 2^32 threads.
  const int64_t ns = (V + kSplitSlice - 1) / kSplitSlice;
  if (rows <= 0 || V < kSplitMinV || ns > kSplitMaxSlices || rows * ns >= (int64_t{1} << 23)) return 0;
  if (kind == kSplitNll && (V < kSplitMinNllV || rows > kSplitMaxNllRows)) return 0;
  // softmax's fourth launch pays from longer rows on, or from more rows than
  // CUs (the one launch's second round): 8 x 9000 27.4 -> 29.6 us, 160 x 12288 35.5 ->
  // 34.8, 256 x 12288 36.0 -> 36.6, 256 x 14000 41.6 -> 40.4, 400 x 8192 55 -> 44.  logProb and
  // topTokens gain from kSplitMinV on (256 x 9000 27.6 -> 27.2, 1 x 8192 23 -> 17; 42 -> 30,
  // 38 -> 20)
  if (kind == kSplitSoftmax && rows <= 256 && V < (rows <= 192 ? 12288 : 14336)) return 0;
  // the list's bound is the m-th largest of up to 64 maxima of 256 logits
  if (kind == kSplitTop && m > std::min<int64_t>(kWave, V / kGroup)) return 0;
  size_t b = (size_t)rows * sizeof(SplitRowInfo) + (size_t)(rows * ns) * (kSplitGroups * 8 + kWpb * 8);
  if (kind == kSplitTop) b += (size_t)(rows * ns) * kSplitGroups * 4 + (size_t)rows * kSplitList * 8;
  return b;
}

// Whether a call that brought the bytes above runs split.  perplexity's one
// launch is bound by one CU's float64 units per row, so its split pays until the
// rows fill the chip by themselves (64 / 96 / 128 / 160 rows, one launch against
// split: V = 50000 16.8 / 17.0 / 17.8 / 18.4 us against 13.9 / 18.1 / 22.5 / 25.4; 65536
// 20.6 / 20.5 / 20.6 / 24.7 against 14.1 / 19.9 / 23.8 / 27.7; 128256 38 / 41 / 43 / 45
// against 25 / 32 / 39 / 46).
bool split_pays(int kind, int64_t rows, int64_t V) {
  return kind != kSplitNll || rows <= (V < 65536 ? 64 : V < 96000 ? 96 : 128);
}

hipError_t launch_split(int kind, SplitArgs a, int rows, void* work, hipStream_t s) {
  a.ns = (int)((a.V + kSplitSlice - 1) / kSplitSlice);
  const int64_t slices = (int64_t)rows * a.ns;
  uint8_t* p = static_cast<uint8_t*>(work);
  a.info = reinterpret_cast<SplitRowInfo*>(p);
  p += (size_t)rows * sizeof(SplitRowInfo);
  a.maps = reinterpret_cast<uint64_t*>(p);
  p += (size_t)slices * kSplitGroups * 8;
  a.part = reinterpret_cast<float2*>(p);
  p += (size_t)slices * kWpb * 8;
  a.list = reinterpret_cast<uint64_t*>(p);  // (topTokens only)
  p += (size_t)rows * kSplitList * 8;
  a.gmax = reinterpret_cast<float*>(p);
  const dim3 grid((unsigned)slices), block(kNT);
  if (kind == kSplitNll) {
    hipLaunchKernelGGL(split_max_kernel<kSplitNll>, grid, block, 0, s, a);
    hipLaunchKernelGGL(split_nll_kernel, dim3((unsigned)rows * kNllParts), dim3(kNllNT), 0, s, a);
    hipLaunchKernelGGL(split_nll_sum_kernel, dim3(rows), dim3(kWave), 0, s, a);
  } else if (kind == kSplitTop) {
    hipLaunchKernelGGL(split_max_kernel<kSplitTop>, grid, block, 0, s, a);
    hipLaunchKernelGGL(split_terms_kernel<kSplitTop>, grid, block, 0, s, a);
    hipLaunchKernelGGL(split_walk_kernel<false>, dim3(rows), dim3(kWalkNT), 0, s, a);
    return launch_split_top(a, rows, s);
  } else {
    hipLaunchKernelGGL(split_max_kernel<kSplitSoftmax>, grid, block, 0, s, a);
    hipLaunchKernelGGL(split_terms_kernel<kSplitSoftmax>, grid, block, 0, s, a);
    if (kind == kSplitLogProb) {
      hipLaunchKernelGGL(split_walk_kernel<true>, dim3(rows), dim3(kWalkNT), 0, s, a);
    } else {
      hipLaunchKernelGGL(split_walk_kernel<false>, dim3(rows), dim3(kWalkNT), 0, s, a);
      hipLaunchKernelGGL(split_out_kernel, grid, block, 0, s, a);
    }
  }
  return hipGetLastError();
}

}  // namespace nls
