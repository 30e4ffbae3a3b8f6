// nls_rowsplit.h -- arguments of the kernels that split a row over workgroups
// (nls_rowsplit.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace nls {

enum { kSplitSoftmax = 0, kSplitLogProb = 1, kSplitTop = 2, kSplitNll = 3 };
constexpr int kSplitNT = 256;
constexpr int kSplitSlice = 4096;                  // logits per workgroup
constexpr int kSplitGroups = kSplitSlice / 256;    // maps per slice
constexpr int kSplitMaxSlices = 256;               // rows up to 1,048,576 logits
constexpr int kSplitMinV = 8192;
constexpr int kSplitMinNllV = 40960;               // perplexity's term
constexpr int kSplitMaxNllRows = 160;
constexpr int kSplitList = 2048;                   // topTokens: logits listed per row

// Relative distance of expf_estimate(d) from the correctly rounded e^d, for
// d in [-87, 0] (nls_expf_forms_device checks it on every input it is given).  Below
// -87 both are under 2^-125.
constexpr float kSplitErr = 0x1p-22f;

struct SplitRowInfo {
  float mx, sum;
  uint32_t bound;  // topTokens: every logit whose key reaches it is listed (both
  int count;       // zeroed by the first launch); the logits listed
  int pad[4];
};

struct SplitArgs {
  const float* logits;
  int64_t V;
  float* out;              // softmax
  const int32_t* targets;  // logProb, perplexity
  float* prob;             // logProb
  double* logp;            // logProb, perplexity
  int32_t* ids;            // topTokens
  float* probs;
  int n, m;                // topTokens: entries per row of ids / probs, and written
  int ns;                  // slices per row
  SplitRowInfo* info;
  uint64_t* maps;
  float2* part;
  uint64_t* list;
  float* gmax;
};

// Workspace bytes, 0 where the one-launch kernels run the call.
size_t split_workspace(int kind, int64_t rows, int64_t V, int m);
bool split_pays(int kind, int64_t rows, int64_t V);
hipError_t launch_split(int kind, SplitArgs a, int rows, void* work, hipStream_t s);
// topTokens' last launch (nls_kernels.hip).
hipError_t launch_split_top(const SplitArgs& a, int rows, hipStream_t s);

// e^d for d <= 0 in fp32: 2^h (1 + t ln2), h + t = d log2(e) with log2(e) in two
// parts.  v_exp_f32 is good to 1 ulp and the rest adds one rounding.  A result
// below 2^-126 may be flushed to zero.
__device__ __forceinline__ float expf_estimate(float d) {
  constexpr float kHi = 1.44269502162933349609375f, kLo = 1.92596299112661746887e-08f;
  d = __builtin_fmaxf(d, -150.0f);  // (-inf, whose h + t is not a number; a NaN too)
  const float h = d * kHi;
  const float t = __builtin_fmaf(d, kLo, __builtin_fmaf(d, kHi, -h));
  const float p = __builtin_amdgcn_exp2f(h);
  return __builtin_fmaf(p, t * 0.693147182464599609375f, p);
}

}  // namespace nls
