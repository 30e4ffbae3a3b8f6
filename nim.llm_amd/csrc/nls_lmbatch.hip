// nls_lmbatch.hip -- the output projection for several hidden states at once
// (the K formats' int8 path) on the int8 matrix cores.
//
// Same results as lm_int1_kernel (nls_lmhead.hip): per block of 256 weights an
// exact integer dot product, then the reference's fp32 term
// (quant.nim:669-760), the terms added in block order.  Here a block's integer
// products are a matrix product: 32 weight rows x 32 states x 256, on
// v_mfma_i32_32x32x32_i8.
//
// A weight enters the sum as p = sc * q (its sub-block's integer scale times
// its level), which takes 10 to 13 bits, so it is split in two signed bytes
// p = L + 2^kShift * H and each plane has its own product; the int32 sums are
// joined exactly afterwards (sumi = S_L + (S_H << kShift)):
//   Q4_K  sc = sl + 8 sh (6 bits): L = q sl, H = q sh (<= 105), kShift 3: one
//         packed 16-bit product per four weights and plane (no carry leaves a
//         byte);
//   Q5_K  p <= 1953 and Q6_K |p| <= 4096 (level q - 32): L = p & 127,
//         H = p >> 7, kShift 7.
// The mins of Q4_K / Q5_K (summ = sum of m_j times the sums of 16 activations)
// are a product over 16 integers of at most 11 bits: one
// v_mfma_f32_32x32x16_f16, exact (every partial sum is below 2^24).
//
// One wave holds 32 rows: lane l's row is l % 32, and of each 32 consecutive
// weights (one matrix step) it owns the 16 from 16 (l / 32) on, read straight
// from the GGUF block and held as both planes in registers (64 VGPRs) for all
// the states.  The states' int8 activations go through LDS, shared by the
// workgroup's four waves, in the order the matrix unit takes them; the next
// block's are loaded while this block is computed.  The result has the rows
// across lanes, so the block scales are one value per lane and the stores are
// contiguous.
//
// Bound: at few states the weights' HBM traffic and the making of the planes
// (about 2 VALU instructions per 4 weights and plane for Q4_K, 7 for Q6_K), at
// many the matrix unit (two planes, 32 cycles per 32 x 32 x 32 step: 57 us of
// about 200 at 255 states) and the 5 to 7 VALU instructions per term (89 us),
// which two waves per SIMD overlap only in part.  A call's time, activations
// quantised in it, lm_int_kernel (one dot-product instruction per four products,
// weights re-read per four states) -> here: 128256 x 2048 Q4_K, 255 states
// 3961 -> 204 us; Q6_K, 24 states 542 -> 74, 5 states 138 -> 72; 32000 x 4096 Q6_K, 3
// states 73 -> 49; fewer rows than fill the chip gain too: 8000 x 2048 Q4_K, 24 states
// 125 -> 16, 16000 x 4096 Q4_K, 8 states 107 -> 27, 8000 x 4096 Q6_K, 5 states 84 -> 47.  Few
// states of long rows do not (int_kernel_wins, nls_lmhead.hip).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "nls_internal.h"
#include "nls_lmhead.h"

namespace nls {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef short v2s __attribute__((ext_vector_type(2)));
typedef unsigned short v2u __attribute__((ext_vector_type(2)));

constexpr int kBWaves = 4;
constexpr int kBNT = 64 * kBWaves;
constexpr int kBRows = 32 * kBWaves;  // weight rows per workgroup
constexpr int kBTiles = 4;            // tiles of 32 states a workgroup holds at most
constexpr int kBPieces = 512;         // 16-byte pieces of a tile's activations (32 x 256)

struct BatchArgs {
  const uint8_t* w;
  int64_t rows, row_bytes;
  const int8_t* aqs;  // [nb][cols]
  const float* ad;    // [nb][nblk]
  int nb, nblk, groups, row_tiles;
  float* y;
};

__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, (v2u)(__builtin_bit_cast(v2u, a) * __builtin_bit_cast(v2u, b)));
}
// the 16-bit halves of a * b + c, and a >> 7 (signed)
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_bit_cast(
      uint32_t, (v2u)(__builtin_bit_cast(v2u, a) * __builtin_bit_cast(v2u, b) + __builtin_bit_cast(v2u, c)));
}
__device__ __forceinline__ uint32_t pk_sar7(uint32_t a) {
  return __builtin_bit_cast(uint32_t, (v2s)(__builtin_bit_cast(v2s, a) >> (short)7));
}
// byte k of `w` in the low byte of both halves (zero or sign extended)
__device__ __forceinline__ uint32_t dup_u8(uint32_t w, int k) {
  return __builtin_amdgcn_perm(0u, w, 0x0c000c00u | (uint32_t)k | ((uint32_t)k << 16));
}
__device__ __forceinline__ uint32_t dup_i8(uint32_t w, int k) {
  return ((uint32_t)__builtin_amdgcn_sbfe((int)w, 8 * k, 8) & 0xFFFFu) * 0x10001u;
}

// The planes of one word of four products from its even and odd 16-bit pairs.
__device__ __forceinline__ void split7(uint32_t pe, uint32_t po, int& lo, int& hi) {
  lo = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) & 0x7F7F7F7Fu);
  hi = (int)__builtin_amdgcn_perm(pk_sar7(po), pk_sar7(pe), 0x06020400u);
}

// One lane's raw bytes of a block (half h of every 32 weights) and the planes
// made from them: L[s], H[s] hold weights 32 s + 16 h .. + 15.
template <int T>
struct Raw;

template <bool FIVE>
struct RawK45 {
  static constexpr int TS = FIVE ? 176 : 144;
  static constexpr bool MIN = true;
  static constexpr int kShift = FIVE ? 7 : 3;
  uint4 hd, qs[4], qh;
  __device__ void load(const uint8_t* blk, int h) {
    hd = lm_ld_16(blk);
#pragma unroll
    for (int j = 0; j < 4; ++j) qs[j] = lm_ld_16(blk + (FIVE ? 48 : 16) + 32 * j + 16 * h);
    if (FIVE) qh = lm_ld_16(blk + 16 + 16 * h);
  }
  __device__ void planes(int h, v4i (&L)[8], v4i (&H)[8], v8h& mins, float& d, float& dmin) const {
    d = lm_half_f(hd.x & 0xFFFF);
    dmin = lm_half_f(hd.x >> 16);
    // getScaleMinK4 (quant.nim:156-162) of the eight sub-blocks
    const uint32_t sc[2] = {hd.y & 0x3F3F3F3Fu, (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u)};
    const uint32_t mn = h ? ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3F3F3F3Fu;
#pragma unroll
    for (int k = 0; k < 8; ++k) mins[k] = (_Float16)(short)((mn >> (8 * (k >> 1))) & 0xFF);
    const uint32_t qhw[4] = {qh.x, qh.y, qh.z, qh.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t q[4] = {qs[j].x, qs[j].y, qs[j].z, qs[j].w};
#pragma unroll
      for (int nib = 0; nib < 2; ++nib) {
        const int s = 2 * j + nib;
        const uint32_t scw = sc[s >> 2];
        if constexpr (!FIVE) {
          const uint32_t sl = dup_u8(scw & 0x07070707u, s & 3), sh = dup_u8((scw >> 3) & 0x07070707u, s & 3);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t v = (nib ? q[k] >> 4 : q[k]) & 0x0F0F0F0Fu;
            L[s][k] = (int)pk_mul(v, sl);
            H[s][k] = (int)pk_mul(v, sh);
          }
        } else {
          const uint32_t m = dup_u8(scw, s & 3);
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t v = ((nib ? q[k] >> 4 : q[k]) & 0x0F0F0F0Fu) | (((qhw[k] >> s) & 0x01010101u) << 4);
            int lo, hi;
            split7(pk_mul(v & 0x00FF00FFu, m), pk_mul((v >> 8) & 0x00FF00FFu, m), lo, hi);
            L[s][k] = lo;
            H[s][k] = hi;
          }
        }
      }
    }
  }
  // a.d * (d * sumi - dmin * summ)  (quant.nim:694, :728)
  __device__ static float term(float ad, float d, float dmin, float sumi, float summ) {
    return __fmul_rn(ad, __fsub_rn(__fmul_rn(d, sumi), __fmul_rn(dmin, summ)));
  }
};
template <>
struct Raw<12> : RawK45<false> {};
template <>
struct Raw<13> : RawK45<true> {};

template <>
struct Raw<14> {
  static constexpr int TS = 210;
  static constexpr bool MIN = false;
  static constexpr int kShift = 7;
  uint4 ql[2][2], qh[2], sc;
  uint32_t dh;
  __device__ void load(const uint8_t* blk, int h) {
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      ql[n][0] = lm_ld_16(blk + 64 * n + 16 * h);
      ql[n][1] = lm_ld_16(blk + 64 * n + 32 + 16 * h);
      qh[n] = lm_ld_16(blk + 128 + 32 * n + 16 * h);
    }
    sc = lm_ld_16(blk + 192);
    dh = lm_ld_u16(blk + 208);
  }
  __device__ void planes(int h, v4i (&L)[8], v4i (&H)[8], v8h&, float& d, float&) const {
    d = lm_half_f(dh);
    const uint32_t scw[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const uint32_t A[2][4] = {{ql[n][0].x, ql[n][0].y, ql[n][0].z, ql[n][0].w},
                                {ql[n][1].x, ql[n][1].y, ql[n][1].z, ql[n][1].w}};
      const uint32_t Q[4] = {qh[n].x, qh[n].y, qh[n].z, qh[n].w};
#pragma unroll
      for (int m = 0; m < 4; ++m) {  // quarter m of the half: weights 128 n + 32 m + 16 h ..
        const int s = 4 * n + m;
        // scale 8 n + 2 m + h: byte 2 (m & 1) + h of word 2 n + (m >> 1)
        const uint32_t w = scw[2 * n + (m >> 1)] >> (8 * h);
        const uint32_t f = dup_i8(w, 2 * (m & 1));
        const uint32_t off = pk_mul(f, 0xFFE0FFE0u);  // -32 f
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t lowq = A[m & 1][k] >> (4 * (m >> 1));
          const uint32_t hiq = m < 2 ? Q[k] << (4 - 2 * m) : Q[k] >> (2 * m - 4);
          const uint32_t v = (lowq & 0x0F0F0F0Fu) | (hiq & 0x30303030u);
          int lo, hi;
          split7(pk_mad(v & 0x00FF00FFu, f, off), pk_mad((v >> 8) & 0x00FF00FFu, f, off), lo, hi);
          L[s][k] = lo;
          H[s][k] = hi;
        }
      }
    }
  }
  // a.d * d * sumi  (quant.nim:759)
  __device__ static float term(float ad, float d, float, float sumi, float) {
    return __fmul_rn(__fmul_rn(ad, d), sumi);
  }
};

// LDS of one block's activations for TILES x 32 states, double-buffered.
template <int TILES>
struct BatchLds {
  v4i act[2][TILES][kBPieces];                // [matrix step][lane], swizzled (below)
  __align__(16) _Float16 bs[2][TILES][32][16];  // the states' sums of 16 activations
  __align__(16) float ad[2][TILES * 32];
};

// Workgroup: rows row_tile * 128 .. (32 per wave), states group * 32 TILES ..
// A tile's activations sit in 16-byte pieces: piece (step s, half h, state b)
// at slot 64 s + 32 h + (b ^ (8 ((2 s + h) & 3))), so that both the staging
// writes (8 states x 8 pieces of a wave) and the operand reads (64 lanes of a
// step) spread over the banks.
template <int T, int TILES>
__global__ __launch_bounds__(kBNT, 2) void lm_batch_kernel(BatchArgs a) {
  using R = Raw<T>;
  __shared__ BatchLds<TILES> sm;
  const int tid = (int)threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  // workgroups of one row tile (its state groups) follow each other on one
  // XCD, so the later ones find the weights in its L2
  const int xcd = (int)blockIdx.x & 7, seq = (int)blockIdx.x >> 3;
  const int row_tile = (seq / a.groups) * 8 + xcd, group = seq % a.groups;
  if (row_tile >= a.row_tiles) return;  // the whole workgroup
  const int h = lane >> 5, li = lane & 31;
  const int64_t r = (int64_t)row_tile * kBRows + wave * 32 + li;
  const uint8_t* wrow = a.w + min(r, a.rows - 1) * a.row_bytes;
  const int b0 = group * 32 * TILES;
  const int cols = a.nblk * 256;
  // staging: this thread's two pieces of a tile are pieces k16 and k16 + 8 of
  // state sb (states past nb repeat the last and are not stored)
  const int sb = tid >> 3, k16 = tid & 7;
  auto src = [&](int t, int ib, int u) {
    const int b = min(b0 + 32 * t + sb, a.nb - 1);
    return a.aqs + (int64_t)b * cols + ib * 256 + 16 * (k16 + 8 * u);
  };
  auto put = [&](int buf, int t, int u, v4i v) {
    const int k = k16 + 8 * u;
    sm.act[buf][t][32 * k + (sb ^ (8 * (k & 3)))] = v;
    if constexpr (R::MIN) {
      int s = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_sdot4(0x01010101, v[j], s, false);
      sm.bs[buf][t][sb][k] = (_Float16)(short)s;
    }
  };
  auto put_ad = [&](int buf, int ib) {
    if (tid < 32 * TILES) sm.ad[buf][tid] = a.ad[(int64_t)min(b0 + tid, a.nb - 1) * a.nblk + ib];
  };
  R raw;
  raw.load(wrow, h);
  put_ad(0, 0);
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u) put(0, t, u, *reinterpret_cast<const v4i*>(src(t, 0, u)));
  v16f acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = v16f{};
  for (int ib = 0; ib < a.nblk; ++ib) {
    const int buf = ib & 1;
    const bool more = ib + 1 < a.nblk;
    const int nx = more ? ib + 1 : ib;  // (the last block is requested twice; nothing reads the second)
    // loads are waited for in order: the first tile's next activations (L2)
    // go out before the next weights (HBM), both as early as registers allow
    v4i nxt[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) nxt[u] = *reinterpret_cast<const v4i*>(src(0, nx, u));
    v4i L[8], H[8];
    v8h mins{};
    float d, dmin = 0.0f;
    raw.planes(h, L, H, mins, d, dmin);
    raw.load(wrow + (int64_t)nx * R::TS, h);
    // block ib's activations are in; every wave is past block ib - 1, whose
    // buffer takes block ib + 1's
    __syncthreads();
    put_ad(buf ^ 1, nx);
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      if (t > 0) {
#pragma unroll
        for (int u = 0; u < 2; ++u) nxt[u] = *reinterpret_cast<const v4i*>(src(t, nx, u));
      }
      v16i sl{}, sh{};
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const v4i x = sm.act[buf][t][64 * s + 32 * h + (li ^ (8 * ((2 * s + h) & 3)))];
        sl = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, L[s], sl, 0, 0, 0);
        sh = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, H[s], sh, 0, 0, 0);
      }
      v16f summ{};
      if constexpr (R::MIN) {
        const v8h x = *reinterpret_cast<const v8h*>(&sm.bs[buf][t][li][8 * h]);
        summ = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, mins, summ, 0, 0, 0);
      }
      // element i of this lane: state 32 t + 8 (i / 4) + 4 h + i % 4, its row
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4f adv = *reinterpret_cast<const v4f*>(&sm.ad[buf][32 * t + 8 * g + 4 * h]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int i = 4 * g + j;
          const float sumi = (float)(sl[i] + (int)((uint32_t)sh[i] << R::kShift));
          acc[t][i] = __fadd_rn(acc[t][i], R::term(adv[j], d, dmin, sumi, summ[i]));
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) put(buf ^ 1, t, u, nxt[u]);
    }
  }
  if (r >= a.rows) return;
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int b = b0 + 32 * t + 8 * (i >> 2) + 4 * h + (i & 3);
      if (b < a.nb) a.y[(int64_t)b * a.rows + r] = acc[t][i];
    }
}

template <int T, int TILES>
void launch(const BatchArgs& a, hipStream_t s) {
  const unsigned grid = (unsigned)((a.row_tiles + 7) / 8 * 8 * a.groups);
  hipLaunchKernelGGL((lm_batch_kernel<T, TILES>), dim3(grid), dim3(kBNT), 0, s, a);
}

template <int T>
hipError_t launch_type(const LmHeadCall& c, hipStream_t s) {
  BatchArgs a{static_cast<const uint8_t*>(c.w), c.rows, c.row_bytes, c.act_qs, c.act_d, c.nb, (int)(c.cols / 256),
              0, (int)((c.rows + kBRows - 1) / kBRows), c.y};
  const int tiles = (c.nb + 31) / 32;
  a.groups = (tiles + kBTiles - 1) / kBTiles;
  // (the grid's index is 32 bits; a matrix past this does not fit the memory)
  if ((c.rows + kBRows - 1) / kBRows > (int64_t{1} << 29) / a.groups) return hipErrorInvalidConfiguration;
  const int per = (tiles + a.groups - 1) / a.groups;
  switch (per) {
    case 1: launch<T, 1>(a, s); break;
    case 2: launch<T, 2>(a, s); break;
    case 3: launch<T, 3>(a, s); break;
    default: launch<T, 4>(a, s); break;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_lm_batch(const LmHeadCall& c, hipStream_t s) {
  switch (c.type) {
    case 12: return launch_type<12>(c, s);
    case 13: return launch_type<13>(c, s);
    default: return launch_type<14>(c, s);
  }
}

}  // namespace nls
