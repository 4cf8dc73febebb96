// q8_pack.hip -- quantize + pack kernel for gfx950.
//
// Bit-exact restatement of pack_q8 (qwen3_mojo/scripts/quantize.py:31-43):
//   per group of G weights along the input dim
//     scale = max|w| / 127             f32, correctly rounded division (:36)
//     scale = max(scale, 1e-8f)        f32; NaN stays NaN (:37)
//     scale16 = RNE f16(scale)         binary16 with denormals (:37)
//     q = rint(w / f32(scale16))       correctly rounded division, ties-even (:38)
//     q = clip(q, -127, 127) -> int8   NaN (0/0 for scale16 == 0) -> 0 (:39)
//   packed row: [scale16 x m/G | int8 x m] (:41-42)
// With SCALE_F32 the f16 rounding is skipped and each scale is an f32.
//
// Mapping: one thread per 16 consecutive weights, so a group of G weights is
// G/16 adjacent lanes of one wavefront (aligned, never straddling a wave).
// The group's |max| is reduced across those lanes with DPP moves; each lane
// writes its 16 codes with one store, and the group's first lane the scale.
//
// What bounds it: HBM, once the divisions are out of the way.  A correctly
// rounded f32 division is about 12 VALU operations per weight, which took
// 100 us for 28672 x 4096 (3.5 TB/s, f16 scales, bf16 source) whatever the
// loads did.  Instead r = w * (1 / scale) decides rint(w / scale) wherever r
// lies further from a tie than the two can differ (see quant16); the rare
// rest divides: 62 us, 5.7 TB/s of the 356 MB read and written.
//
// This file must be compiled without fast-math and with correctly rounded
// f32 division (-fhip-fp32-correctly-rounded-divide-sqrt, hipcc's default).
#include "q8_device.h"
#include "q8_launch.h"

namespace q8 {
namespace {

template <int CTRL>
__device__ __forceinline__ float dpp_max_step(float v) {
  float o = __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                         0xf, 0xf, false));
  return nanmax(v, o);
}

// 16 weights at element e; 16-byte loads at the source's own alignment
// (VEC_LOAD: 16 bytes, else that of one element).
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
template <bool SRC_F32, bool VEC_LOAD>
__device__ __forceinline__ void load16(const void *src, int64_t e, float (&v)[16]) {
  if constexpr (SRC_F32) {
    const float *p = reinterpret_cast<const float *>(src) + e;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x4 a = VEC_LOAD ? *reinterpret_cast<const f32x4 *>(p + 4 * c)
                               : *reinterpret_cast<const f32x4_a4 *>(p + 4 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[4 * c + i] = a[i];
    }
  } else {
    const uint16_t *p = reinterpret_cast<const uint16_t *>(src) + e;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const u32x4 a = VEC_LOAD ? *reinterpret_cast<const u32x4 *>(p + 8 * c)
                               : *reinterpret_cast<const u32x4_a2 *>(p + 8 * c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[8 * c + 2 * i] = __builtin_bit_cast(float, a[i] << 16);
        v[8 * c + 2 * i + 1] = __builtin_bit_cast(float, a[i] & 0xffff0000u);
      }
    }
  }
}

__device__ __forceinline__ int32_t quant1(float w, float sf) {
  float r = w / sf;                 // correctly rounded f32 division
  float q = __builtin_rintf(r);     // round half to even
  if (q != q) return 0;             // NaN -> 0 (numpy's float->int8 cast)
  q = q > 127.0f ? 127.0f : q;
  q = q < -127.0f ? -127.0f : q;
  return (int32_t)q;
}

// 16 codes, four per dword.  t = w / sf exactly; the code is rint(fl(t)).
// r = fl(w * rcp(sf)) is within 2^-22 |t| of t (1 ulp of the reciprocal, half
// an ulp of the product) and fl(t) within 2^-24 |t|, so where r is further
// than 5e-7 |r| (2^-20.9) from a half-integer both round to the same
// integer.  Anything else -- near ties, NaN and infinities, sf zero or past
// the normal range -- takes the division.
__device__ __forceinline__ u32x4 quant16(const float (&v)[16], float sf) {
  const float inv = __builtin_amdgcn_rcpf(sf);
  bool exact = !(sf > 1e-37f && sf < 8e37f);
  u32x4 o;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    uint32_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float r = v[4 * d + i] * inv;
      float q = __builtin_rintf(r);
      exact |= !(__builtin_fmaf(__builtin_fabsf(r), 5e-7f, __builtin_fabsf(r - q)) < 0.5f);
      q = __builtin_amdgcn_fmed3f(q, -127.0f, 127.0f);
      b[i] = (uint32_t)(int32_t)q;
    }
    // low bytes of the four
    o[d] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u),
                                 __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u), 0x05040100u);
  }
  if (exact) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) w |= ((uint32_t)quant1(v[4 * d + i], sf) & 0xffu) << (8 * i);
      o[d] = w;
    }
  }
  return o;
}

template <int G, int KIND, bool SRC_F32, bool VEC_LOAD>
__global__ __launch_bounds__(256) void pack_kernel(
    const void *__restrict__ src, int64_t n, int64_t m,
    uint8_t *__restrict__ dst, int64_t dst_row_bytes) {
  constexpr int LPG = G / 16;                      // lanes per group
  constexpr int SB = ScaleTraits<KIND>::bytes;
  const int64_t cpr = m / 16;                      // chunks per row
  const int64_t total = n * cpr;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = t < total;
  int64_t j = 0, c = 0;                            // row, chunk within it
  if (live) {
    j = total <= INT32_MAX ? (int64_t)((uint32_t)t / (uint32_t)cpr) : t / cpr;
    c = t - j * cpr;
  }

  float v[16];
  if (live) {
    load16<SRC_F32, VEC_LOAD>(src, j * m + c * 16, v);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = 0.0f;
  }
  // |max| of each half of the chunk; bit patterns of |v| order as the values
  // do, with NaN above infinity.  With a NaN the halves are scanned in order
  // (the first NaN of a half is its maximum).
  uint32_t h0 = 0, h1 = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    h0 = max(h0, __builtin_bit_cast(uint32_t, v[i]) & 0x7fffffffu);
    h1 = max(h1, __builtin_bit_cast(uint32_t, v[8 + i]) & 0x7fffffffu);
  }
  float a = __builtin_bit_cast(float, h0), b = __builtin_bit_cast(float, h1);
  if (__builtin_amdgcn_ballot_w64(max(h0, h1) > 0x7f800000u)) {
    a = b = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      a = nanmax(a, __builtin_fabsf(v[i]));
      b = nanmax(b, __builtin_fabsf(v[8 + i]));
    }
  }
  // Reduce over the group as a tree of its eighths (halves a, b of the LPG
  // lanes): neighbours, then pairs, then for G = 64 eighth i with 7 - i.
  const float a1 = nanmax(a, b), b1 = nanmax(b, a);
  a = dpp_max_step<0xb1>(a1);                      // quad_perm [1,0,3,2]
  b = dpp_max_step<0xb1>(b1);
  float amax = a;
  if constexpr (LPG == 4)                          // quad_perm [3,2,1,0]
    amax = nanmax(a, dpp_mov<0x1b>(b));
  static_assert(LPG == 2 || LPG == 4, "G must be 32 or 64");

  float sc = amax / 127.0f;
  if (!(sc >= 1e-8f)) sc = (sc != sc) ? sc : 1e-8f;
  float sf;
  uint32_t sbits;
  if constexpr (KIND == SCALE_F16) {
    uint16_t h = f32_to_f16_bits(sc);
    sbits = h;
    sf = f16_bits_to_f32(h);
  } else {
    sf = sc;
    sbits = __builtin_bit_cast(uint32_t, sc);
  }
  if (!live) return;

  uint8_t *row = dst + j * dst_row_bytes;
  // Codes start after (m/G) scales, at 2-byte alignment in general.
  *reinterpret_cast<u32x4_a2 *>(row + (m / G) * SB + c * 16) = quant16(v, sf);
  if (c % LPG == 0) {
    uint16_t *sp = reinterpret_cast<uint16_t *>(row + c / LPG * SB);
    sp[0] = (uint16_t)sbits;
    if constexpr (SB == 4) sp[1] = (uint16_t)(sbits >> 16);
  }
}

template <int G, int KIND>
hipError_t launch_pack_g(const PackArgs &a, hipStream_t st) {
  const int64_t total = a.n * (a.m / 16);
  const int64_t blocks = (total + 255) / 256;
  const uintptr_t base = reinterpret_cast<uintptr_t>(a.src);
  const bool vec = (base % 16 == 0);   // m % 32 == 0 keeps every row aligned
  dim3 grid((unsigned)blocks), block(256);
  if (a.src_is_f32) {
    if (vec)
      hipLaunchKernelGGL((pack_kernel<G, KIND, true, true>), grid, block, 0, st,
                         a.src, a.n, a.m, a.dst, a.dst_row_bytes);
    else
      hipLaunchKernelGGL((pack_kernel<G, KIND, true, false>), grid, block, 0, st,
                         a.src, a.n, a.m, a.dst, a.dst_row_bytes);
  } else {
    if (vec)
      hipLaunchKernelGGL((pack_kernel<G, KIND, false, true>), grid, block, 0, st,
                         a.src, a.n, a.m, a.dst, a.dst_row_bytes);
    else
      hipLaunchKernelGGL((pack_kernel<G, KIND, false, false>), grid, block, 0, st,
                         a.src, a.n, a.m, a.dst, a.dst_row_bytes);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pack(const PackArgs &a, hipStream_t st) {
  if (a.n == 0) return hipSuccess;
  if (a.G == 64 && a.kind == SCALE_F16) return launch_pack_g<64, SCALE_F16>(a, st);
  if (a.G == 64 && a.kind == SCALE_F32) return launch_pack_g<64, SCALE_F32>(a, st);
  if (a.G == 32 && a.kind == SCALE_F16) return launch_pack_g<32, SCALE_F16>(a, st);
  if (a.G == 32 && a.kind == SCALE_F32) return launch_pack_g<32, SCALE_F32>(a, st);
  return hipErrorInvalidValue;
}

}  // namespace q8
