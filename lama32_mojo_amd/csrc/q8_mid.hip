// q8_mid.hip -- Q8 linear at any alignment for two activation rows and up,
// with f32-level error (gfx950).
//
// y[b, j] = sum_g scale[j, g] * sum_{k in g} x[b, k] * q[j, k]
// (k_mm_q8, src/llama_q8.mojo:54-93: unscaled dot per group, then one scale
// multiply per group), in two launches (a third, splitk_reduce_kernel, adds
// the partial sums when K is split over workgroups):
//   1. frag_kernel writes x as bf16 MFMA fragments: bf16 x as it is (NT = 1),
//      f32 x cut into NT = 3 terms of 8 bits each, whose sum is x.  (Each row
//      is scaled by a power of two so that its largest finite |x| lies in
//      [2^14, 2^15), which keeps the terms of the smallest rows in bf16's
//      range: what they leave out lies below 2^-140 of the row's largest
//      value.)
//   2. mid_kernel runs v_mfma_f32_32x32x16_bf16 on the fragments and the
//      codes.  |q| <= 127 is exact in bf16, so the products are exact;
//      a group's partial starts from 0 and is folded into the output with
//      one f32 FMA by the group's scale, as the reference does.
// Its error is that of the f32 sums (0.8-2e-7 of float64).  Two binary16
// terms of a scaled row take two MFMAs instead of three and are 10-30 %
// faster at much the same error on ordinary rows (200 x 1600 x 4800 28 us
// against 32.6, 512 x 11008 x 4096 127 against 172), but carry x to 2^-39 of
// its row's largest value only: beside a channel of 2^34 the rest lost
// percents.
//
// Where it runs: rows or x that are not 16-byte aligned (a row is (m / G) SB
// + m bytes, so most widths that are no multiple of 512 at G = 64 with f16
// scales) with more than a few products, against one wave per output with
// one code per lane and load: 200 x 1600 x 4800 1030 -> 32.6 us, 512 x 11008 x
// 4096 24390 -> 172 us, 20 x 11008 x 4096 960 -> 29 us; and 17 .. 31 aligned
// rows of 4096 codes or more, but for some n (31 x 4096 x 28672 68 -> 45 us);
// both lines are drawn in the dispatch.
//
// Layout: a workgroup owns 32 RT rows x 32 KW columns, wave w 32 columns of
// them, and a range of 64-code units of K.  Per phase of two units (PU)
// the workgroup stages the tile's x fragments in LDS (double-buffered, one
// barrier per phase) and each wave its own codes: loaded LPR lanes to a row,
// in runs of 64 PU bytes, and read back from LDS as the MFMA takes them, 16
// bytes of column l % 32 per lane.  (Loading them in that layout directly
// costs the L1 one access per lane, since neighbouring lanes then sit on
// different rows: 16 x 4096 x 28672 took 45 us that way against 37.)
// The order of k within a unit is free as long as a step stays in its
// group: lane half h feeds codes 32 h + 16 p + 8 e .. +8 in step 2 p + e
// (G = 64), or 32 p + 16 h + 8 e .. +8 (G = 32); frag_kernel lays x out to
// match, one contiguous KiB per (32 rows, step, term).
// What bounds it: below about 100 rows the codes' way through a phase of
// two units (1.1 us at RT = 1 and 256 workgroups), then the MFMAs; about 5 us
// per launch are its start, the first loads and the last stores, and the two
// launches around it cost 3 us each, which is what small shapes pay (16 x
// 1600 x 4800: 14 us).
//
// Alignment: packed rows start at any even byte, so codes and scales are
// loaded as vectors of 2-byte alignment (one instruction; the hardware
// splits those that straddle a line), f32 x as vectors of 4-byte alignment.
#include "q8_device.h"
#include "q8_launch.h"

namespace q8 {
namespace {

// 16 bytes at 2-byte (packed rows), 4-byte (f32 x) or 2-byte (bf16 x) alignment
struct __attribute__((packed, aligned(2))) Codes16 { uint32_t d[4]; };
struct __attribute__((packed, aligned(4))) Floats4 { float v[4]; };

__device__ __forceinline__ u32x4 load_codes16(const uint8_t *p) {
  const Codes16 c = *reinterpret_cast<const Codes16 *>(p);
  return u32x4{c.d[0], c.d[1], c.d[2], c.d[3]};
}

constexpr int kUnit = 64;            // codes of a row per unit
constexpr int PU = 2;                // units per phase
// Workgroups that the K split aims at, one per CU: 512 made 16 x 4096 x
// 28672 41.8 -> 44.0 us and 200 x 1600 x 4800 28.2 -> 35.8 us.
constexpr int kTarget = 256;

// ---- 1. x as bf16 fragments ---------------------------------------------------
// One 256-thread block per row r.  Fragment block (row tile r / 32, unit,
// step, term) is 64 lanes x 8 values; see the file comment for the order of
// k.  Values past m (a last unit of 32 codes, and one unit of zeros behind
// the row) are zeros.  The exponent is
// that of the largest finite value: infinities and NaN stay what they are in
// the first term (the others 0) and do not change the rest of their row.
// With CH > 0 the row (m <= 2048 CH) stays in registers between the maximum
// and the conversion; CH = 0 reads it twice.
template <bool XF32, int NT, int G, int CH>
__global__ __launch_bounds__(256) void frag_kernel(const void *__restrict__ xv, int64_t m,
                                                   __bf16 *__restrict__ xf,
                                                   int *__restrict__ ex) {
  __shared__ float red[4];
  const int64_t r = blockIdx.x;
  const int tid = threadIdx.x;
  const int64_t nu = (m + kUnit - 1) / kUnit;
  auto load8 = [&](int64_t k, float (&v)[8]) {
    if constexpr (XF32) {
      const Floats4 *p = reinterpret_cast<const Floats4 *>(static_cast<const float *>(xv) + r * m + k);
      const Floats4 a = p[0], b = p[1];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v[c] = a.v[c];
        v[4 + c] = b.v[c];
      }
    } else {
      const Codes16 d = *reinterpret_cast<const Codes16 *>(static_cast<const uint16_t *>(xv) + r * m + k);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        v[2 * c] = __builtin_bit_cast(float, d.d[c] << 16);
        v[2 * c + 1] = __builtin_bit_cast(float, d.d[c] & 0xffff0000u);
      }
    }
  };
  float mx = 0.0f;
  auto maximum = [&](const float (&v)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float a = fabsf(v[j]);
      mx = fmaxf(mx, a <= 3.4028235e38f ? a : 0.0f);
    }
  };
  float rv[CH > 0 ? CH : 1][8];
  if constexpr (CH > 0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t k = 8 * tid + 2048 * c;
      if (k < m) {
        load8(k, rv[c]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) rv[c][j] = 0.0f;
      }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) maximum(rv[c]);
  } else {
    for (int64_t k = 8 * tid; k < m; k += 2048) {
      load8(k, rv[0]);
      maximum(rv[0]);
    }
  }
  mx = wave_max(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  int e = 0;
  if (mx > 0.0f) {
    e = (int)((__builtin_bit_cast(uint32_t, mx) >> 23) & 255u) - 127 - 14;
    e = e < -126 ? -126 : e;                 // (subnormal maxima: as far as 2^126 goes)
  }
  __bf16 *row = xf + (r >> 5) * (nu + 1) * (4 * NT * 512) + (r & 31) * 8;
  auto store8 = [&](int64_t k, const float (&v)[8]) {
    const int kk = (int)(k & 63);
    const int hf = G == 64 ? kk >> 5 : (kk >> 4) & 1;
    const int p = G == 64 ? (kk >> 4) & 1 : kk >> 5;
    const int step = 2 * p + ((kk >> 3) & 1);
    __bf16 *dst = row + ((k >> 6) * 4 + step) * (NT * 512) + hf * 256;
    float rest[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) rest[j] = __builtin_ldexpf(v[j], -e);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      // the upper 8 bits of what is left; the subtraction is exact
      u32x4 o;
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = pk_hi16(rest[2 * c], rest[2 * c + 1]);
      *reinterpret_cast<u32x4 *>(dst + 512 * t) = o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = rest[j] - __builtin_bit_cast(
            float, __builtin_bit_cast(uint32_t, rest[j]) & 0xffff0000u);
        rest[j] = d == d ? d : 0.0f;           // inf - inf and NaN: the first term alone
      }
    }
  };
  const int64_t kend = (nu + 1) * kUnit;
  if constexpr (CH > 0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int64_t k = 8 * tid + 2048 * c;
      if (k < m) store8(k, rv[c]);
    }
  } else {
    for (int64_t k = 8 * tid; k < m; k += 2048) {
      load8(k, rv[0]);
      store8(k, rv[0]);
    }
  }
  for (int64_t k = m + 8 * tid; k < kend; k += 2048) {
    const float zero[8] = {};
    store8(k, zero);
  }
  if (tid == 0) ex[r] = e;
}

template <bool XF32, int NT, int G>
void launch_frag(const LinearArgs &a, __bf16 *xf, int *ex, hipStream_t st) {
  const dim3 grid((unsigned)a.s), block(256);
  if (a.m <= 4096)
    hipLaunchKernelGGL((frag_kernel<XF32, NT, G, 2>), grid, block, 0, st, a.x, a.m, xf, ex);
  else if (a.m <= 16384)
    hipLaunchKernelGGL((frag_kernel<XF32, NT, G, 8>), grid, block, 0, st, a.x, a.m, xf, ex);
  else
    hipLaunchKernelGGL((frag_kernel<XF32, NT, G, 0>), grid, block, 0, st, a.x, a.m, xf, ex);
}

// ---- 2. the linear ------------------------------------------------------------
template <int N> struct __attribute__((packed, aligned(2))) Dwords { uint32_t d[N]; };

// One workgroup: 32 RT rows x 32 KW columns over units [u0, u1) of K, wave
// w owning columns 32 w .. of the tile.
template <int G, int KIND, int NT, int RT, int KW>
__global__ __launch_bounds__(64 * KW) __attribute__((amdgpu_waves_per_eu(2)))
void mid_kernel(const uint8_t *__restrict__ w, int64_t row_bytes, const __bf16 *__restrict__ xf,
                const int *__restrict__ ex, float *__restrict__ y, int s, int m, int64_t n,
                int ncb, int nrb, int nks, int upk, float *__restrict__ ws) {
  constexpr int SB = ScaleTraits<KIND>::bytes;
  constexpr int GPU_ = kUnit / G;                      // groups per unit
  constexpr int UB = GPU_ * SB;                        // scale bytes per unit
  constexpr int SD = PU * UB / 4;                      // scale dwords per phase
  constexpr int SPG = 4 / GPU_;                        // steps per group
  constexpr int XU = 4 * NT;                           // fragments of a row tile per unit
  constexpr int XF = PU * RT * XU;                     // ... of the tile per phase
  constexpr int XL = XF / KW;                          // ... loaded by each wave
  constexpr int LPR = 4 * PU, RPI = 64 / LPR;          // lanes per row, rows per load of codes
  constexpr int WL = 32 / RPI;                         // loads of codes per column tile
  static_assert(XF % KW == 0 && PU * UB % 4 == 0, "whole fragments and scale dwords");
  __shared__ bf16x8_t xs[2][XF][64];
  __shared__ __attribute__((aligned(16))) int exs[32 * RT];
  __shared__ __attribute__((aligned(16))) uint8_t cl[KW][32][PU * kUnit + 16];

  // Workgroups go to the 8 XCDs in turn: workgroup id runs on XCD id % 8.
  // The row blocks of a (column block, K split) take consecutive turns of
  // one XCD, so its L2 serves the codes to all but the first of them.
  const int id = blockIdx.x, per = id >> 3;
  const int cs = (per / nrb) * 8 + (id & 7), rb = per % nrb;
  const int cb = cs / nks, ks = cs % nks;
  if (cb >= ncb) return;
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = ((int64_t)cb * KW + wid) * 32;
  const int nu = (m + kUnit - 1) / kUnit;
  const int u0 = ks * upk;                             // (no split is empty)
  const int u1 = u0 + upk < nu ? u0 + upk : nu;

  // row exponents: loaded ahead of everything, published by the first barrier
  static_assert(32 * RT <= 64 * KW, "one row exponent per thread");
  const int et = threadIdx.x < 32 * RT ? threadIdx.x : 0;
  const int exv = ex[min(rb * 32 * RT + et, s - 1)];

  // Codes are loaded LPR lanes to a row (PU 64-byte units in one run) and
  // scales by the lane whose column it is; rows past n read the last one and
  // are not stored.
  const int64_t nb = n0 < n ? n0 : n - 1;
  const uint8_t *wb = w + nb * row_bytes;
  const int last = (int)(n - 1 - nb < 32 ? n - 1 - nb : 31);
  const int piece = lane % LPR;
  const uint32_t soff = (uint32_t)(min(lr, last) * row_bytes);
  uint32_t coff[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i)
    coff[i] = (uint32_t)(min(i * RPI + lane / LPR, last) * row_bytes + (m / G) * SB);
  // the fragments this wave stages: numbers wid + KW i of the phase's XF
  // (unit, row tile, fragment)
  const int ntile = (s + 31) / 32;
  const __bf16 *xt[XL];                              // (uniform: scalar base, lane offset)
  int xun[XL];                                         // unit of the phase
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int f = wid + KW * i;
    const int t = rb * RT + f / XU % RT;
    xun[i] = f / (XU * RT);
    xt[i] = xf + ((int64_t)(t < ntile ? t : ntile - 1) * (nu + 1) * XU + f % XU) * 512;
  }

  const uint32_t lane16 = 16u * lane;
  u32x4 W[2][WL];
  bf16x8_t X[2][XL];
  Dwords<SD> SC[2];
  // Units past u1 take the unit of zeros behind the row of x and reread the
  // codes of the last unit, and a last unit of 32 codes reads its first
  // piece twice: no load leaves its row.  (A scale load that starts in
  // a row's scale section reads at most 32 - SB bytes past it, and the codes
  // that follow are at least 32 bytes.)
  // A phase past u1 (two are loaded behind the last) reads one line per load:
  // its offsets are masked to 0.
  auto load_phase = [&](int st, int up) {
    const uint32_t on = up < u1 ? 0xffffffffu : 0u;
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int u = up + xun[i] < u1 ? up + xun[i] : nu;
      X[st][i] = *reinterpret_cast<const bf16x8_t *>(
          reinterpret_cast<const uint8_t *>(xt[i] + (int64_t)u * (XU * 512)) + (lane16 & on));
    }
    const int us = up < u1 ? up : u1 - 1;
    SC[st] = *reinterpret_cast<const Dwords<SD> *>(wb + ((soff + (uint32_t)(us * UB)) & on));
    const int un = up + piece / 4 < u1 ? up + piece / 4 : u1 - 1;
    const int k = un * kUnit + 16 * (un * kUnit + 32 < m ? piece & 3 : piece & 1);
#pragma unroll
    for (int i = 0; i < WL; ++i) W[st][i] = load_codes16(wb + ((coff[i] + (uint32_t)k) & on));
    __builtin_amdgcn_sched_barrier(0);
  };
  // register stage st to x buffer st and the wave's code rows (a wave's LDS
  // operations run in order: its reads of the phase before are done)
  auto store_phase = [&](int st) {
#pragma unroll
    for (int i = 0; i < XL; ++i) xs[st][wid + KW * i][lane] = X[st][i];
#pragma unroll
    for (int i = 0; i < WL; ++i)
      *reinterpret_cast<u32x4 *>(&cl[wid][i * RPI + lane / LPR][16 * piece]) = W[st][i];
  };

  f32x16 acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[t][v] = 0.0f;

  // The PU RT blocks (unit up + v, row tile t) of a phase, from register
  // stage and x buffer st, as a chain of groups.  A group sums its terms from
  // the smallest up, so that only the last of them round at the size of the
  // sum (200 x 1600 x 4800 in order of the steps 1.13e-7 of float64, now
  // 0.83e-7).  Fragments are read from LDS AH ahead of their MFMA (4 of three
  // terms: 1 % slower; 6: spills), and a group's partials are folded into the
  // output behind the MFMAs of the next group.  Nothing is skipped: units
  // past u1 and groups past m met zeros of x, and their scale is forced to 0.
  auto compute = [&](int st, int up, const Dwords<SD> &scd) {
    constexpr int FPG = SPG * NT;              // fragments per group
    constexpr int NG = PU * RT * GPU_, NF = NG * FPG, AH = NT == 1 ? 4 : 3;
    bf16x8_t a[AH + 1], b[4];
    u32x4 q[2][2];
    f32x16 d[2];
    auto read_a = [&](int f) {
      const int r = f % FPG;
      a[f % (AH + 1)] = xs[st][(f / FPG * SPG + r % SPG) * NT + NT - 1 - r / SPG][lane];
    };
    auto read_q = [&](int v) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
        q[v & 1][p] = *reinterpret_cast<const u32x4 *>(
            &cl[wid][lr][kUnit * v + (G == 64 ? 32 * lh + 16 * p : 32 * p + 16 * lh)]);
    };
    auto fold = [&](int j) {
      const int blk = j / GPU_, g = j % GPU_, v = blk / RT, t = blk % RT;
      const bool live = up + v < u1 && (up + v) * kUnit + g * G < m;
      const int byte = v * UB + g * SB;
      const uint32_t raw = scd.d[byte >> 2];
      float sc = KIND == SCALE_F16 ? f16_bits_to_f32((uint16_t)(raw >> (8 * (byte & 3))))
                                   : __builtin_bit_cast(float, raw);
      sc = live ? sc : 0.0f;
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[t][e] = __builtin_fmaf(sc, d[j & 1][e], acc[t][e]);
    };
    read_q(0);
#pragma unroll
    for (int f = 0; f < AH; ++f) read_a(f);
#pragma unroll
    for (int j = 0; j < NG; ++j) {
      const int blk = j / GPU_, v = blk / RT;
#pragma unroll
      for (int r = 0; r < FPG; ++r) {
        const int f = j * FPG + r;
        if (f + AH < NF) read_a(f + AH);
        if (r == 0 && j % GPU_ == 0 && blk % RT == RT - 1 && v + 1 < PU) read_q(v + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (r == 0 && j % (GPU_ * RT) == 0) {  // the unit's codes, step 2 p + e
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            b[2 * p] = codes_to_bf16(q[v & 1][p].x, q[v & 1][p].y);
            b[2 * p + 1] = codes_to_bf16(q[v & 1][p].z, q[v & 1][p].w);
          }
        }
        f32x16 z;
#pragma unroll
        for (int e = 0; e < 16; ++e) z[e] = 0.0f;
        d[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            a[f % (AH + 1)], b[j % GPU_ * SPG + r % SPG], r == 0 ? z : d[j & 1], 0, 0, 0);
      }
      if (j > 0) fold(j - 1);
    }
    fold(NG - 1);
  };

  // Phase p loads phase p + 2 into register stage p & 1 (stored to LDS in
  // phase p - 1), computes its PU units from LDS, then stores phase p + 1
  // (its x into the buffer last read in phase p - 1).  Two phases per turn,
  // whole: a phase past u1 computes on zeros (a branch between the loads and
  // their use would make the compiler wait for all of them there).
  load_phase(0, u0);
  load_phase(1, u0 + PU);
  exs[et] = exv;                       // (the threads past the rows rewrite row 0's)
  store_phase(0);
  __syncthreads();
  int up = u0;
  do {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const Dwords<SD> scd = SC[st];
      load_phase(st, up + 2 * PU);
      compute(st, up, scd);
      store_phase(st ^ 1);
      __syncthreads();
      up += PU;
    }
  } while (up < u1);

  // D layout: lane -> column lane % 32, element v -> row 8 (v / 4) +
  // 4 (lane / 32) + v % 4.  A K split writes its partial sums to ws.
  float *out = nks > 1 ? ws + (int64_t)ks * s * n : y;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int r0 = (rb * RT + t) * 32 + 4 * lh;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      typedef int i32x4 __attribute__((ext_vector_type(4)));
      const i32x4 e = *reinterpret_cast<const i32x4 *>(&exs[t * 32 + 8 * b + 4 * lh]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t j = n0 + lr;
        const int r = r0 + 8 * b + i;
        if (r < s && j < n) out[(int64_t)r * n + j] = __builtin_ldexpf(acc[t][4 * b + i], e[i]);
      }
    }
  }
}

template <int G, int KIND, int NT, int RT, int KW>
hipError_t launch_t(const LinearArgs &a, const __bf16 *xf, const int *ex, hipStream_t st) {
  const int64_t ncb = (a.n + 32 * KW - 1) / (32 * KW), nrb = (a.s + 32 * RT - 1) / (32 * RT);
  const int nu = (int)((a.m + kUnit - 1) / kUnit);
  int nks = 1;
  if (a.ws)
    while (ncb * nrb * (nks + 1) <= kTarget && nu / (nks + 1) >= 4 &&
           (nks + 1) * a.s * a.n <= a.ws_floats)
      ++nks;
  const int upk = ((nu + nks - 1) / nks + 2 * PU - 1) / (2 * PU) * (2 * PU);
  nks = (nu + upk - 1) / upk;                          // no empty split
  const int64_t blocks = (ncb * nks + 7) / 8 * 8 * nrb;
  hipLaunchKernelGGL((mid_kernel<G, KIND, NT, RT, KW>), dim3((unsigned)blocks), dim3(64 * KW),
                     0, st, a.w, a.row_bytes, xf, ex, a.y, (int)a.s, (int)a.m, a.n, (int)ncb,
                     (int)nrb, nks, upk, a.ws);
  if (nks > 1) return launch_splitk_reduce(a.ws, a.y, a.s * a.n, nks, st);
  return hipGetLastError();
}

template <int G, int KIND>
hipError_t launch_g(const LinearArgs &a, __bf16 *xf, int *ex, hipStream_t st) {
  if (a.x_is_bf16) {
    launch_frag<false, 1, G>(a, xf, ex, st);
    if (a.s <= 32) return launch_t<G, KIND, 1, 1, 4>(a, xf, ex, st);
    return launch_t<G, KIND, 1, 2, 8>(a, xf, ex, st);
  }
  launch_frag<true, 3, G>(a, xf, ex, st);
  if (a.s <= 32) return launch_t<G, KIND, 3, 1, 4>(a, xf, ex, st);
  return launch_t<G, KIND, 3, 2, 8>(a, xf, ex, st);
}

}  // namespace

int64_t mid_rows(int64_t bytes, int64_t m, bool x_is_bf16) {
  const int64_t nu = (m + kUnit - 1) / kUnit;
  const int64_t tile = (nu + 1) * kUnit * 32 * (x_is_bf16 ? 2 : 6) + 32 * 4;
  return bytes / tile * 32;
}

hipError_t launch_mid(const LinearArgs &a, void *scratch, int64_t bytes, hipStream_t st) {
  if (a.s == 0 || a.n == 0) return hipSuccess;
  const int64_t rows = mid_rows(bytes, a.m, a.x_is_bf16);
  if (rows == 0 || a.m >= ((int64_t)1 << 30)) return hipErrorInvalidValue;
  const int64_t nu = (a.m + kUnit - 1) / kUnit;
  const int64_t s = a.s, xb = a.x_is_bf16 ? 2 : 4;
  LinearArgs la = a;
  for (int64_t r0 = 0; r0 < s; r0 += rows) {
    la.s = s - r0 < rows ? s - r0 : rows;
    la.x = static_cast<const uint8_t *>(a.x) + r0 * a.m * xb;
    la.y = a.y + r0 * a.n;
    __bf16 *xf = static_cast<__bf16 *>(scratch);
    int *ex = reinterpret_cast<int *>(static_cast<uint8_t *>(scratch) +
                                      rows * (nu + 1) * kUnit * (a.x_is_bf16 ? 2 : 6));
    hipError_t e = hipErrorInvalidValue;
    if (a.G == 64 && a.kind == SCALE_F16) e = launch_g<64, SCALE_F16>(la, xf, ex, st);
    if (a.G == 64 && a.kind == SCALE_F32) e = launch_g<64, SCALE_F32>(la, xf, ex, st);
    if (a.G == 32 && a.kind == SCALE_F16) e = launch_g<32, SCALE_F16>(la, xf, ex, st);
    if (a.G == 32 && a.kind == SCALE_F32) e = launch_g<32, SCALE_F32>(la, xf, ex, st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace q8
