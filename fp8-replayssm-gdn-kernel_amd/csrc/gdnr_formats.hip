// gdnr_formats.hip -- every checkpoint format of the reference's quantiser on
// gfx950: head, row, tile and vblock granularity, fp8 e4m3fn or int8 codes
// (prototype/gdn_replay_fp8_reference.py:36-37,40-106 quantise, :109-134
// dequantise), for a per-layer choice of format. The decode path itself
// reads vblock/32 fp8; these kernels build and read that and the others.
//
// A scale group is the set of state elements that share one scale:
//   head    rows [0, V)           x columns [0, K)
//   row     row r                 x columns [0, K)
//   tile    rows [i t, (i+1) t)   x columns [j t, (j+1) t)
//   vblock  rows [i t, (i+1) t)   x columns [0, K)
// Quantise: amax = max |x| over the group (NaN propagates), s = amax / qmax
// (qmax 448, or 127 for int8), 1 when amax is not > 0; the stored scale is
// fp16(s). The codes divide by the UNROUNDED s for tile and vblock and by the
// fp16-rounded scale for head and row, as the reference does (ref:83-94).
// fp8: clamp to +-448 keeping NaN, round to nearest even, NaN -> 0x7F|sign.
// int8: round half to even, clamp to +-127, NaN -> 0.
// Dequantise: code * float(stored scale).
//
// Both directions are bound by HBM (4 bytes of state and 1 of code an
// element). stripe_quantize_kernel and stripe_dequantize_kernel take the
// layouts of a GDN state (K = 128, whole 32-row stripes, aligned rows; groups
// of 2^n rows up to 32, or whole stripes up to 8): a wave owns a stripe of 32
// rows, every load and store instruction covers two whole rows, the state
// stays in registers between the amax and the codes (one read), and a group's
// amax is a reduction over the lanes and registers that hold it. At B=64,
// HV=32, V=128 (134 MB of state, 34 of codes; us, against the generic kernels,
// and for vblock32 against a kernel whose lanes held 64 bytes of a row):
//   quantise:   vblock32 29.9 (30.2), tile16 int8 30.6 (256), head 29 (106),
//               row 36 (337): 4.7 to 5.8 TB/s
//   dequantise: vblock32 26.2 (47.7), tile16 int8 27.2 (169), row 27.2 (134):
//               6.2 to 6.4 TB/s
// (Plain instead of non-temporal loads of the state: 31.6 for vblock32; a
// quotient by two f32 corrections instead of one f64 product: 40.6 for row.)
// Other layouts take the generic kernels: one workgroup per scale group, two
// passes over its elements, byte stores.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gdnr_device.h"
#include "gdnr_internal.h"

namespace gdnr {
namespace {

struct Group {
  int r0, c0, R, C;  // rows [r0, r0 + R) x columns [c0, c0 + C) of the head
  int gi, gj;        // index of the group's scale along the scale's last two dims
};

__device__ __forceinline__ Group group_of(const FormatArgs& a, int g) {
  Group q;
  switch (a.gran) {
    case kGranHead: q = {0, 0, a.V, a.K, 0, 0}; break;
    case kGranRow: q = {g, 0, 1, a.K, g, 0}; break;
    case kGranTile: {
      const int nc = a.K / a.tile, i = g / nc, j = g - i * nc;
      q = {i * a.tile, j * a.tile, a.tile, a.tile, i, j};
      break;
    }
    default: q = {g * a.tile, 0, a.tile, a.K, g, 0}; break;  // vblock
  }
  return q;
}

__device__ __forceinline__ int groups_per_head(const FormatArgs& a) {
  switch (a.gran) {
    case kGranHead: return 1;
    case kGranRow: return a.V;
    case kGranTile: return (a.V / a.tile) * (a.K / a.tile);
    default: return a.V / a.tile;
  }
}

__global__ __launch_bounds__(256) void format_quantize_kernel(const FormatArgs a) {
  __shared__ uint32_t red[4];
  __shared__ int red_sat[4];
  const int gph = groups_per_head(a);
  const int64_t item = blockIdx.x;  // (b, hv, group)
  const int g = (int)(item % gph);
  const int hv = (int)((item / gph) % a.HV);
  const int b = (int)(item / ((int64_t)gph * a.HV));
  const Group q = group_of(a, g);
  const float* src = a.state + (int64_t)b * a.st_b + (int64_t)hv * a.st_h;
  const int n = q.R * q.C;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // pass 1: max |x| as bits (NaN above every finite value)
  uint32_t am = 0;
  for (int e = threadIdx.x; e < n; e += 256) {
    const int r = e / q.C, c = e - r * q.C;
    am = max(am, __float_as_uint(src[(int64_t)(q.r0 + r) * a.st_v + q.c0 + c]) & 0x7FFFFFFFu);
  }
  am = wave_max_u32(am);
  if (lane == 0) red[wave] = am;
  __syncthreads();
  am = max(max(red[0], red[1]), max(red[2], red[3]));
  const float qmax = a.int8 ? 127.0f : 448.0f;
  const float amax = __uint_as_float(am);
  const float s32 = (amax > 0.0f) ? amax / qmax : 1.0f;
  const float s16 = (float)(_Float16)s32;
  const float div = (a.gran == kGranHead || a.gran == kGranRow) ? s16 : s32;
  // pass 2: codes
  int sat = 0;
  uint8_t* dst = (uint8_t*)a.payload + (int64_t)b * a.pl_b + (int64_t)hv * a.pl_h;
  for (int e = threadIdx.x; e < n; e += 256) {
    const int r = e / q.C, c = e - r * q.C;
    const int64_t row = q.r0 + r;
    const float y = src[row * a.st_v + q.c0 + c] / div;
    sat += fabsf(y) > qmax ? 1 : 0;
    uint8_t code;
    if (a.int8) {
      const float t = rintf(y);
      code = (uint8_t)(int8_t)(int)((t != t) ? 0.0f : fminf(fmaxf(t, -127.0f), 127.0f));
    } else {
      code = (uint8_t)(f32x4_to_fp8_ref(y, 0.0f, 0.0f, 0.0f) & 0xFFu);
    }
    dst[row * a.pl_v + q.c0 + c] = code;
  }
  sat = wave_sum_i32(sat);
  if (lane == 0) red_sat[wave] = sat;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int64_t so = (int64_t)b * a.sc_b + (int64_t)hv * a.sc_h + (int64_t)q.gi * a.sc_r + (int64_t)q.gj * a.sc_c;
    if (a.scale_dt == DT_F32) ((float*)a.scale)[so] = s16;
    else ((_Float16*)a.scale)[so] = (_Float16)s32;
    if (a.saturated)
      a.saturated[(int64_t)b * a.sa_b + (int64_t)hv * a.sa_h + (int64_t)q.gi * a.sa_r + (int64_t)q.gj * a.sa_c] =
          red_sat[0] + red_sat[1] + red_sat[2] + red_sat[3];
  }
}

__global__ __launch_bounds__(256) void format_dequantize_kernel(const FormatArgs a) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t total = (int64_t)a.B * a.HV * a.V * a.K;
  if (e >= total) return;
  const int c = (int)(e % a.K);
  const int r = (int)((e / a.K) % a.V);
  const int hv = (int)((e / ((int64_t)a.K * a.V)) % a.HV);
  const int b = (int)(e / ((int64_t)a.K * a.V * a.HV));
  int64_t so;
  switch (a.gran) {
    case kGranHead: so = 0; break;
    case kGranRow: so = (int64_t)r * a.sc_r; break;
    case kGranTile: so = (int64_t)(r / a.tile) * a.sc_r + (int64_t)(c / a.tile) * a.sc_c; break;
    default: so = (int64_t)(r / a.tile) * a.sc_r; break;
  }
  so += (int64_t)b * a.sc_b + (int64_t)hv * a.sc_h;
  const float sc = a.scale_dt == DT_F32 ? ((const float*)a.scale)[so] : (float)((const _Float16*)a.scale)[so];
  const uint8_t code = ((const uint8_t*)a.payload)[(int64_t)b * a.pl_b + (int64_t)hv * a.pl_h + (int64_t)r * a.pl_v + c];
  float x;
  if (a.int8) {
    x = (float)(int8_t)code;
  } else {
    float f[4];
    fp8x4_to_f32((uint32_t)code, f);
    x = f[0];
  }
  ((float*)a.state)[(int64_t)b * a.st_b + (int64_t)hv * a.st_h + (int64_t)r * a.st_v + c] = x * sc;
}

// ---- stripes ---------------------------------------------------------------
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kStripe = 32;    // rows of a wave
constexpr int kMaxStripes = 8; // stripes (waves) of one group

// x over the lanes of the group's columns (2^LC lanes of a row's 32) and, for
// a group of several rows, over the two rows a load covers, in every one of them
template <int LC, bool ROWS, class Op>
__device__ __forceinline__ uint32_t group_reduce(uint32_t x, Op op) {
  if constexpr (LC > 0) x = op(x, dpp_u<kDppXor1>(x));
  if constexpr (LC > 1) x = op(x, dpp_u<kDppXor2>(x));
  if constexpr (LC > 2) x = op(x, dpp_u<kDppHalfMirror>(x));
  if constexpr (LC > 3) x = op(x, dpp_u<kDppMirror>(x));
  if constexpr (LC > 4) {
    const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = op(p[0], p[1]);
  }
  if constexpr (ROWS) {
    const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    x = op(p[0], p[1]);
  }
  return x;
}

struct Stripe {
  int b, hv, row0;
};
// the stripe of a wave: flat over (b, hv, V / 32)
__device__ __forceinline__ Stripe stripe_of(const FormatArgs& a, int64_t item) {
  const int per = a.V / kStripe;
  return {(int)(item / ((int64_t)per * a.HV)), (int)((item / per) % a.HV), (int)(item % per) * kStripe};
}

// R rows of the wave's stripe per group (WAVES: the group spans the whole
// workgroup's stripes, R = 32), 2^LC lanes of 4 columns per group. Load j of
// the wave: rows 2 j (lanes 0..31) and 2 j + 1.
template <int R, bool WAVES, int LC, bool INT8>
__global__ __launch_bounds__(WAVES ? 64 * kMaxStripes : 256) void stripe_quantize_kernel(const FormatArgs a) {
  constexpr int JG = R > 1 ? R / 2 : 1;  // loads per group
  constexpr int NG = 16 / JG;            // groups of a lane
  constexpr float qmax = INT8 ? 127.0f : 448.0f;
  __shared__ uint32_t red[WAVES ? kMaxStripes : 1][32], red_sat[WAVES ? kMaxStripes : 1][32];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int64_t item = (int64_t)blockIdx.x * waves + wave;
  if (!WAVES && item >= (int64_t)a.B * a.HV * (a.V / kStripe)) return;
  const Stripe st = stripe_of(a, item);
  const int half = lane >> 5, c4 = lane & 31;
  const float* src = a.state + (int64_t)st.b * a.st_b + (int64_t)st.hv * a.st_h + (int64_t)(st.row0 + half) * a.st_v + 4 * c4;
  u32x4_t x[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) x[j] = __builtin_nontemporal_load((const u32x4_t*)(src + (int64_t)(2 * j) * a.st_v));
  // amax per group as bits of |x| (NaN above every finite value)
  auto umax = [](uint32_t u, uint32_t v) { return max(u, v); };
  uint32_t am[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    am[g] = 0;
#pragma unroll
    for (int j = g * JG; j < (g + 1) * JG; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) am[g] = max(am[g], x[j][e] & 0x7FFFFFFFu);
    am[g] = group_reduce<LC, (R > 1)>(am[g], umax);
  }
  const int gj = c4 >> LC;  // the lane's column group
  if constexpr (WAVES) {
    if (half == 0 && (c4 & ((1 << LC) - 1)) == 0) red[wave][gj] = am[0];
    __syncthreads();
    for (int k = 0; k < waves; ++k) am[0] = max(am[0], red[k][gj]);
  }
  // s = amax / qmax (1 when amax is not > 0); head and row divide by the
  // stored fp16 scale, tile and vblock by s itself
  const bool by16 = a.gran == kGranHead || a.gran == kGranRow;
  float s32[NG], div[NG];
  double rcp[NG];
  bool fast = true;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const float amax = __uint_as_float(am[g]);
    s32[g] = amax > 0.0f ? amax / qmax : 1.0f;
    div[g] = by16 ? (float)(_Float16)s32[g] : s32[g];
    rcp[g] = 1.0 / (double)div[g];
    // (quotient_f64's conditions; an fp16 scale that rounded to zero or
    // infinity fails them)
    fast = fast && quotient_fast(am[g], div[g]) && div[g] < __builtin_inff();
  }
  uint8_t* dst = (uint8_t*)a.payload + (int64_t)st.b * a.pl_b + (int64_t)st.hv * a.pl_h + (int64_t)(st.row0 + half) * a.pl_v + 4 * c4;
  uint32_t sat[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) sat[g] = 0;
  auto codes = [&](auto count, auto quotient, auto fp8) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int g = j / JG;
      float y[4];
      uint32_t w = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = quotient(__uint_as_float(x[j][e]), g);
        if constexpr (decltype(count)::value) sat[g] += fabsf(y[e]) > qmax ? 1 : 0;
        if constexpr (INT8) {
          const float t = rintf(y[e]);
          w |= ((uint32_t)(int)((t != t) ? 0.0f : fminf(fmaxf(t, -127.0f), 127.0f)) & 0xFFu) << (8 * e);
        }
      }
      if constexpr (!INT8) w = fp8(y);
      *(uint32_t*)(dst + (int64_t)(2 * j) * a.pl_v) = w;
    }
  };
  if (__all(fast)) {
    // |y| <= 448 (1 + 2^-23) by s itself, which needs no clamp; an fp16 scale
    // may round far below s (a subnormal one)
    auto quotient = [&](float v, int g) { return quotient_f64(v, rcp[g]); };
    auto fp8 = [&](const float* y) { return f32x4_to_fp8(y[0], y[1], y[2], y[3]); };
    auto fp8_clamped = [&](const float* y) {
      return f32x4_to_fp8(__builtin_amdgcn_fmed3f(y[0], -448.0f, 448.0f), __builtin_amdgcn_fmed3f(y[1], -448.0f, 448.0f),
                          __builtin_amdgcn_fmed3f(y[2], -448.0f, 448.0f), __builtin_amdgcn_fmed3f(y[3], -448.0f, 448.0f));
    };
    if (by16) codes(std::true_type{}, quotient, fp8_clamped);
    else if (a.saturated) codes(std::true_type{}, quotient, fp8);
    else codes(std::false_type{}, quotient, fp8);
  } else {
    codes(std::true_type{}, [&](float v, int g) { return v / div[g]; },
          [&](const float* y) { return f32x4_to_fp8_ref(y[0], y[1], y[2], y[3]); });
  }
  auto uadd = [](uint32_t u, uint32_t v) { return u + v; };
  if (a.saturated) {
#pragma unroll
    for (int g = 0; g < NG; ++g) sat[g] = group_reduce<LC, (R > 1)>(sat[g], uadd);
    if constexpr (WAVES) {
      if (half == 0 && (c4 & ((1 << LC) - 1)) == 0) red_sat[wave][gj] = sat[0];
      __syncthreads();
      sat[0] = 0;
      for (int k = 0; k < waves; ++k) sat[0] += red_sat[k][gj];
    }
  }
  // one lane per group stores its scale (a group of one row: one per half)
  if ((c4 & ((1 << LC) - 1)) != 0 || (R > 1 && half != 0) || (WAVES && wave != 0)) return;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int gi = WAVES ? st.row0 / (kStripe * waves) : R == 1 ? st.row0 + 2 * g + half : st.row0 / R + g;
    const int64_t so = (int64_t)st.b * a.sc_b + (int64_t)st.hv * a.sc_h + (int64_t)gi * a.sc_r + (int64_t)gj * a.sc_c;
    st_dt(a.scale, so, a.scale_dt, (float)(_Float16)s32[g]);
    if (a.saturated)
      a.saturated[(int64_t)st.b * a.sa_b + (int64_t)st.hv * a.sa_h + (int64_t)gi * a.sa_r + (int64_t)gj * a.sa_c] = (int)sat[g];
  }
}

// the same stripes back: lr = log2 of the rows per group within a stripe (5:
// whole stripes, grows rows in all), lc = log2 of the lanes per column group
template <bool INT8>
__global__ __launch_bounds__(256) void stripe_dequantize_kernel(const FormatArgs a, int lr, int grows, int lc) {
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= (int64_t)a.B * a.HV * (a.V / kStripe)) return;
  const Stripe st = stripe_of(a, item);
  const int half = lane >> 5, c4 = lane & 31;
  const uint8_t* src = (const uint8_t*)a.payload + (int64_t)st.b * a.pl_b + (int64_t)st.hv * a.pl_h + (int64_t)(st.row0 + half) * a.pl_v + 4 * c4;
  float* dst = a.state + (int64_t)st.b * a.st_b + (int64_t)st.hv * a.st_h + (int64_t)(st.row0 + half) * a.st_v + 4 * c4;
  const int64_t so = (int64_t)st.b * a.sc_b + (int64_t)st.hv * a.sc_h + (int64_t)(c4 >> lc) * a.sc_c;
  uint32_t w[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) w[j] = *(const uint32_t*)(src + (int64_t)(2 * j) * a.pl_v);
  float sc[16];
  if (lr == 5) {
    sc[0] = ld_dt(a.scale, so + (int64_t)(st.row0 / grows) * a.sc_r, a.scale_dt);
#pragma unroll
    for (int j = 1; j < 16; ++j) sc[j] = sc[0];
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j)
      sc[j] = ld_dt(a.scale, so + (int64_t)((st.row0 + 2 * j + half) >> lr) * a.sc_r, a.scale_dt);
  }
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    float f[4];
    if constexpr (INT8) {
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = (float)(int8_t)(w[j] >> (8 * e));
    } else {
      fp8x4_to_f32(w[j], f);
    }
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    const f32x4_t y = {f[0] * sc[j], f[1] * sc[j], f[2] * sc[j], f[3] * sc[j]};
    *(f32x4_t*)(dst + (int64_t)(2 * j) * a.st_v) = y;
  }
}

// How a layout splits into stripes: rows per group within a stripe (0: the
// generic kernels), stripes per group, log2 of the lanes per column group.
struct StripePlan {
  int rows, stripes, lc;
};
StripePlan stripe_plan(const FormatArgs& a) {
  const StripePlan none = {0, 0, 0};
  auto mult = [](int64_t x, int m) { return x % m == 0; };
  if (a.K != 128 || a.V % kStripe || (uintptr_t)a.state % 16 || (uintptr_t)a.payload % 4 || !mult(a.st_b, 4) ||
      !mult(a.st_h, 4) || !mult(a.st_v, 4) || !mult(a.pl_b, 4) || !mult(a.pl_h, 4) || !mult(a.pl_v, 4))
    return none;
  const int rows = a.gran == kGranHead ? a.V : a.gran == kGranRow ? 1 : a.tile;
  int lc = 5;
  if (a.gran == kGranTile) {  // (divides K: a power of two)
    if (a.tile < 4) return none;
    for (lc = 0; (4 << lc) < a.tile;) ++lc;
  }
  if (rows <= kStripe) return (rows & (rows - 1)) ? none : StripePlan{rows, 1, lc};
  return rows % kStripe == 0 && rows / kStripe <= kMaxStripes ? StripePlan{kStripe, rows / kStripe, lc} : none;
}

template <int R, bool WAVES, int LC>
void launch_stripe(const FormatArgs& a, int stripes, hipStream_t s) {
  const int64_t items = (int64_t)a.B * a.HV * (a.V / kStripe);
  const dim3 grid((unsigned)(WAVES ? items / stripes : (items + 3) / 4)), block(WAVES ? 64 * stripes : 256);
  if (a.int8) hipLaunchKernelGGL((stripe_quantize_kernel<R, WAVES, LC, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((stripe_quantize_kernel<R, WAVES, LC, false>), grid, block, 0, s, a);
}

// false: no instantiation (the generic kernel takes it)
bool launch_stripe_quantize(const FormatArgs& a, const StripePlan& p, hipStream_t s) {
  if (p.lc == 5) {
    if (p.stripes > 1) return launch_stripe<32, true, 5>(a, p.stripes, s), true;
    switch (p.rows) {
      case 1: return launch_stripe<1, false, 5>(a, 1, s), true;
      case 2: return launch_stripe<2, false, 5>(a, 1, s), true;
      case 4: return launch_stripe<4, false, 5>(a, 1, s), true;
      case 8: return launch_stripe<8, false, 5>(a, 1, s), true;
      case 16: return launch_stripe<16, false, 5>(a, 1, s), true;
      case 32: return launch_stripe<32, false, 5>(a, 1, s), true;
      default: return false;
    }
  }
  switch (p.lc) {  // tiles of 4 .. 64
    case 0: return launch_stripe<4, false, 0>(a, 1, s), true;
    case 1: return launch_stripe<8, false, 1>(a, 1, s), true;
    case 2: return launch_stripe<16, false, 2>(a, 1, s), true;
    case 3: return launch_stripe<32, false, 3>(a, 1, s), true;
    case 4: return launch_stripe<32, true, 4>(a, p.stripes, s), true;
    default: return false;
  }
}

}  // namespace

int launch_format_quantize(const FormatArgs& a, void* stream) {
  const StripePlan plan = stripe_plan(a);
  if (plan.rows && launch_stripe_quantize(a, plan, (hipStream_t)stream)) return (int)hipGetLastError();
  int gph;
  switch (a.gran) {
    case kGranHead: gph = 1; break;
    case kGranRow: gph = a.V; break;
    case kGranTile: gph = (a.V / a.tile) * (a.K / a.tile); break;
    default: gph = a.V / a.tile; break;
  }
  const int64_t groups = (int64_t)a.B * a.HV * gph;
  hipLaunchKernelGGL(format_quantize_kernel, dim3((unsigned)groups), dim3(256), 0, (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

int launch_format_dequantize(const FormatArgs& a, void* stream) {
  const StripePlan plan = stripe_plan(a);
  if (plan.rows) {
    int lr = 0;
    while ((1 << lr) < plan.rows) ++lr;
    const int64_t items = (int64_t)a.B * a.HV * (a.V / kStripe);
    const dim3 grid((unsigned)((items + 3) / 4));
    if (a.int8)
      hipLaunchKernelGGL(stripe_dequantize_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, a, lr, plan.rows * plan.stripes, plan.lc);
    else
      hipLaunchKernelGGL(stripe_dequantize_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, a, lr, plan.rows * plan.stripes, plan.lc);
    return (int)hipGetLastError();
  }
  const int64_t total = (int64_t)a.B * a.HV * a.V * a.K;
  hipLaunchKernelGGL(format_dequantize_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, a);
  return (int)hipGetLastError();
}

}  // namespace gdnr
