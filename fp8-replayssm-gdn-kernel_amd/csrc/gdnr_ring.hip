// gdnr_ring.hip -- the ReplaySSM decode step on gfx950 (MI355X) for rings of
// 17 to 64 tokens with 16-bit activations at any batch: replay or flush per
// sequence, optionally fused with the full-contract preparation of the new
// token.
//
// Workgroup: 4 waves of 32 VB V-rows = GW value heads of one key head and
// sequence (WPH waves a head). No wave streams on its own: all four stage the
// key ring, form the Gram matrix and stream checkpoint rows, and meet at three
// barriers. Three workgroups share a compute unit (40 KiB of LDS, 155 VGPRs:
// held to 128, for four, the flush spills and every launch with one is slower,
// B=64, L=64 20.3 to 31.6 us against 21.7), so one's serial part (the
// coefficient chain) overlaps the others' streams.
//
// Bound: a replay at full batch by its bytes and its VALU issue (B=64, L=64,
// fill 32: 60 MB in 19.0 us, 3.2 TB/s, against 25.8 for the per-token chain of
// gdnr_kernels.hip that this kernel replaces; fill 63 23.9 against 36.9); a
// flush by its waves' own latency (6 us to the factors, then 3.7 us a tile: a
// launch of 24 flushes 26 us against 193). A step of B=64, L=64 with staggered
// fills (one sequence flushing) takes 18.6 us against 134. Short fills gain
// nothing, and where many rounds of small workgroups repeat the staging (V=64
// or an odd group) they lose: B=200, L=17 at fill 8, 16 heads of V=64 17.1
// against 14.1.
//
// Replay (the adjoint of the reference's reverse chain,
// prototype/gdn_replayssm_fp8_kernel.py:121-173, in Gram form over the whole
// ring): G = K K^T by MFMA, s_t = beta_t (k_t . q - sum_{u>t} G_tu s_u),
// c_t = s_t prod_{u>t} gamma_u, T_0 = lam (q - sum_t s_t k_t),
// o = (scale codes T_0 + sum_t c_t v_t) K^-1/2, T_0 as three bf16 rows (24
// bits) against the codes in bf16 (exact).
//
// Flush (the forward rebuild of kernel:177-242 over 16-token chunks):
//   Q_c = X_c S_c^T = lam_{<c} X_c S_0^T + sum_{c'<c} G_cc' U~_c'
// (S_c the state before chunk c; X_c S_0^T an exact-operand MFMA on the
// codes; the cross-chunk products f32 MFMAs on G, so the state itself is
// formed only once), W = V - pre Q, U = (I + M_c)^-1 W, U~ = post U, every
// earlier U~ decayed by lam_c; then S_n = lam S_0 + sum_c K_c^T U~_c with U~
// in three bf16 parts (24 bits), o from the same factors, and the reference
// quantiser in place (ref:36-37,83-99).
//
// Operand layouts are those of gdnr_decode.hip (lane = 16 q4 + l16): X rows
// in LDS in row form, tile i of a wave = rows 32 (i >> 1) + 2 nn + (i & 1).
// The K^T operands of the flush's last product come from the X rows by
// transposing LDS reads (ds_read_b64_tr_b16), in U~'s own token order.
//
// Compiled once per 16-bit activation dtype (GDNR_ACT = 0 bf16, 1 f16).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#ifndef GDNR_ACT
#error "compile with -DGDNR_ACT=0|1|2"
#endif

#if GDNR_ACT != 2
#include "gdnr_act16.h"

namespace gdnr {
namespace {

constexpr int NW = 4;                  // waves per workgroup
constexpr int NC = kMaxRing / NT;      // 16-token chunks of the longest ring
constexpr int kXS = 272;               // X row stride (256 + 16: the rows' banks differ)
constexpr int kGS = 20;                // floats per row of a 16 x 16 Gram tile

// LDS (bytes). Tile (r, c), r <= c, of the Gram matrix is tile c (c + 1) / 2 + r.
constexpr int kLdsX = 0;                                 // X rows [64][kXS]
constexpr int kLdsG = kLdsX + kMaxRing * kXS;            // Gram tiles f32 [10][16][kGS]
constexpr int kLdsQ = kLdsG + NC * (NC + 1) / 2 * 16 * kGS * 4;  // the query row, act [128]
constexpr int kLdsDq = kLdsQ + 256;                      // k_t . q f32 [64]
constexpr int kLdsZ = kLdsDq + 256;                      // replay or flush blocks:
// replay: per head T_0 as hi, mid, lo rows bf16 [3][128]; per head c_t f32
// [64]; per wave the sums of c_t v_t f32 [32 VB]
constexpr int kT0Bytes = 768, kCoefBytes = 256;
// flush: per head R_c = (I + M_c)^-1 f32 [4][16][16] (M_c while it is
// formed); per head (pre, post) f32 [64][2]; per head lam_c f32 [4], the decay after
// chunk c f32 [4] and lam f32; the
// tiles' amax f32 [2][4]
constexpr int kRBytes = NC * 1024, kFacBytes = kMaxRing * 8, kLamBytes = 48;

constexpr int ring_lds(int gw, int vb) {
  const int replay = gw * (kT0Bytes + kCoefBytes) + NW * 32 * vb * 4, flush = gw * (kRBytes + kFacBytes + kLamBytes) + 2 * NW * 4;
  return kLdsZ + (replay > flush ? replay : flush);
}
static_assert(ring_lds(2, 2) <= 40 * 1024, "a compute unit holds four workgroups' LDS (and three's registers)");

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

extern __shared__ __attribute__((aligned(16))) uint8_t ring_smem[];

// x in three bf16 parts (24 bits), pairs packed
struct Split3 {
  uint32_t hi, mid, lo;
};
__device__ __forceinline__ Split3 split3(float x, float y) {
  Split3 s;
  s.hi = pack_bf16x2(x, y);
  const float rx = x - __uint_as_float(s.hi << 16), ry = y - __uint_as_float(s.hi & 0xFFFF0000u);
  s.mid = pack_bf16x2(rx, ry);
  s.lo = pack_bf16x2(rx - __uint_as_float(s.mid << 16), ry - __uint_as_float(s.mid & 0xFFFF0000u));
  return s;
}
// the same in the activation type (f16: 33 bits of a value scaled to 2^13)
__device__ __forceinline__ Split3 split3_act(float x, float y) {
  if constexpr (kBF16) return split3(x, y);
  Split3 s;
  auto part = [](float& u, float& v) {
    const uint32_t w = act_bits(u) | (act_bits(v) << 16);
    const float2 f = Act::from_pair(w);
    u -= f.x, v -= f.y;
    return w;
  };
  s.hi = part(x, y);
  s.mid = part(x, y);
  s.lo = part(x, y);
  return s;
}
// 4 tokens (rows t0 .. t0 + 3 of X) of the lane's column in the K^T operand of
// column group ct: lane l16 of each 16-lane row reads 8 bytes of row
// t0 + l16 / 4 at columns 32 (l16 & 3) + 4 ct, and gets column
// 32 (l16 >> 2) + 4 ct + (l16 & 3) of the four rows
__device__ __forceinline__ uint2 kt_read(int off) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(ring_smem + off)));
}
// double-precision decays of a flush: DPP moves and products over a 16-lane row
template <int CTRL>
__device__ __forceinline__ double dpp_row64(double x, double fill) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x), f = __builtin_bit_cast(uint64_t, fill);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)f, (int)(uint32_t)b, CTRL, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(f >> 32), (int)(b >> 32), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
// every lane of each 16-lane row gets lane n of its row
__device__ __forceinline__ double row_bcast64(double x, int n) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __float_as_uint(row_bcast_n(__uint_as_float((uint32_t)b), n));
  const uint32_t hi = __float_as_uint(row_bcast_n(__uint_as_float((uint32_t)(b >> 32)), n));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double rdl64(double x, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ void lds_barrier() {
  GDNR_WAIT_LGKM0();
  __builtin_amdgcn_s_barrier();
  GDNR_COMPILER_FENCE();
}
__device__ __forceinline__ constexpr int gram_tile(int r, int c) { return kLdsG + (c * (c + 1) / 2 + r) * 16 * kGS * 4; }

template <int VB, int WPH, bool FUSED, bool GATE_F32, bool SLOTS>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(3))) void ring_kernel(
    const uint8_t* m_len, const uint8_t* m_pos, const uint8_t* m_flush, uint32_t m_vs, uint32_t m_ps, uint32_t m_fs,
    int32_t m_L, int32_t m_grp, int32_t m_order, int32_t m_G, const StepArgs a) {
  constexpr int ES = 2;
  constexpr int GW = NW / WPH;            // value heads per workgroup
  constexpr int RPW = 32 * VB;            // V-rows per wave
  constexpr int TPW = 2 * VB;             // 16-row tiles per wave
  uint8_t* const lds = ring_smem;
  const int lane = threadIdx.x & 63;
  const int q4 = lane >> 4, l16 = lane & 15;
  const int w = uni(threadIdx.x >> 6);
  const int n_grp = m_grp;              // head groups per key head
  const int r = blockIdx.x;
  const int h = uni(r / n_grp), grp = r - h * n_grp;
  const int j = w / WPH, part = w % WPH;  // value head in the workgroup, row block of it
  const int hv = h * m_G + grp * GW + j;
  const int R0 = RPW * part;

  // ---- the sequence and its metadata: how much of the ring to read is known
  // before any of it is requested. (These arguments are preloaded into SGPRs
  // at wave launch.) A launch that may hold flushes and takes more than one
  // round of workgroups (m_order: 1 + the grid's rows past the batch) takes
  // the flushing sequences first, and a few of them with two workgroups each:
  // a flush runs longer than a replay, and one that starts in the last round
  // ends the launch late. B=64, L=64, one flush a step: 24.5 us in the batch's
  // order, 22.0 flushes first, 18.6 in halves too (replays alone, at fill 32,
  // 18.5 in the batch's order and 19.0 with the order looked for). The
  // blockIdx.y-th sequence of that order is found from every sequence's flag;
  // its lane holds its metadata too.
  int b = blockIdx.y, bs = b, n, pos = -1;
  bool do_flush = false, split = false, spare = false;
  int half = 0;
  if (m_order) {
    constexpr int NO = kRingOrder / 64;
    uint32_t f[NO];
    int vl[NO], ps[NO], sl[NO];
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      if (64 * i >= a.B) break;
      const uint32_t bq = (uint32_t)min(64 * i + lane, a.B - 1);
      f[i] = m_flush[bq * m_fs];
      vl[i] = *(const int*)(m_len + bq * m_vs);
      if constexpr (FUSED) ps[i] = *(const int*)(m_pos + bq * m_ps);
      if constexpr (SLOTS) sl[i] = *(const int*)(a.slot + bq * a.sl_s);
    }
    uint64_t fm[NO], zm[NO];  // flushing and other sequences
    int nf = 0;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      if (64 * i >= a.B) break;
      const uint64_t valid = __ballot(64 * i + lane < a.B);
      fm[i] = __ballot(f[i] != 0) & valid;
      zm[i] = ~fm[i] & valid;
      nf += __popcll(fm[i]);
    }
    // a few flushing sequences (as many as the grid has rows past the batch)
    // get two workgroups each, for half of the vblocks (the rows then left
    // over are spare: they take the last sequence's requests and end)
    const int twice = nf < m_order ? nf : 0, y = blockIdx.y;
    split = uni(y < 2 * twice) != 0;
    half = uni(split ? y & 1 : 0);
    int want = split ? y >> 1 : y - twice;
    spare = uni(want >= a.B) != 0;
    want = min(want, a.B - 1);
    half = spare ? 1 : half;
    int at_f = 0, at_z = nf;
#pragma unroll
    for (int i = 0; i < NO; ++i) {
      if (64 * i >= a.B) break;
      const uint64_t below = (1ull << lane) - 1;
      const bool is_f = (fm[i] >> lane) & 1, is_z = (zm[i] >> lane) & 1;
      const int rank = is_f ? at_f + __popcll(fm[i] & below) : at_z + __popcll(zm[i] & below);
      const uint64_t hit = __ballot((is_f || is_z) && rank == want);
      if (hit) {
        const int l = __builtin_ctzll(hit);
        b = 64 * i + l;
        do_flush = (fm[i] >> l) & 1;
        n = __builtin_amdgcn_readlane(vl[i], l);
        if constexpr (FUSED) pos = __builtin_amdgcn_readlane(ps[i], l);
        if constexpr (SLOTS) bs = __builtin_amdgcn_readlane(sl[i], l);
      }
      at_f += __popcll(fm[i]);
      at_z += __popcll(zm[i]);
    }
    b = uni(b);
    if constexpr (!SLOTS) bs = b;
  } else {
    n = (int)ld_u32_uniform(m_len + b * m_vs);
    if constexpr (FUSED) pos = (int)ld_u32_uniform(m_pos + b * m_ps);
    if constexpr (SLOTS) bs = (int)ld_u32_uniform(a.slot + b * a.sl_s);
    if (m_flush) {
      const uintptr_t fa = (uintptr_t)(m_flush + b * m_fs);
      const uint32_t word = ld_u32_uniform((const void*)(fa & ~(uintptr_t)3));
      do_flush = ((word >> (8u * (uint32_t)(fa & 3))) & 0xFFu) != 0;
    }
  }
  do_flush = uni(do_flush) != 0;
  n = min(max(uni(n), 0), m_L);
  pos = uni(pos);
  if (pos < 0 || pos >= m_L) pos = -1;
  bs = uni(bs);
  if constexpr (SLOTS)
    if (bs < 0 || bs >= a.n_slots) bs = 0;

  // ---- requests: the wave's 16 key rows in the X operand layout, the query
  // (and new key) row, the gates by token, then the codes
  const int tw = NT * w + l16;            // the key row this lane stages
  u32x4_t kx[4];
  {
    const uint8_t* krow = sbase(a.k, bs, a.k_b) + (h * a.k_h + (uint32_t)(tw < n ? tw : 0) * a.k_t) + 64 * q4;
#pragma unroll
    for (int m = 0; m < 4; ++m) kx[m] = ld16(krow + 16 * m);
  }
  uint32_t qbits, kbits = 0, ab0 = 0, ab1 = 0;
  float alog = 0.f, dtb = 0.f;
  if constexpr (FUSED) {
    const uint8_t* row = a.mixed + b * a.mx_b;
    qbits = ld32(row + (h * K + 2 * lane) * ES);
    kbits = ld32(row + (a.H * K + h * K + 2 * lane) * ES);
    ab0 = gate_bits<GATE_F32>(a.a + (b * a.a_b + hv * a.a_h));
    ab1 = gate_bits<GATE_F32>(a.bgate + (b * a.bg_b + hv * a.bg_h));
    alog = *(const float*)(a.a_log + hv * a.al_s);
    dtb = *(const float*)(a.dt_bias + hv * a.db_s);
  } else {
    qbits = ld32(a.q + (b * a.q_b + h * a.q_h) + 4 * lane);
  }
  const uint32_t tg = lane < n ? lane : 0;  // lane t: token t's gates
  const uint32_t g_raw = *(const uint16_t*)(sbase(a.g, bs, a.g_b) + (tg * a.g_t + hv * a.g_h));
  const uint32_t be_raw = *(const uint16_t*)(sbase(a.beta, bs, a.be_b) + (tg * a.be_t + hv * a.be_h));
  GDNR_COMPILER_FENCE();

  uint8_t* const v_rows = sbase(a.v, bs, a.v_b) + (hv * a.v_h + R0 * ES);
  const uint8_t* const v_new = FUSED ? a.mixed + (b * a.mx_b + (2 * a.H * K + hv * a.V + R0) * ES) : nullptr;
  uint8_t* const out_rows = a.out + (b * a.o_b + hv * a.o_h + R0 * ES);

  // ---- X rows: tokens at or past the fill are zero, to the end of the fill's
  // chunk, or of the chunks a flush takes (2 or 4: its loops are compiled for
  // either, with no branch at each chunk); the new token's row and the query
  // row are wave 0's (normalised as the preparation does, rounded to the ring
  // dtype)
  const int nx = do_flush ? (n <= 2 * NT ? 2 * NT : NC * NT) : n;
  auto stage_x = [&]() {
    if (NT * w < nx) {
      const bool keep = tw < n;
      if (!FUSED || !keep || tw != pos) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
          *(u32x4_t*)(lds + kLdsX + tw * kXS + 64 * q4 + 16 * m) = keep ? kx[m] : u32x4_t{0u, 0u, 0u, 0u};
      }
    }
    if (w == 0) {
      uint32_t qw = qbits;
      if constexpr (FUSED) {
        const float2 qr = Act::from_pair(qbits), kr = Act::from_pair(kbits);
        const float qd = sqrtf(wave_sum(fmaf(qr.y, qr.y, qr.x * qr.x)) + 1e-6f);
        const float kd = sqrtf(wave_sum(fmaf(kr.y, kr.y, kr.x * kr.x)) + 1e-6f);
        qw = act_bits(Act::round(qr.x / qd)) | (act_bits(Act::round(qr.y / qd)) << 16);
        const uint32_t kw = act_bits(Act::round(kr.x / kd)) | (act_bits(Act::round(kr.y / kd)) << 16);
        if (pos >= 0 && pos < n) *(uint32_t*)(lds + kLdsX + pos * kXS + 4 * lane) = kw;
        if (grp == 0 && half == 0) {
          *(uint32_t*)(a.q_out + (b * a.qo_b + h * a.qo_h) + 4 * lane) = qw;
          if (pos >= 0) *(uint32_t*)(sbase(a.k, bs, a.k_b) + ((uint32_t)pos * a.k_t + h * a.k_h) + 4 * lane) = kw;
        }
      }
      *(uint32_t*)(lds + kLdsQ + 4 * lane) = qw;
    }
  };
  auto x_op = [&](int c, int m) { return *(const u32x4_t*)(lds + kLdsX + (NT * c + l16) * kXS + 64 * q4 + 16 * m); };
  auto q_op = [&](int m) { return *(const u32x4_t*)(lds + kLdsQ + 64 * q4 + 16 * m); };
  // Gram tiles (r <= c) and k_t . q, dealt over the waves. Replay: row = token
  // of chunk r, column = token of chunk c (the later one), the diagonal tiles
  // strictly upper. Flush: row = token of chunk c, column = token of chunk r.
  auto gram = [&](auto flush) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
      for (int rr = 0; rr <= c; ++rr) {
        if (((c * (c + 1) / 2 + rr) & (NW - 1)) != w || NT * c >= nx) continue;
        f32x4_t g = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < 4; ++m)
          g = decltype(flush)::value ? mfma16(x_op(rr, m), x_op(c, m), g) : mfma16(x_op(c, m), x_op(rr, m), g);
        if (!decltype(flush)::value && rr == c) {
#pragma unroll
          for (int e = 0; e < 4; ++e) g[e] = 4 * q4 + e > l16 ? g[e] : 0.f;
        }
        *(f32x4_t*)(lds + gram_tile(rr, c) + 4 * (l16 * kGS + 4 * q4)) = g;
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (((NC * (NC + 1) / 2 + c) & (NW - 1)) != w || NT * c >= nx) continue;
      f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < 4; ++m) d = mfma16(x_op(c, m), l16 == 0 ? q_op(m) : u32x4_t{0u, 0u, 0u, 0u}, d);
      if (l16 == 0) *(f32x4_t*)(lds + kLdsDq + 4 * (NT * c + 4 * q4)) = d;
    }
  };
  // lane t: the log decay g and beta (0 at or past the fill) of token t, the new
  // token's from the preparation formulas (kernel:534-562) and appended
  const bool on = lane < n;
  auto gates = [&](float& gg, float& bet) {
    gg = act_val(g_raw);
    float bb = act_val(be_raw);
    if constexpr (FUSED) {
      const float x = gate_value<GATE_F32>(ab0) + dtb;
      const float sp = x <= 20.0f ? logf(1.0f + expf(x)) : x;  // kernel:560, as written there
      const float gate_new = Act::round(-expf(alog) * sp);
      const float beta_new = Act::round(1.0f / (1.0f + expf(-gate_value<GATE_F32>(ab1))));
      if (pos >= 0 && lane == 0 && half == 0) {
        *(uint16_t*)(sbase(a.g, bs, a.g_b) + ((uint32_t)pos * a.g_t + hv * a.g_h)) = (uint16_t)act_bits(gate_new);
        *(uint16_t*)(sbase(a.beta, bs, a.be_b) + ((uint32_t)pos * a.be_t + hv * a.be_h)) = (uint16_t)act_bits(beta_new);
      }
      gg = lane == pos ? gate_new : gg;
      bb = lane == pos ? beta_new : bb;
    }
    bet = on ? bb : 0.f;
  };
  constexpr int CPT = RPW * ES / 16;      // 16-byte pieces of a token's v rows of the wave
  constexpr int TPL = 64 / CPT;           // tokens per load
  constexpr int NVL = kMaxRing / TPL;     // loads per lane

  if (spare) return;  // (here, not where it is found: the arguments' scalar loads would sink past it)
  if (!do_flush) {
    // ================= replay =====================================================
    u32x4_t cw[TPW][2];
    {
      // (non-temporal: read once a step)
      const uint8_t* ck_rows = sbase(a.ckpt, bs, a.ck_b) + (hv * a.ck_h + R0 * a.ck_v);
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const uint8_t* row = ck_rows + (uint32_t)(32 * (i >> 1) + 2 * l16 + (i & 1)) * a.ck_v + 32 * q4;
        cw[i][0] = __builtin_nontemporal_load((g_u32x4*)row);
        cw[i][1] = __builtin_nontemporal_load((g_u32x4*)(row + 16));
      }
    }
    GDNR_COMPILER_FENCE();
    stage_x();
    // v rows, in 16-byte pieces: load k of lane l is token k TPL + l / CPT,
    // piece l % CPT (slots at or past the fill re-read slot 0); the new
    // token's piece from mixed_qkv
    u32x4_t vq[NVL], vnew;
    const int vp = lane % CPT, vt = lane / CPT;
#pragma unroll
    for (int k = 0; k < NVL; ++k) {
      const int t = k * TPL + vt;
      vq[k] = *(g_u32x4*)(v_rows + ((uint32_t)(t < n ? t : 0) * a.v_t + 16 * vp));
    }
    if constexpr (FUSED) vnew = *(g_u32x4*)(v_new + 16 * vp);
    const uint8_t* sc_rows = sbase(a.scale, bs, a.sc_b) + (hv * a.sc_h + (R0 / kVBlock) * a.sc_v);
    float sct[VB];
#pragma unroll
    for (int p = 0; p < VB; ++p) sct[p] = f16_bits_to_f32(ld_u16_uniform(sc_rows + p * a.sc_v));
    lds_barrier();
    gram(std::false_type{});
    lds_barrier();
    if (part == 0) {
      // the head's coefficient chain (lane t: token t), as the chunked chain
      // of gdnr_decode.hip runs it
      float gg, bet;
      gates(gg, bet);
      const float gam = on ? expf(gg) : 1.f;
      const float suf_in = row_suffix_prod(gam);
      const float suf_ex = dpp_row<0x101>(suf_in, 1.f);
      const float lamc = row_bcast<0>(suf_in);
      const float bd = on ? bet * *(const float*)(lds + kLdsDq + 4 * lane) : 0.f;
      float acc = 0.f, ax = 0.f, ay = 0.f, s_mine = 0.f;
#pragma unroll
      for (int c = NC - 1; c >= 0; --c) {
        if (NT * c >= n) continue;
        float gb[NT];
        // (lanes of chunks past c are done; they read tile (c, c))
        const int rr = q4 < c ? q4 : c;
        const uint8_t* gr = lds + gram_tile(rr, c) + 4 * l16 * kGS;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 g4 = *(const float4*)(gr + 16 * i);
          gb[4 * i] = g4.x, gb[4 * i + 1] = g4.y, gb[4 * i + 2] = g4.z, gb[4 * i + 3] = g4.w;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(gb[t]));
#pragma unroll
        for (int hf = 1; hf >= 0; --hf) {
          // (8 key words at a time, behind one wait)
          uint32_t xw[NT / 2];
#pragma unroll
          for (int t = 0; t < NT / 2; ++t)
            xw[t] = *(const uint32_t*)(lds + kLdsX + (NT * c + NT / 2 * hf + t) * kXS + 4 * lane);
#pragma unroll
          for (int t = 0; t < NT / 2; ++t) asm volatile("" : "+v"(xw[t]));
#pragma unroll
          for (int t = NT / 2 - 1; t >= 0; --t) {
            const float st = rdl(fmaf(-bet, acc, bd), NT * c + NT / 2 * hf + t);
            acc = fmaf(gb[NT / 2 * hf + t], st, acc);
            const float2 xv = Act::from_pair(xw[t]);
            ax = fmaf(st, xv.x, ax);
            ay = fmaf(st, xv.y, ay);
          }
        }
        s_mine = q4 == c ? fmaf(-bet, acc, bd) : s_mine;
      }
      const float l1 = rdl(lamc, NT), l2 = rdl(lamc, 2 * NT), l3 = rdl(lamc, 3 * NT);
      const float later = (q4 < 1 ? l1 : 1.f) * (q4 < 2 ? l2 : 1.f) * (q4 < 3 ? l3 : 1.f);
      const float lam_all = rdl(lamc, 0) * l1 * l2 * l3;
      *(float*)(lds + kLdsZ + GW * kT0Bytes + j * kCoefBytes + 4 * lane) = on ? s_mine * (suf_ex * later) : 0.f;
      const float2 qv = Act::from_pair(*(const uint32_t*)(lds + kLdsQ + 4 * lane));
      Split3 t0 = split3(lam_all * (qv.x - ax), lam_all * (qv.y - ay));
      if (n == 0) {
        // (an infinite query entry of an empty ring stays one: its lower parts
        // are inf - inf)
        if (__builtin_fabsf(qv.x) == __builtin_inff()) t0.mid &= 0xFFFF0000u, t0.lo &= 0xFFFF0000u;
        if (__builtin_fabsf(qv.y) == __builtin_inff()) t0.mid &= 0xFFFFu, t0.lo &= 0xFFFFu;
      }
      uint8_t* tr = lds + kLdsZ + j * kT0Bytes + 4 * lane;
      *(uint32_t*)tr = t0.hi;
      *(uint32_t*)(tr + 256) = t0.mid;
      *(uint32_t*)(tr + 512) = t0.lo;
    }
    // the new token's v rows, appended and taken in place of the ring's
    if constexpr (FUSED) {
      if (pos >= 0 && vt == pos % TPL) *(u32x4_t*)(v_rows + ((uint32_t)pos * a.v_t + 16 * vp)) = vnew;
#pragma unroll
      for (int k = 0; k < NVL; ++k)
        if (k * TPL + vt == pos) vq[k] = vnew;
    }
    lds_barrier();
    // ---- sum_t c_t v_t: 8 rows a lane over its tokens, then over the lanes
    // that share a piece; row 8 vp + e in LDS
    float* const vs = (float*)(lds + kLdsZ + GW * (kT0Bytes + kCoefBytes)) + w * RPW;
    {
      float sv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) sv[e] = 0.f;
#pragma unroll
      for (int k = 0; k < NVL; ++k) {
        if (k * TPL >= n) break;
        const int t = k * TPL + vt;
        const float ct = *(const float*)(lds + kLdsZ + GW * kT0Bytes + j * kCoefBytes + 4 * t);
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2) {
          const float2 v2 = Act::from_pair(t < n ? vq[k][e2] : 0u);
          sv[2 * e2] = fmaf(ct, v2.x, sv[2 * e2]);
          sv[2 * e2 + 1] = fmaf(ct, v2.y, sv[2 * e2 + 1]);
        }
      }
      // reduce-scatter over lane bits 5, 4 and 3 (and a sum over bit 2 where
      // 16 lanes share a piece)
      float s4[4], s2[2];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(sv[e]), __float_as_uint(sv[e + 4]), false, false);
        s4[e] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(s4[e]), __float_as_uint(s4[e + 2]), false, false);
        s2[e] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
      }
      const bool b3 = (lane & 8) != 0;
      float s1 = (b3 ? s2[1] : s2[0]) + dpp_row<0x128>(b3 ? s2[0] : s2[1], 0.f);  // (row_ror:8 = lane ^ 8)
      if constexpr (CPT == 4)
        s1 += __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, s1), 0x101F));  // lane ^ 4
      const int e = ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + (b3 ? 1 : 0);
      if (CPT == 8 || (lane & 4) == 0) vs[8 * vp + e] = s1;
    }
    // ---- S_0 T_0 by MFMA (A rows 0..2: hi, mid, lo), tile by tile
    const uint8_t* trow = lds + kLdsZ + j * kT0Bytes + 256 * (l16 < 3 ? l16 : 0) + 64 * q4;
    u32x4_t ta[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const u32x4_t x = *(const u32x4_t*)(trow + 16 * m);
      ta[m] = l16 < 3 ? x : u32x4_t{0u, 0u, 0u, 0u};
    }
    GDNR_WAIT_LGKM0();
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const u32x4_t cwm = cw[i][m >> 1];
        const uint2 lo = fp8x4_to_bf16x4((m & 1) ? cwm[2] : cwm[0]), hi = fp8x4_to_bf16x4((m & 1) ? cwm[3] : cwm[1]);
        c = mfma_bf16(ta[m], u32x4_t{lo.x, lo.y, hi.x, hi.y}, c);
      }
      if (q4 == 0) {
        const int row = 32 * (i >> 1) + 2 * l16 + (i & 1);
        Act::st(out_rows, row, fmaf(c[0] + (c[1] + c[2]), sct[i >> 1], vs[row]) * a.out_scale);
      }
    }
    return;
  }

  // ================= flush ========================================================
  // Two waves share a vblock, one 16-row tile each (the state of one tile is
  // 32 VGPRs): waves 2 x and 2 x + 1 take the vblocks of their rows in turn,
  // wave w rows [16 (w & 1), +16) of each
  constexpr int FV = 2 * VB;              // vblocks of a wave pair
  const int P0 = RPW * (part & ~1);       // the pair's first row in the head
  const int f0 = P0 + 16 * (w & 1);       // the wave's first row in the head
  uint8_t* const fc_rows = sbase(a.ckpt, bs, a.ck_b) + (hv * a.ck_h + f0 * a.ck_v);
  uint8_t* const fs_rows = sbase(a.scale, bs, a.sc_b) + (hv * a.sc_h + (P0 / kVBlock) * a.sc_v);
  const uint8_t* const f_rows = sbase(a.v, bs, a.v_b) + (hv * a.v_h + f0 * ES);
  const uint8_t* const f_new = FUSED ? a.mixed + (b * a.mx_b + (2 * a.H * K + hv * a.V + f0) * ES) : nullptr;
  uint8_t* const fo_rows = a.out + (b * a.o_b + hv * a.o_h + f0 * ES);
  u32x4_t cw[2];
  uint32_t vw[NC][2], vwn = 0;            // v of tokens 16 c + 4 q4 + e, in pairs, and of the new token
  auto load_codes = [&](int p) {
    const uint8_t* row = fc_rows + (uint32_t)(32 * p + l16) * a.ck_v + 32 * q4;
    cw[0] = __builtin_nontemporal_load((g_u32x4*)row);
    cw[1] = __builtin_nontemporal_load((g_u32x4*)(row + 16));
  };
  auto load_v = [&](int p) {
    const uint8_t* const vb = f_rows + 32 * p * ES;
    // (one lane offset; the token offsets scalar, past the ring's end the
    // last slot's)
    const uint32_t vo = 4 * q4 * a.v_t + ES * l16;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const bool whole = NT * (c + 1) <= a.L;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        auto v1 = [&](int d) {
          if (whole) return *(const uint16_t*)(vb + (uint32_t)(NT * c + d) * a.v_t + vo);
          return *(const uint16_t*)(vb + ((uint32_t)min(NT * c + 4 * q4 + d, a.L - 1) * a.v_t + ES * l16));
        };
        const u16x2_t v2 = {v1(2 * e), v1(2 * e + 1)};
        vw[c][e] = __builtin_bit_cast(uint32_t, v2);
      }
    }
    if constexpr (FUSED) vwn = *(const uint16_t*)(f_new + (32 * p + l16) * ES);
  };
  // (the pair's v rows, one cache line a token and wave: they are read again,
  // tile by tile, from the cache)
  const uint32_t warm = ld32(v_rows + (uint32_t)(lane < n ? lane : 0) * a.v_t);
  const int p0 = split ? half * (FV / 2) : 0, p1 = split ? p0 + FV / 2 : FV;  // the workgroup's vblocks
  load_codes(p0);
  GDNR_COMPILER_FENCE();
  stage_x();
  asm volatile("" ::"v"(warm));
  lds_barrier();
  gram(std::true_type{});
  lds_barrier();
  uint8_t* const rl = lds + kLdsZ + j * kRBytes;
  uint8_t* const fl = lds + kLdsZ + GW * kRBytes + j * kFacBytes;
  float* const ll = (float*)(lds + kLdsZ + GW * (kRBytes + kFacBytes) + j * kLamBytes);
  if (part == 0) {
    // the head's flush factors, chunk q4 in row q4 of the wave: pre_t =
    // prod_{x<=t} gamma_x, post_t = beta_t prod_{x>t} gamma_x, lam_c,
    // M[t][s] = beta_s prod_{s<x<=t} gamma_x G[s][t] (s < t) and
    // R = (I + M)^-1 by forward substitution, lane = column
    // (the decays in double: f32 products of up to 64 gammas cost a quarter of
    // the rounding that shows in the codes, 5.3e-6 of them against 3.9e-6 a
    // rounding off the exact state's; 1 us of a 25 us launch of 24 flushes)
    float gg, bet;
    gates(gg, bet);
    const double gam = on ? exp((double)gg) : 1.0;
    double pre = gam, suf_in = gam;
    pre *= dpp_row64<0x111>(pre, 1.0), suf_in *= dpp_row64<0x101>(suf_in, 1.0);
    pre *= dpp_row64<0x112>(pre, 1.0), suf_in *= dpp_row64<0x102>(suf_in, 1.0);
    pre *= dpp_row64<0x114>(pre, 1.0), suf_in *= dpp_row64<0x104>(suf_in, 1.0);
    pre *= dpp_row64<0x118>(pre, 1.0), suf_in *= dpp_row64<0x108>(suf_in, 1.0);
    const double suf_ex = dpp_row64<0x101>(suf_in, 1.0);
    *(float2*)(fl + 8 * lane) = make_float2((float)pre, (float)((double)bet * suf_ex));
    // lam_c, and the decay from chunk c's end to the ring's (lane 16 c); [8]: lam
    const double l1 = rdl64(suf_in, NT), l2 = rdl64(suf_in, 2 * NT), l3 = rdl64(suf_in, 3 * NT);
    const double after = q4 == 0 ? l1 * l2 * l3 : q4 == 1 ? l2 * l3 : q4 == 2 ? l3 : 1.0;
    if (l16 == 0) {
      ll[q4] = (float)suf_in;
      ll[4 + q4] = (float)after;
      if (q4 == 0) ll[8] = (float)(suf_in * after);
    }
    const int nc = min(max(n - NT * q4, 0), NT);
    float gcol[NT];
    {
      const uint8_t* gr = lds + gram_tile(q4, q4) + 4 * l16 * kGS;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float4 g4 = *(const float4*)(gr + 16 * i);
        gcol[4 * i] = g4.x, gcol[4 * i + 1] = g4.y, gcol[4 * i + 2] = g4.z, gcol[4 * i + 3] = g4.w;
      }
    }
    float* Mm = (float*)rl + q4 * 256;
    {
      double run = bet;
#pragma unroll
      for (int t = 1; t < NT; ++t) {
        const double gt = row_bcast64(gam, t);  // (in every lane: the moves read the whole row)
        run = t > l16 ? run * gt : run;
        Mm[t * NT + l16] = (l16 < t && t < nc) ? (float)(run * (double)gcol[t]) : 0.f;
      }
    }
    float rc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float x = (t == l16) ? 1.f : 0.f;
#pragma unroll
      for (int s4 = 0; s4 < t; s4 += 4) {
        const float4 m4 = *(const float4*)(Mm + t * NT + s4);
        x = fmaf(-m4.x, rc[s4], x);
        if (s4 + 1 < t) x = fmaf(-m4.y, rc[s4 + 1], x);
        if (s4 + 2 < t) x = fmaf(-m4.z, rc[s4 + 2], x);
        if (s4 + 3 < t) x = fmaf(-m4.w, rc[s4 + 3], x);
      }
      rc[t] = x;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) Mm[t * NT + l16] = rc[t];
  }
  lds_barrier();

  // ---- the pair's vblocks: rebuilt, emitted and requantised in place
  float* const red = (float*)(lds + kLdsZ + GW * (kRBytes + kFacBytes + kLamBytes));
  auto rebuild = [&](auto chunks) {
    constexpr int NF = decltype(chunks)::value;  // chunks (past the fill: zero keys, zero U~)
    float sct[FV];
#pragma unroll
    for (int p = 0; p < FV; ++p) sct[p] = f16_bits_to_f32(ld_u16_uniform(fs_rows + p * a.sc_v));
#pragma unroll 1
    for (int p = p0; p < p1; ++p) {
      float scp = sct[0];
#pragma unroll
      for (int k = 1; k < FV; ++k) scp = p == k ? sct[k] : scp;
      load_v(p);
      // q[c] = X_c S^T, from S_0: on the codes, and on the query as a block of
      // its own
      f32x4_t q[NF], pq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NF; ++c) q[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const u32x4_t bv = codes8(cw, m);
        pq = mfma16(q_op(m), bv, pq);
#pragma unroll
        for (int c = 0; c < NF; ++c) q[c] = mfma16(x_op(c, m), bv, q[c]);
        if (m & 1) GDNR_COMPILER_FENCE();
      }
      int t0 = 4 * q4;
      asm volatile("" : "+v"(t0));            // (the 16 tokens are compared as they come up)
      float o = q4 == 0 ? scp * pq[0] : 0.f;  // (S_0 q at every q4: counted once)
#pragma unroll
      for (int c = 0; c < NF; ++c) q[c] *= scp;
      // chunk by chunk: U~_c from q[c], then q of every later chunk taken to
      // the state after chunk c (two accumulators where the next step waits)
#pragma unroll
      for (int c = 0; c < NF; ++c) {
        const f32x4_t f01 = *(const f32x4_t*)(fl + 8 * (NT * c + 4 * q4));
        const f32x4_t f23 = *(const f32x4_t*)(fl + 8 * (NT * c + 4 * q4) + 16);
        const float pre[4] = {f01[0], f01[2], f23[0], f23[2]}, post[4] = {f01[1], f01[3], f23[1], f23[3]};
        const f32x4_t rr = *(const f32x4_t*)(rl + 1024 * c + 4 * (l16 * NT + 4 * q4));
        const f32x4_t dq = *(const f32x4_t*)(lds + kLdsDq + 4 * (NT * c + 4 * q4));
        const float lc = ll[c];
        float we[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          we[e] = fmaf(-pre[e], q[c][e], act_val(e & 1 ? vw[c][e >> 1] >> 16 : vw[c][e >> 1]));
        if ((FUSED && c == pos / NT) || NT * (c + 1) > n) {  // (the new token's chunk, the fill's end)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int t = t0 + NT * c + e;
            if (FUSED && t == pos) we[e] = fmaf(-pre[e], q[c][e], act_val(vwn));
            we[e] = t < n ? we[e] : 0.f;
          }
        }
        f32x4_t ua = {0.f, 0.f, 0.f, 0.f}, ub = ua;
        ua = __builtin_amdgcn_mfma_f32_16x16x4f32(rr[0], we[0], ua, 0, 0, 0);
        ub = __builtin_amdgcn_mfma_f32_16x16x4f32(rr[1], we[1], ub, 0, 0, 0);
        ua = __builtin_amdgcn_mfma_f32_16x16x4f32(rr[2], we[2], ua, 0, 0, 0);
        ub = __builtin_amdgcn_mfma_f32_16x16x4f32(rr[3], we[3], ub, 0, 0, 0);
        o *= lc;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          q[c][e] = (ua[e] + ub[e]) * post[e];
          o = fmaf(q[c][e], dq[e], o);
        }
#pragma unroll
        for (int cc = c + 1; cc < NF; ++cc) {
          const f32x4_t g4 = *(const f32x4_t*)(lds + gram_tile(c, cc) + 4 * (l16 * kGS + 4 * q4));
          f32x4_t qa = q[cc] * lc, qb = {0.f, 0.f, 0.f, 0.f};
          qa = __builtin_amdgcn_mfma_f32_16x16x4f32(g4[0], q[c][0], qa, 0, 0, 0);
          qb = __builtin_amdgcn_mfma_f32_16x16x4f32(g4[1], q[c][1], qb, 0, 0, 0);
          qa = __builtin_amdgcn_mfma_f32_16x16x4f32(g4[2], q[c][2], qa, 0, 0, 0);
          qb = __builtin_amdgcn_mfma_f32_16x16x4f32(g4[3], q[c][3], qb, 0, 0, 0);
          q[cc] = qa + qb;
        }
      }
      // U~ decayed to the end of the ring, and the checkpoint's own weight
#pragma unroll
      for (int c = 0; c < NF - 1; ++c) q[c] *= ll[4 + c];
      const float lam = ll[8] * scp;
      GDNR_COMPILER_FENCE();
      // the f16 parts of a row's U~ scaled by a power of two (the row's largest
      // to [2^13, 2^14)), undone on the row's state
      float up = 1.f, down = 1.f;
      if constexpr (!kBF16) {
        float mx = 0.f;
#pragma unroll
        for (int c = 0; c < NF; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) mx = fmaxf(mx, fabsf(q[c][e]));
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (mx > 0x1p-80f && mx < 0x1p80f) {
          int ex;
          (void)frexpf(mx, &ex);
          up = ldexpf(1.f, 14 - ex);
          down = ldexpf(1.f, ex - 14);
        }
      }
      // S_n of the tile's 8 column groups: lane (nn, q4) gets
      // S_n[row][32 q4 + 4 ct + e], code byte 4 ct + e of its 32; U~ of two
      // chunks at a time in three parts
      const float ls = lam * up;
      const int ko = kLdsX + (4 * q4 + (l16 >> 2)) * kXS + 64 * (l16 & 3);
      f32x4_t sv[8];
#pragma unroll
      for (int ct = 0; ct < 8; ++ct) {
        float f[4];
        fp8x4_to_f32(cw[ct >> 2][ct & 3], f);
        sv[ct] = f32x4_t{ls * f[0], ls * f[1], ls * f[2], ls * f[3]};
      }
#pragma unroll
      for (int hh = 0; hh < NF / 2; ++hh) {
        u32x4_t ub[3];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const f32x4_t x = q[2 * hh + d] * up;
          const Split3 s01 = split3_act(x[0], x[1]), s23 = split3_act(x[2], x[3]);
          ub[0][2 * d] = s01.hi, ub[0][2 * d + 1] = s23.hi;
          ub[1][2 * d] = s01.mid, ub[1][2 * d + 1] = s23.mid;
          ub[2][2 * d] = s01.lo, ub[2][2 * d + 1] = s23.lo;
        }
        u32x4_t k8[8];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          // (two groups' K^T operands at a time)
#pragma unroll
          for (int ct = 4 * g; ct < 4 * g + 4; ++ct) {
            const uint2 k0 = kt_read(ko + 2 * NT * hh * kXS + 8 * ct);
            const uint2 k1 = kt_read(ko + (2 * hh + 1) * NT * kXS + 8 * ct);
            k8[ct] = u32x4_t{k0.x, k0.y, k1.x, k1.y};
          }
#pragma unroll
          for (int d = 2; d >= 0; --d)
#pragma unroll
            for (int ct = 4 * g; ct < 4 * g + 4; ++ct) sv[ct] = mfma16(k8[ct], ub[d], sv[ct]);
          GDNR_COMPILER_FENCE();
        }
      }
      if constexpr (!kBF16) {
#pragma unroll
        for (int ct = 0; ct < 8; ++ct) sv[ct] *= down;
      }
      // A value that is infinite in the last token makes its row of the state
      // +-inf (beta v k^T) in the recurrence, and the row's vblock is scaled
      // by that; the products make NaN of the whole row (0 inf, and inf - inf
      // between U~'s parts). Such rows are found and written here. (An infinity
      // anywhere else in the ring, or a NaN, makes NaN of the row in the
      // recurrence too.)
      if (__builtin_expect(__any(!(__builtin_fabsf(o) < __builtin_inff())), 0)) {
        bool rest = scp < __builtin_inff(), mine = false, neg = false;
        auto finite = [](float x) { return __builtin_fabsf(x) < __builtin_inff(); };
        // (v and the codes read again: the loop's registers are left alone)
#pragma unroll 1
        for (int k = 0; k < 4 * NF; ++k) {
          const int t = NT * (k >> 2) + 4 * q4 + (k & 3);
          if (t >= n) continue;
          const uint8_t* vt = FUSED && t == pos ? f_new : f_rows + (uint32_t)t * a.v_t;
          const float x = act_val(*(const uint16_t*)(vt + (32 * p + l16) * ES));
          const float2 f = *(const float2*)(fl + 8 * t);
          rest = rest && finite(f.x) && finite(f.y) && finite(*(const float*)(lds + kLdsDq + 4 * t));
          if (t + 1 < n) rest = rest && finite(x);
          else mine = __builtin_fabsf(x) == __builtin_inff() && f.y != 0.f, neg = (x < 0.f) != (f.y < 0.f);
        }
#pragma unroll 1
        for (int k = 0; k < 8; ++k) {
          const uint32_t w = ld32(fc_rows + (uint32_t)(32 * p + l16) * a.ck_v + 32 * q4 + 4 * k);
          rest = rest && (((w & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u) == 0;
        }
        // (the four lanes of a row)
        uint64_t rm = __ballot(rest), im = __ballot(mine), nm = __ballot(mine && neg);
        rm &= rm >> 32, im |= im >> 32, nm |= nm >> 32;
        rm &= rm >> 16, im |= im >> 16, nm |= nm >> 16;
        if (((rm & im) >> l16) & 1) {
          const float x = (nm >> l16) & 1 ? -__builtin_inff() : __builtin_inff();
#pragma unroll
          for (int ct = 0; ct < 8; ++ct) {
            const uint2 kw = *(const uint2*)(lds + kLdsX + (n - 1) * kXS + 64 * q4 + 8 * ct);
            const float2 k01 = Act::from_pair(kw.x), k23 = Act::from_pair(kw.y);
            sv[ct] = f32x4_t{x * k01.x, x * k01.y, x * k23.x, x * k23.y};
          }
        }
      }
      // (the next vblock's codes, while this one is requantised)
      if (p + 1 < p1) load_codes(p + 1);
      // the reference quantiser (ref:36-37,83-99), as gdnr_decode.hip applies
      // it; the vblock's amax over the pair's two tiles through LDS (two slots
      // in turn: one barrier a vblock)
      float am = 0.f, am1 = 0.f;
#pragma unroll
      for (int ct = 0; ct < 8; ++ct) {
        am = max3_abs(am, sv[ct][0], sv[ct][1]);
        am1 = max3_abs(am1, sv[ct][2], sv[ct][3]);
      }
      const float am_mine = __uint_as_float(wave_max_u32(__float_as_uint(__builtin_elementwise_maximum(am, am1))));
      float* const rp = red + NW * (p & 1);
      if (lane == 0) rp[w] = am_mine;
      lds_barrier();
      const uint32_t am_bits = (uint32_t)uni((int)max(__float_as_uint(am_mine), __float_as_uint(rp[w ^ 1])));
      const float amax = __uint_as_float(am_bits);
      const float s32 = (amax > 0.0f) ? amax / 448.0f : 1.0f;
      {
        o = rows_reduce_scatter(o, 0.f, 0.f, 0.f);
        if (q4 == 0) Act::st(fo_rows, 32 * p + l16, o * a.out_scale);
      }
      uint8_t* const row = fc_rows + (uint32_t)(32 * p + l16) * a.ck_v + 32 * q4;
      auto store_codes = [&](auto quant) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          uint32_t wd[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) wd[k] = quant(sv[4 * hh + k]);
          *(g_u32x4_w*)(row + 16 * hh) = u32x4_t{wd[0], wd[1], wd[2], wd[3]};
        }
      };
      if (quotient_fast(am_bits, s32)) {
        const double r64 = 1.0 / (double)s32;
        store_codes([&](const f32x4_t& v) {
          return f32x4_to_fp8(quotient_f64(v[0], r64), quotient_f64(v[1], r64), quotient_f64(v[2], r64),
                              quotient_f64(v[3], r64));
        });
      } else {
        store_codes([&](const f32x4_t& v) {
          return f32x4_to_fp8_ref_cold(v[0] / s32, v[1] / s32, v[2] / s32, v[3] / s32);
        });
      }
      if (lane == 0 && (w & 1) == 0) *(uint16_t*)(fs_rows + p * a.sc_v) = __builtin_bit_cast(uint16_t, (_Float16)s32);
    }
  };
  if (n <= 2 * NT)
    rebuild(std::integral_constant<int, 2>{});
  else
    rebuild(std::integral_constant<int, NC>{});
  // the new token's v rows
  if constexpr (FUSED) {
    if (pos >= 0 && half == 0 && lane < CPT) *(u32x4_t*)(v_rows + (uint32_t)pos * a.v_t + 16 * lane) = *(const g_u32x4*)(v_new + 16 * lane);
  }
}

template <int VB, int WPH, bool FUSED, bool GATE_F32, bool SLOTS>
int launch_variant(const StepArgs& a, hipStream_t s) {
  const int extra = a.seq_major ? std::min(a.B, kRingHalves) : 0;
  const dim3 grid((unsigned)(a.H * a.units), (unsigned)(a.B + extra));
  hipLaunchKernelGGL((ring_kernel<VB, WPH, FUSED, GATE_F32, SLOTS>), grid, dim3(64 * NW), ring_lds(NW / WPH, VB), s,
                     a.valid_len, a.pos, a.flush, a.vl_s, a.pos_s, a.fl_s, a.L, a.units,
                     a.seq_major ? 1 + extra : 0, a.G, a);
  return (int)hipGetLastError();
}

template <int VB, int WPH>
int launch_shape(const StepArgs& a, bool fused, bool gate_f32, hipStream_t s) {
  if (!fused) return launch_variant<VB, WPH, false, false, false>(a, s);
  if (a.slot && gate_f32) return launch_variant<VB, WPH, true, true, true>(a, s);
  if (a.slot) return launch_variant<VB, WPH, true, false, true>(a, s);
  if (gate_f32) return launch_variant<VB, WPH, true, true, false>(a, s);
  return launch_variant<VB, WPH, true, false, false>(a, s);
}

}  // namespace

// a.nwh waves of a.V / a.nwh rows per value head (launch_ring in gdnr_abi.cpp)
int GDNR_SUFFIX(launch_ring)(const StepArgs& a, bool fused, bool gate_f32, void* stream) {
  const hipStream_t s = (hipStream_t)stream;
  if (a.nwh == 2) return a.V == 128 ? launch_shape<2, 2>(a, fused, gate_f32, s) : launch_shape<1, 2>(a, fused, gate_f32, s);
  return a.V == 256 ? launch_shape<2, 4>(a, fused, gate_f32, s) : launch_shape<1, 4>(a, fused, gate_f32, s);
}

}  // namespace gdnr

#endif  // GDNR_ACT != 2
