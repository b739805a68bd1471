// Paged int8 attention for long query windows (chunked prefill, whole
// prompts, a cascade's shared prefix): more query rows per KV head than the
// verify kernel of attn_mfma.hip holds in one workgroup.  Same semantics (the
// SDPA call with L > 1 new rows and the block-causal mask of
// Sources/KrillEngine/BatchedDecode.swift:299-312), same flat block split,
// same partial slots.
//
// Bound: the matrix cores and the VALU in turn, and the clock, which falls to
// 1.6 - 2.0 GHz under this load.  Per (64 keys x 16 rows) the matrix cores run
// D / 32 steps of Q.K^T and, the weights being pairs of fp16 operands, twice
// that of P.V; the VALU runs the softmax and the scales.  So the work that does
// not depend on the rows is done once per workgroup of 64 or 128 rows, and what
// depends on (row, key) is kept to the fewest instructions:
//  * a block's K and V bytes go global -> registers -> fp16 tiles in LDS
//    (exact u - 128; row mode: dequantized as the reference does), converted
//    once for all waves; the next block's bytes are in flight meanwhile.
//    Scale and zero words become fp32 (K scale, z + 128 s) and fp16 (V scale)
//    arrays beside them;
//  * the zero-point term sum_g (z + 128 s)_g * (sum of q over group g) is a
//    contraction over the scale groups: fp32 MFMA, four groups a step;
//  * the softmax scale rides on the scales of K and the scores' accumulators
//    start at minus the running reference (row mode: both in the exponent's
//    fma);
//  * weights p * s_v are split into fp16 high and low parts in three full-rate
//    instructions each, alternating with the products of the step before.
// Measured on one card, calls with their append (the verify kernel, or at
// head_dim 512 the decode kernel, before): 8 x 512 rows on contexts of
// 2048-6144, Hq 40, D 128: 789 us = 463 TFLOP/s (1108); a 3900-row prompt, row
// mode, Hq 32: 242 us = 515 TFLOP/s (534); 2 x 256 rows at head_dim 512: 145 us
// (310); 4 x 512 rows, window 1024, head_dim 256: 169 us (304).  Other cards
// differ by up to 5 %.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "attn_common.hpp"

namespace krill {

// One workgroup's LDS: fp16 K tile [token][d], fp16 V^T tile [d][position],
// rows padded by 16 bytes (the 8 rows a group of lanes reads start in
// different banks), and the blocks' scales.
template <int D, int MODE>
struct PrefillLds {
  static constexpr int G = MODE == MODE_AFFINE ? D / 64 : 1;
  static constexpr int KTS = D * 2 + 16, VTS = 64 * 2 + 16;
  static constexpr int GZ = (G + 3) / 4 * 4;  // groups of the zero-point contraction
  static constexpr bool AFF = MODE == MODE_AFFINE;
  __attribute__((aligned(16))) uint8_t k[64 * KTS];
  __attribute__((aligned(16))) uint8_t v[D * VTS];
  __attribute__((aligned(16))) float ks[AFF ? G * 64 : 4];      // [g][token]: s times the softmax scale
  __attribute__((aligned(16))) float kz[AFF ? GZ * 64 : 4];     // [g][token]: z + 128 s, the same
  __attribute__((aligned(16))) float vz[AFF ? G * 64 : 4];      // [g][position]: z + 128 s
  __attribute__((aligned(16))) _Float16 vs[AFF ? G * 64 : 8];   // [g][position]
  int big;  // last block with a V scale past kBigScale
};

__device__ __forceinline__ float4_t mfma16x16x4f32(float a, float b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The larger of two, one instruction (fmaxf first quiets operands the compiler
// cannot see through).
__device__ __forceinline__ float max2(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, INFINITY); }
// Two binary32 weights as fp16 high parts (round to nearest), and the fp16
// rounding of their remainders.  The empty asm keeps the conversions packed
// and the compiler from v_fma_mixlo_f16 / v_fma_mixhi_f16, which run at half
// rate (8 cycles against 4 for the others); `one` is 1.0 where it cannot see
// it, so that a remainder is one mixed fma.
__device__ __forceinline__ half2_t round_pair(float &w0, float &w1) {
  asm("" : "+v"(w0), "+v"(w1));
  uint32_t u = h2_as_u32(half2_t{(_Float16)w0, (_Float16)w1});
  asm("" : "+v"(u));
  return u32_as_h2(u);
}
__device__ __forceinline__ half2_t rest_pair(float w0, float w1, half2_t h, float one) {
  float r0 = __builtin_fmaf(w0, one, -(float)h[0]), r1 = __builtin_fmaf(w1, one, -(float)h[1]);
  asm("" : "+v"(r0), "+v"(r1));
  return half2_t{(_Float16)r0, (_Float16)r1};
}
// Nothing crosses: the schedule is written out (an MFMA occupies the matrix
// core for four VALU slots, and a wave issues in order, so products and VALU
// work only overlap within a wave where they alternate).
__device__ __forceinline__ void fence_all() { __builtin_amdgcn_sched_barrier(0); }
// A raised reference lies kMaxGap below the row's maximum (log2 units): the
// weights then sit high in fp16's range, where the low parts of p s_v keep
// their 11 bits (at the maximum itself most were subnormal: 4.8e-6 of the
// result against 64 bits, about 2e-7 so).  It is raised when a score exceeds it
// by kMaxOver, so p < 2^8 and p s_v stays finite in fp16 for |s_v| <= kBigScale
// (V values of some +-32000 in one group, or scales brought in from outside).
// A block with a larger scale raises it to the maximum itself: p <= 1 there.
// (The test takes 9 of 762 us on the 8 x 512-row chunks; kMaxOver 6.9, which
// bounds p s_v for the quantizer's own scales only, takes the same: more raises.)
constexpr float kMaxGap = 5.0f, kMaxOver = 8.0f, kBigScale = 248.0f;
// No LDS read crosses: what is read above stays above, in flight.
__device__ __forceinline__ void fence_lds() { __builtin_amdgcn_sched_barrier(0x47f); }

// Waves of a workgroup: one per (32-token group, 16-position half) of a V row.
constexpr int kPrefillWaves = 4;
// Where in a head region the loads of a block lie: piece k of wave `wid` starts
// at `piece` bytes (a scalar offset), each lane reads at its own offset from
// there.  The range check of a buffer load does not cover the scalar offset, so
// the sums must lie in the region by themselves.
constexpr int prefill_k_piece(int wid, int k) { return (wid + kPrefillWaves * k) * 1024; }
template <int D>
constexpr int prefill_v_piece(int wid, int k) {
  return v_offset(D) + ((wid >> 1) & 1) * 32 * D + (wid & 1) * 1024 + k * (64 / (D / 64) * 16);
}
// row `lane` of a 64-row run of V^T
template <int D>
constexpr int prefill_v_lane(int lane) { return 2 * (lane % (D / 64)) * 1024 + lane / (D / 64) * 16; }
// affine metadata, runs of 64 words: 128 G words, at G = 1 half of what the four
// waves would load -- the other two read the same words again (unused)
template <int D, int G>
constexpr int prefill_meta_piece(int wid, int k) {
  const int run = wid + kPrefillWaves * k;
  return km_offset(D) + 256 * (2 * G < kPrefillWaves ? run % (2 * G) : run);
}
template <int D, int G>
constexpr bool prefill_loads_inside(int k_pieces, int v_pieces, int meta_pieces) {
  for (int w = 0; w < kPrefillWaves; ++w)
    for (int lane = 0; lane < 64; ++lane) {
      for (int k = 0; k < k_pieces; ++k)
        if (prefill_k_piece(w, k) + 16 * lane + 16 > v_offset(D)) return false;
      for (int k = 0; k < v_pieces; ++k)
        if (prefill_v_piece<D>(w, k) + prefill_v_lane<D>(lane) + 16 > km_offset(D)) return false;
      for (int k = 0; k < meta_pieces; ++k)
        if (prefill_meta_piece<D, G>(w, k) + 4 * lane + 4 > head_region_bytes(D, G)) return false;
    }
  return true;
}
// Waves per SIMD the registers are budgeted for: the accumulators and queries
// of NRT row tiles take 6 NRT D / 16 registers a lane.
template <int D, int NRT>
constexpr int prefill_min_waves() { return NRT * D >= 512 ? 1 : 2; }

// VAR: 0 plain; 1 RoPE of the queries; 2 sliding window.
template <int D, int MODE, int NRT, int VAR>
__global__ __launch_bounds__(256, (prefill_min_waves<D, NRT>())) void k_attn_prefill(AttnArgs a) {
  constexpr bool ROPE = VAR == 1, WIN = VAR == 2, AFF = MODE == MODE_AFFINE;
  constexpr int G = AFF ? D / 64 : 1;
  constexpr int GZ4 = (G + 3) / 4;
  constexpr int KS = D / 32;      // 32-d steps of Q.K^T
  constexpr int NDT = D / 16;     // 16-d tiles of P.V
  constexpr int W = kPrefillWaves;
  constexpr int RR = 16 * NRT;    // query rows per wave
  constexpr int KP = D / 16 / W;  // 16-byte K pieces per thread
  constexpr int VP = D / 16 / W;  // 16-byte V pieces per thread
  constexpr int MW = AFF ? (128 * G + 64 * W - 1) / (64 * W) : 0;  // metadata words per thread
  static_assert(W == 4 && D % 64 == 0, "a wave per (token group, half) of V");
  static_assert(prefill_loads_inside<D, G>(KP, VP, MW), "a block's loads stay in its head region");
  using Lds = PrefillLds<D, MODE>;
  constexpr int KTS = Lds::KTS, VTS = Lds::VTS;
  __shared__ Lds lds;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, q4 = lane >> 4;
  // Workgroup order: KV head fastest (workgroups go to the 8 XCDs round-robin,
  // so with 8 heads each head's blocks stay in one XCD's L2), then the block
  // ranges, the row groups with the most visible keys first
  const int RGB = (a.row_groups + W - 1) / W;
  const int hk = (int)(blockIdx.x % (unsigned)a.Hkv);
  const int rest = (int)(blockIdx.x / (unsigned)a.Hkv);
  const int rg = (RGB - 1 - rest / a.waves) * W + wid;
  const int wv = __builtin_amdgcn_readfirstlane(rest % a.waves);
  const int rbase = rg * RR;  // rg >= row_groups (a workgroup's spare wave): no valid row

  // ---- this workgroup's flat blocks [i0, iend) of the (head, row group) order
  int c0 = 0, lenv = lane < a.B ? seq_len_view<WIN>(a, lane) : 0;
  int nbv = seq_blocks_rg(a, lenv, rg);
  int incl = wave_incl_scan(nbv);
  int T = __builtin_amdgcn_readlane(incl, 63);
  for (int cc = 64; cc < a.B; cc += 64) {
    const int bb = cc + lane;
    T += __builtin_amdgcn_readfirstlane(wave_allsum_int(bb < a.B ? seq_blocks_rg(a, seq_len_view<WIN>(a, bb), rg) : 0));
  }
  const int Wt = min(a.waves, T);
  if (wv >= Wt) return;
  const int i0 = __builtin_amdgcn_readfirstlane((int)(((int64_t)wv * T + Wt - 1) / Wt));
  const int iend = __builtin_amdgcn_readfirstlane((int)(((int64_t)(wv + 1) * T + Wt - 1) / Wt));
  int b = -1, s = 0;
  {
    int carry = 0;
    for (c0 = 0; c0 < a.B; c0 += 64) {
      if (c0 > 0) {
        const int bb = c0 + lane;
        lenv = bb < a.B ? seq_len_view<WIN>(a, bb) : 0;
        nbv = seq_blocks_rg(a, lenv, rg);
        incl = wave_incl_scan(nbv) + carry;
      }
      const unsigned long long m = __ballot(c0 + lane < a.B && incl > i0);
      if (m) {
        const int l = __builtin_ctzll(m);
        b = c0 + l;
        s = __builtin_amdgcn_readlane(incl - nbv, l);
        break;
      }
      carry = __builtin_amdgcn_readlane(incl, 63);
    }
  }
  if (b < 0) return;
  auto seq_len = [&](int bs) -> int { return bs - c0 < 64 ? __builtin_amdgcn_readlane(lenv, bs - c0) : seq_len_view<WIN>(a, bs); };

  // block-table entries of flat blocks tab0 .. tab0 + 63, lane j: block
  // tab0 + j; reloaded every 64 blocks, walking on from sequence b
  int tab = 0, tab0 = i0;
  auto load_table = [&](int from) {
    const int f = from + lane;
    int bs = b, ss = s;
    tab = 0;
    while (bs < a.B && ss < min(iend, from + 64)) {
      const int nbs = seq_blocks_rg(a, seq_len(bs), rg);
      if (f < iend && f >= ss && f < ss + nbs) {
        const int phys = a.tables[(int64_t)bs * a.max_blocks + table_offset<WIN>(a, bs) + (f - ss)];
        tab = (unsigned)phys < (unsigned)a.lv.num_blocks ? phys : 0;
      }
      ss += nbs;
      ++bs;
    }
    tab0 = from;
  };
  load_table(i0);

  // ---- the block in registers: K piece k is 16-d chunk wid + W k of token
  // `lane`; V piece k holds positions 16 h .. +15 of token group tg, row d =
  // 64 k + lane, the same (tg, h) for all pieces of a wave
  const int vtg = (wid >> 1) & 1, vh = wid & 1;
  uint4 kraw[KP], vraw[VP];
  uint32_t mraw[AFF ? MW : 1];  // affine: words tid + 64 W k of the block's metadata; row mode: K word of token `lane`
  uint32_t vmeta = 0u;          // row mode: V word of token `lane`
  const int vlane = prefill_v_lane<D>(lane);
  auto issue = [&](int i) {
    // after the last block: an empty resource (the offsets in scalars may escape
    // the range check: then block 0 or a block of this range is read, unused)
    const int bytes = __builtin_amdgcn_readfirstlane(i < iend ? a.lv.head_bytes : 0);
    if (i < iend && i - tab0 == 64) load_table(i);
    const int phys = __builtin_amdgcn_readlane(tab, __builtin_amdgcn_readfirstlane((i - tab0) & 63));
    const __amdgpu_buffer_rsrc_t r = block_rsrc(head_region(a.lv, phys, hk), bytes);
    // (per-lane offset, the wave's and piece's offset in a scalar)
    auto ld16 = [&](int off, int soff) {
      return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
    };
#pragma unroll
    for (int k = 0; k < KP; ++k) kraw[k] = ld16(lane * 16, prefill_k_piece(wid, k));
#pragma unroll
    for (int k = 0; k < VP; ++k) vraw[k] = ld16(vlane, prefill_v_piece<D>(wid, k));
    if constexpr (AFF) {
#pragma unroll
      for (int k = 0; k < MW; ++k)
        mraw[k] = __builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, prefill_meta_piece<D, G>(wid, k), 0);
    } else {
      mraw[0] = __builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, km_offset(D), 0);
      vmeta = __builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, vm_offset(D, G), 0);
    }
  };

  // ---- Q^T operands of sequence bq: lane holds q[row n][32 ks + 8 q4 .. +8]
  half8_t qB[NRT][KS];
  float qz[AFF ? NRT : 1][GZ4];  // sum of the row's fp16 query over group 4 j + q4 (0 past the groups)
  // the lane's row (row mode): the query's 2^k times |softmax scale| in log2
  // units; in affine mode the scales of K carry that scale
  float q_up[AFF ? 1 : NRT];
  float q_dn[AFF ? NRT : 1];  // affine: 2^-k alone
  bool any_up = false;        // affine: some row of the wave has a 2^k other than 1
  bool rvalid[NRT];
#pragma unroll
  for (int rt = 0; rt < NRT; ++rt) rvalid[rt] = rbase + 16 * rt + n < a.NR;
  // row mode: the sign of the scale goes to the queries (zero scale: zero queries)
  const float qsign = AFF || a.scale_log2 > 0.0f ? 1.0f : a.scale_log2 < 0.0f ? -1.0f : 0.0f;
  const float qscale = AFF || qsign == 0.0f ? 1.0f : fabsf(a.scale_log2);
  auto load_q = [&](int bq) {
    bool ups = false;
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const int r = rvalid[rt] ? rbase + 16 * rt + n : 0;
      const int hq = hk * a.R + r % a.R, j = r / a.R;
      const uint16_t *qp = q_row(a, bq, hq, j);
      uint4 qraw[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qraw[ks] = *reinterpret_cast<const uint4 *>(qp + 32 * ks + 8 * q4);
      if constexpr (ROPE) {
        // query position j = r / R, token len - Lq + j: the 8 elements of
        // step ks < KS/2 turn with those of step ks + KS/2
        const float *crow = rope_row(a, seq_len(bq) - a.Lq + j, D);
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks) {
          const int d = 32 * ks + 8 * q4;
          uint32_t lo[4] = {qraw[ks].x, qraw[ks].y, qraw[ks].z, qraw[ks].w};
          uint32_t hi[4] = {qraw[ks + KS / 2].x, qraw[ks + KS / 2].y, qraw[ks + KS / 2].z, qraw[ks + KS / 2].w};
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const float2 c2 = *reinterpret_cast<const float2 *>(crow + d + 2 * w);
            const float2 s2 = *reinterpret_cast<const float2 *>(crow + D / 2 + d + 2 * w);
            if (a.q_dtype == DT_BF16)
              rope_pair_words<DT_BF16>(lo[w], hi[w], c2, s2);
            else
              rope_pair_words<DT_F16>(lo[w], hi[w], c2, s2);
          }
          qraw[ks] = uint4{lo[0], lo[1], lo[2], lo[3]};
          qraw[ks + KS / 2] = uint4{hi[0], hi[1], hi[2], hi[3]};
        }
      }
      // bf16 rows at the fp16 range limit are scaled by 2^-k before the
      // rounding, their scores by 2^k (q_range_scale); the row's elements
      // sit in lanes n, n + 16, n + 32, n + 48
      float down = 1.0f, up = 1.0f;
      if (a.q_dtype == DT_BF16) {
        float mx = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const uint32_t w4[4] = {qraw[ks].x, qraw[ks].y, qraw[ks].z, qraw[ks].w};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            mx = fmaxf(mx, fmaxf(fabsf(__builtin_bit_cast(float, w4[e] << 16)),
                                 fabsf(__builtin_bit_cast(float, w4[e] & 0xffff0000u))));
        }
        mx = fmaxf(mx, shfl_xor(mx, 16));
        mx = fmaxf(mx, shfl_xor(mx, 32));
        down = q_range_scale(mx, up);
      }
      q_up[rt] = qscale * up;
      if constexpr (AFF) q_dn[rt] = down;
      ups |= up != 1.0f;
      float qsum[G];
#pragma unroll
      for (int g = 0; g < G; ++g) qsum[g] = 0.0f;
      const float mul = rvalid[rt] ? qsign : 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const uint32_t w4[4] = {qraw[ks].x, qraw[ks].y, qraw[ks].z, qraw[ks].w};
        half8_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float lo, hi;
          if (a.q_dtype == DT_BF16) {
            lo = __builtin_bit_cast(float, w4[e] << 16) * down;
            hi = __builtin_bit_cast(float, w4[e] & 0xffff0000u) * down;
          } else {
            lo = f16_bits_to_f32((uint16_t)(w4[e] & 0xffffu));
            hi = f16_bits_to_f32((uint16_t)(w4[e] >> 16));
          }
          const _Float16 hl = mul != 0.0f ? (_Float16)(lo * mul) : (_Float16)0.0f;
          const _Float16 hh = mul != 0.0f ? (_Float16)(hi * mul) : (_Float16)0.0f;
          v[2 * e] = hl;
          v[2 * e + 1] = hh;
          qsum[AFF ? ks / 2 : 0] += (float)hl + (float)hh;
        }
        qB[rt][ks] = v;
      }
      if constexpr (AFF) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          qsum[g] += shfl_xor(qsum[g], 16);
          qsum[g] += shfl_xor(qsum[g], 32);
        }
#pragma unroll
        for (int j4 = 0; j4 < GZ4; ++j4) {
          float v = 0.0f;
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (4 * j4 + k < G) v = q4 == k ? qsum[4 * j4 + k] : v;
          qz[rt][j4] = v;
        }
      }
    }
    any_up = __any(ups);
  };

  // ---- fragment loads: K tile t, fragments CH c .. +CH-1, the scales of
  // their groups; V^T slice sl of token group tg, its group's scales
  constexpr int CH = KS < 4 ? KS : 4, CPT = KS / CH, NSL = D / 64;
  struct VMeta {
    half8_t s;
    float4_t z[2];
  };
  auto ldk = [&](half8_t(&f)[4], int t, int c) {
    const uint8_t *kt = lds.k + (16 * t + n) * KTS + 16 * q4;
#pragma unroll
    for (int j = 0; j < CH; ++j) f[j] = *reinterpret_cast<const half8_t *>(kt + 64 * (CH * c + j));
  };
  auto ldv = [&](half8_t(&f)[4], int tg, int sl) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      f[j] = *reinterpret_cast<const half8_t *>(lds.v + (64 * sl + 16 * j + n) * VTS + tg * 64 + 16 * q4);
  };
  auto ldvm = [&](VMeta &m, int tg, int sl) {
    if constexpr (AFF) {
      const int o = sl * 64 + 32 * tg + 8 * q4;
      m.s = *reinterpret_cast<const half8_t *>(lds.vs + o);
      m.z[0] = *reinterpret_cast<const float4_t *>(lds.vz + o);
      m.z[1] = *reinterpret_cast<const float4_t *>(lds.vz + o + 4);
    }
  };

  if constexpr (AFF && Lds::GZ > G) {  // the zero-point contraction's unused groups
    for (int k = tid; k < (Lds::GZ - G) * 64; k += 64 * W) lds.kz[G * 64 + k] = 0.0f;
  }
  if (AFF && tid == 0) lds.big = -1;
  issue(i0);
  load_q(b);

  float one = 1.0f;
  asm volatile("" : "+v"(one));
  int i = i0;
  while (true) {
    const int len = seq_len(b);
    const int e = s + seq_blocks_rg(a, len, rg);
    const int seg_end = __builtin_amdgcn_readfirstlane(min(e, iend));
    int lim[NRT];
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      const int r = rbase + 16 * rt + n;
      lim[rt] = rvalid[rt] ? key_limit(a, len, r / a.R) : 0;
    }
    const int lim_lo = key_limit(a, len, rbase / a.R);  // keys seen by the wave's first row
    int lo[NRT], wst = 0, lo_hi = 0;  // sliding window: per-row first key, first retained key, the wave's largest
    if constexpr (WIN) {
      wst = win_view_start(a, b);
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        const int r = rbase + 16 * rt + n;
        lo[rt] = max(wst, len - a.Lq + r / a.R - a.window + 1);
      }
      const int rlast = min(a.NR, rbase + RR) - 1;
      lo_hi = max(wst, len - a.Lq + rlast / a.R - a.window + 1);
    }
    float m_run[NRT], l_part[NRT], c_part[NRT][G];
    float nm[NRT];  // affine: the scores' accumulators start here, -m 2^-k (0 before the first block)
    float4_t oacc[NRT][NDT];
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      m_run[rt] = -INFINITY;
      l_part[rt] = 0.0f;
      nm[rt] = 0.0f;
#pragma unroll
      for (int g = 0; g < G; ++g) c_part[rt][g] = 0.0f;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) oacc[rt][dt] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }

    for (; i < seg_end; ++i) {
      const int tbase = (i - s) << 6;
      // ---- convert the block into the workgroup's tiles once every wave is
      // past its reads of the previous block
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      // (the lane as an unknown of each block: its LDS addresses are computed
      // here instead of held in registers through the products)
      int ln = lane;
      asm volatile("" : "+v"(ln));
      if constexpr (AFF) {
#pragma unroll
        for (int k = 0; k < KP; ++k) {
          uint8_t *o = lds.k + ln * KTS + (wid + W * k) * 32;
          *reinterpret_cast<half8_t *>(o) = bytes8_centred(uint2{kraw[k].x, kraw[k].y});
          *reinterpret_cast<half8_t *>(o + 16) = bytes8_centred(uint2{kraw[k].z, kraw[k].w});
        }
#pragma unroll
        for (int k = 0; k < VP; ++k) {
          uint8_t *o = lds.v + (64 * k + ln) * VTS + vtg * 64 + vh * 32;
          *reinterpret_cast<half8_t *>(o) = bytes8_centred(uint2{vraw[k].x, vraw[k].y});
          *reinterpret_cast<half8_t *>(o + 16) = bytes8_centred(uint2{vraw[k].z, vraw[k].w});
        }
#pragma unroll
        for (int k = 0; k < MW; ++k) {
          const int m = 64 * wid + ln + 64 * W * k;
          const int mm = m & (64 * G - 1), t = mm / G, g = mm % G;
          const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)(mraw[k] & 0xffffu));
          const float sf = (float)sh, zf = fmaf(128.0f, sf, f16_bits_to_f32((uint16_t)(mraw[k] >> 16)));
          if (m < 64 * G) {
            lds.ks[g * 64 + t] = sf * a.scale_log2;
            lds.kz[g * 64 + t] = zf * a.scale_log2;
          } else if (m < 128 * G) {
            // rows past the sequence's end or below the window are not data
            bool data = tbase + t < len;
            if constexpr (WIN) data = data && tbase + t >= wst;
            const int p = (t & 32) + vpos(t & 31);
            lds.vs[g * 64 + p] = data ? sh : (_Float16)0.0f;
            lds.vz[g * 64 + p] = data ? zf : 0.0f;
            if (data && fabsf(sf) > kBigScale) lds.big = i;
          }
        }
      } else {
        const half2_t m1024 = half2_t{(_Float16)-1024.0f, (_Float16)-1024.0f};
        const _Float16 sk = __builtin_bit_cast(_Float16, (uint16_t)(mraw[0] & 0xffffu));
        const _Float16 zk = __builtin_bit_cast(_Float16, (uint16_t)(mraw[0] >> 16));
        const half2_t ks2 = half2_t{sk, sk}, kz2 = half2_t{zk, zk};
#pragma unroll
        for (int k = 0; k < KP; ++k) {
          const uint32_t w4[4] = {kraw[k].x, kraw[k].y, kraw[k].z, kraw[k].w};
          uint32_t o8[8];
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            o8[2 * x] = h2_as_u32((bytes01_plus1024(w4[x]) + m1024) * ks2 + kz2);
            o8[2 * x + 1] = h2_as_u32((bytes23_plus1024(w4[x]) + m1024) * ks2 + kz2);
          }
          uint8_t *o = lds.k + ln * KTS + (wid + W * k) * 32;
          *reinterpret_cast<uint4 *>(o) = uint4{o8[0], o8[1], o8[2], o8[3]};
          *reinterpret_cast<uint4 *>(o + 16) = uint4{o8[4], o8[5], o8[6], o8[7]};
        }
        // the pieces' 16 positions (the wave's tg and h): fp16 scales and zero
        // points, pairs per word, from the lanes of their tokens
        bool data = tbase + ln < len;
        if constexpr (WIN) data = data && tbase + ln >= wst;
        const uint32_t vw = data ? vmeta : 0u;
        uint32_t sc8[8], zc8[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          const uint32_t w0 = __builtin_amdgcn_readlane(vw, 32 * vtg + 8 * vh + vtok(2 * x));
          const uint32_t w1 = __builtin_amdgcn_readlane(vw, 32 * vtg + 8 * vh + vtok(2 * x + 1));
          sc8[x] = (w0 & 0xffffu) | (w1 << 16);
          zc8[x] = (w0 >> 16) | (w1 & 0xffff0000u);
        }
#pragma unroll
        for (int k = 0; k < VP; ++k) {
          uint8_t *o = lds.v + (64 * k + ln) * VTS + vtg * 64 + vh * 32;
          *reinterpret_cast<half8_t *>(o) =
              bytes8_dequant_ref(uint2{vraw[k].x, vraw[k].y}, uint4{sc8[0], sc8[1], sc8[2], sc8[3]},
                                 uint4{zc8[0], zc8[1], zc8[2], zc8[3]});
          *reinterpret_cast<half8_t *>(o + 16) =
              bytes8_dequant_ref(uint2{vraw[k].z, vraw[k].w}, uint4{sc8[4], sc8[5], sc8[6], sc8[7]},
                                 uint4{zc8[4], zc8[5], zc8[6], zc8[7]});
        }
      }
      issue(i + 1);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

      // some row of this wave does not see every token of the block (causal
      // edge or the sequence's last block): only then are scores masked
      bool edge = tbase + 64 > lim_lo;
      if constexpr (WIN) edge = edge || tbase < lo_hi;  // or below some row's window

      // ---- S^T = K . Q^T, four 16-token tiles: lane holds tokens
      // 16 t + 4 q4 + e of row n.  Steps of CH operand fragments, their LDS
      // reads issued a step ahead (the fences keep the scheduler from sinking
      // them to their use).  Affine mode: the scores start at -m plus the
      // zero-point term; each scale group's sums are scaled and added while
      // the next group's MFMAs run.
      float4_t sc[4][NRT];
      half8_t fr[2][4];
      constexpr int NGRP = 4 * G;  // (tile, scale group) pairs
      float4_t sacc[AFF ? 2 : 1][NRT], ksg[AFF ? 2 : 1];
      ldk(fr[0], 0, 0);
      if constexpr (AFF) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          float zA[GZ4];
#pragma unroll
          for (int j4 = 0; j4 < GZ4; ++j4) zA[j4] = lds.kz[(4 * j4 + q4) * 64 + 16 * t + n];
#pragma unroll
          for (int rt = 0; rt < NRT; ++rt) {
            sc[t][rt] = float4_t{nm[rt], nm[rt], nm[rt], nm[rt]};
#pragma unroll
            for (int j4 = 0; j4 < GZ4; ++j4) sc[t][rt] = mfma16x16x4f32(zA[j4], qz[rt][j4], sc[t][rt]);
          }
        }
      }
      auto scale = [&](int j, int rt, int h) {  // pair j (tile j / G), row tile rt, half of its tokens
#pragma unroll
        for (int x = 2 * h; x < 2 * h + 2; ++x)
          sc[j / G][rt][x] = __builtin_fmaf(ksg[j & 1][x], sacc[j & 1][rt][x], sc[j / G][rt][x]);
      };
#pragma unroll
      for (int u = 0; u < 4 * CPT; ++u) {
        const int t = u / CPT, c = u % CPT;
        if (u + 1 < 4 * CPT)
          ldk(fr[(u + 1) & 1], (u + 1) / CPT, (u + 1) % CPT);
        else
          ldv(fr[(u + 1) & 1], 0, 0);
        if constexpr (AFF) {
#pragma unroll
          for (int g = 0; g < CH / 2; ++g) {
            const int j = u * (CH / 2) + g;
            ksg[j & 1] = *reinterpret_cast<const float4_t *>(lds.ks + (j % G) * 64 + 16 * t + 4 * q4);
            fence_lds();
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int rt = 0; rt < NRT; ++rt) {
                sacc[j & 1][rt] = mfma16x16x32(fr[u & 1][2 * g + h], qB[rt][CH * c + 2 * g + h],
                                               h == 0 ? float4_t{0.0f, 0.0f, 0.0f, 0.0f} : sacc[j & 1][rt]);
                if (j > 0) {
                  fence_all();
                  scale(j - 1, rt, h);
                  fence_all();
                }
              }
          }
        } else {
          fence_lds();
          // (a chain of 128 dims, then one sum: head_dim 512 in one chain of
          // 16 products rounds worse, 2.6e-7 against 1.7e-7)
#pragma unroll
          for (int rt = 0; rt < NRT; ++rt) {
            float4_t v = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
            if (CPT <= 2 && c > 0) v = sc[t][rt];
#pragma unroll
            for (int j = 0; j < CH; ++j) v = mfma16x16x32(fr[u & 1][j], qB[rt][CH * c + j], v);
            sc[t][rt] = CPT <= 2 || c == 0 ? v : sc[t][rt] + v;
          }
        }
      }
      float over_by = kMaxOver;
      if constexpr (AFF) {
        if (lds.big == i) over_by = 0.0f;
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) {
          scale(NGRP - 1, rt, 0);
          scale(NGRP - 1, rt, 1);
        }
      }
      if constexpr (AFF) {
        if (any_up) {
          asm volatile("; rows scaled by 2^k");  // (a branch, not a multiplication by one)
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
              for (int x = 0; x < 4; ++x) sc[t][rt][x] *= 1.0f / q_dn[rt];
        }
      }
      if (edge) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              const int tok = tbase + 16 * t + 4 * q4 + x;
              if (tok >= lim[rt] || (WIN && tok < lo[rt])) sc[t][rt][x] = -INFINITY;
            }
      }

      // ---- online softmax with a lazily raised running reference m (log2
      // units; the row's 64 scores live in lanes n, n+16, n+32, n+48): it
      // only moves when some score exceeds it by more than kMaxOver, so the
      // weights stay below 2^8 and most blocks skip the rescale
      // (affine mode: scores relative to the running max, 0 before the first)
      float mb[NRT];
      bool over = false;
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        float v = max2(sc[0][rt][0], sc[0][rt][1]);
#pragma unroll
        for (int k = 2; k < 16; k += 2) v = fmaxf(fmaxf(v, sc[k / 4][rt][k % 4]), sc[k / 4][rt][k % 4 + 1]);
        float va = v, vb = v;
        row_swap16(va, vb);
        va = vb = max2(va, vb);
        row_swap32(va, vb);
        v = max2(va, vb);
        if constexpr (AFF) {
          mb[rt] = v;
          over |= v > (m_run[rt] == -INFINITY ? -INFINITY : over_by);
        } else {
          mb[rt] = v * q_up[AFF ? 0 : rt];
          over |= mb[rt] > m_run[rt] + over_by;
        }
      }
      if (__any(over)) {
        const float gap = AFF && over_by == 0.0f ? 0.0f : kMaxGap;
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt) {
          const float mu = m_run[rt] == -INFINITY ? 0.0f : m_run[rt];
          const float mn = fmaxf(m_run[rt], (AFF ? mb[rt] + mu : mb[rt]) - gap);
          const float al = m_run[rt] == -INFINITY ? 0.0f : fast_exp2(m_run[rt] - mn);
          if constexpr (AFF) {
            const float down = mn == -INFINITY ? 0.0f : mn - mu;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
              for (int x = 0; x < 4; ++x) sc[t][rt][x] = fminf(sc[t][rt][x] - down, gap);
            nm[rt] = mn == -INFINITY ? 0.0f : -mn * q_dn[rt];
          }
          m_run[rt] = mn;
          l_part[rt] *= al;
#pragma unroll
          for (int g = 0; g < G; ++g) c_part[rt][g] *= al;
#pragma unroll
          for (int dt = 0; dt < NDT; ++dt) oacc[rt][dt] *= al;
        }
      }
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        const float mu = m_run[rt] == -INFINITY ? 0.0f : m_run[rt];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            sc[t][rt][x] = fast_exp2(AFF ? sc[t][rt][x] : __builtin_fmaf(sc[t][rt][x], q_up[AFF ? 0 : rt], -mu));
          }
      }

      // ---- O^T += V^T . P^T over two 32-token groups: position k of quarter
      // q4 is token 32 tg + 4 q4 + k (k < 4) or 32 tg + 16 + 4 q4 + k - 4.
      // Steps of one 64-d slice (four d tiles, one scale group); the next
      // step's weights are split while this step's MFMAs run.
      half8_t Bh[2][NRT], Bl[2][NRT];
      VMeta mv;
      float ps[NRT];  // the block's sums
      float w0 = 0.0f, w1 = 0.0f;
      half2_t wh;
      // part 2 i + h of the split of step u: pair i = (row tile, positions
      // 2 (i % 4), +1); h = 0 the weights and high parts, 1 the low parts
      auto build = [&](int u, int part) {
        const int tg = u / NSL, sl = u % NSL, bb = AFF ? u & 1 : tg;
        const int rt = part / 8, k = part / 2 % 4 * 2;
        if (part % 2 == 0) {
          w0 = sc[2 * tg + (k >> 2)][rt][k & 3];
          w1 = sc[2 * tg + (k >> 2)][rt][(k & 3) + 1];
          if (sl == 0) ps[rt] = k == 0 && tg == 0 ? w0 + w1 : ps[rt] + w0 + w1;
          if constexpr (AFF) {
            c_part[rt][sl] = __builtin_fmaf(w0, mv.z[k >> 2][k & 3], c_part[rt][sl]);
            c_part[rt][sl] = __builtin_fmaf(w1, mv.z[k >> 2][(k & 3) + 1], c_part[rt][sl]);
            w0 = __builtin_fmaf(w0, (float)mv.s[k], 0.0f);
            w1 = __builtin_fmaf(w1, (float)mv.s[k + 1], 0.0f);
          }
          wh = round_pair(w0, w1);
          Bh[bb][rt][k] = wh[0];
          Bh[bb][rt][k + 1] = wh[1];
        } else {
          const half2_t l = rest_pair(w0, w1, wh, one);
          Bl[bb][rt][k] = l[0];
          Bl[bb][rt][k + 1] = l[1];
        }
      };
      ldvm(mv, 0, 0);
#pragma unroll
      for (int part = 0; part < 8 * NRT; ++part) build(0, part);
      if constexpr (AFF) ldvm(mv, 1 / NSL, 1 % NSL);
#pragma unroll
      for (int u = 0; u < 2 * NSL; ++u) {
        const int sl = u % NSL, bb = AFF ? u & 1 : u / NSL;
        constexpr int F0 = 4 * CPT;  // the fragment buffer of step 0
        const bool next = u + 1 < 2 * NSL && (AFF || (u + 1) % NSL == 0);
        if (u + 1 < 2 * NSL) ldv(fr[(F0 + u + 1) & 1], (u + 1) / NSL, (u + 1) % NSL);
        fence_lds();
#pragma unroll
        for (int m = 0; m < 8 * NRT; ++m) {
          const int j = m / NRT % 4, rt = m % NRT;
          oacc[rt][4 * sl + j] =
              mfma16x16x32(fr[(F0 + u) & 1][j], m < 4 * NRT ? Bh[bb][rt] : Bl[bb][rt], oacc[rt][4 * sl + j]);
          if (next && m > 0) {
            fence_all();
            build(u + 1, m - 1);
            if (m == 8 * NRT - 1) build(u + 1, m);
            fence_all();
          }
        }
        if (AFF && u + 2 < 2 * NSL) ldvm(mv, (u + 2) / NSL, (u + 2) % NSL);
      }
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) l_part[rt] += ps[rt];
    }

    // ---- end of the segment: lane holds O^T[d = 16*dt + 4*q4 + e][row n].
    // The whole sequence in this workgroup -> output; otherwise a partial in
    // slot (hk * row_groups + rg) * (waves + B) + range + b
    const bool whole = !a.partial_only && s >= i0 && e <= iend;
    const int64_t slot = ((int64_t)hk * a.row_groups + rg) * (a.waves + a.B) + wv + b;
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
      float l = l_part[rt];
      l += shfl_xor(l, 16);
      l += shfl_xor(l, 32);
      float cg[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float c = c_part[rt][g];
        c += shfl_xor(c, 16);
        c += shfl_xor(c, 32);
        cg[g] = c;
      }
      if (!rvalid[rt]) continue;
      const float mul = !whole ? 1.0f : l > 0.0f ? 1.0f / l : 0.0f;
      const int64_t pi = slot * RR + 16 * rt + n;
      const int64_t ob = (whole ? out_row_base(a, b, hk, rbase + 16 * rt + n, D) : pi * D) + 4 * q4;
      auto put = [&](void *out, auto dtype) {
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
          float run[4];
#pragma unroll
          for (int x = 0; x < 4; ++x) run[x] = (oacc[rt][dt][x] + cg[AFF ? dt / 4 : 0]) * mul;
          store_run<4>(out, ob + 16 * dt, run, decltype(dtype)::value);
        }
      };
      if (!whole)
        put(a.ws_o, std::integral_constant<int, DT_F32>{});
      else if (a.out_dtype == DT_F32)
        put(a.out, std::integral_constant<int, DT_F32>{});
      else if (a.out_dtype == DT_F16)
        put(a.out, std::integral_constant<int, DT_F16>{});
      else
        put(a.out, std::integral_constant<int, DT_BF16>{});
      if (!whole && q4 == 0) reinterpret_cast<float2 *>(a.ws_ml)[pi] = float2{m_run[rt], l};
    }
    if (i >= iend) break;
    // next sequence with blocks for this row group (the merge zero-fills the others)
    ++b;
    s = e;
    while (b < a.B && seq_blocks_rg(a, seq_len(b), rg) == 0) ++b;
    if (b >= a.B) break;
    load_q(b);
  }
}

template <int D, int MODE, int NRT>
static hipError_t launch_prefill(const AttnArgs &args, unsigned groups, hipStream_t st) {
  const dim3 grid((unsigned)args.waves * (unsigned)args.Hkv * groups), block(64 * kPrefillWaves);
  if (args.rope_cs) {  // (head_dim 512 comes here with several new rows only, RoPE with one)
    if constexpr (D <= 256)
      k_attn_prefill<D, MODE, NRT, 1><<<grid, block, 0, st>>>(args);
    else
      return hipErrorInvalidValue;
  } else if (args.window > 0)
    k_attn_prefill<D, MODE, NRT, 2><<<grid, block, 0, st>>>(args);
  else
    k_attn_prefill<D, MODE, NRT, 0><<<grid, block, 0, st>>>(args);
  return hipGetLastError();
}

// Shapes the plan may choose: waves of 16 rows, or of 32 (head_dim <= 128).
template <int D, int MODE>
static hipError_t launch_prefill_dm(const AttnArgs &args, const AttnPlan &p, hipStream_t st) {
  const unsigned groups = (unsigned)((p.row_groups + p.group_waves - 1) / p.group_waves);
  if (p.group_waves != kPrefillWaves) return hipErrorInvalidValue;
  if (p.nrt == 1) return launch_prefill<D, MODE, 1>(args, groups, st);
  if constexpr (D <= 128) {
    if (p.nrt == 2) return launch_prefill<D, MODE, 2>(args, groups, st);
  }
  return hipErrorInvalidValue;
}

// Two waves per SIMD up to head_dim 256 (the registers), one at 512 (the
// registers and 147 KB of LDS).
int32_t prefill_groups_per_cu(const PoolGeometry &g) { return g.D >= 512 ? 1 : 2; }

hipError_t launch_attn_prefill(const PoolGeometry &g, int32_t layer, const AttnLaunch &a, const AttnPlan &p,
                               hipStream_t st) {
  if (p.waves < 1) return hipErrorInvalidValue;
  if (p.token_split != 1 || p.rows_per_group != 16 * p.nrt || (int64_t)p.row_groups * p.rows_per_group < p.NR)
    return hipErrorInvalidValue;
  const int64_t groups = (p.row_groups + p.group_waves - 1) / p.group_waves;
  if ((int64_t)p.waves * g.Hkv * groups > INT32_MAX) return hipErrorInvalidValue;
  const AttnArgs args = make_attn_args(g, layer, a, p);
  switch (g.D) {
    case 64:
      return g.mode == MODE_REF ? launch_prefill_dm<64, MODE_REF>(args, p, st)
                                : launch_prefill_dm<64, MODE_AFFINE>(args, p, st);
    case 128:
      return g.mode == MODE_REF ? launch_prefill_dm<128, MODE_REF>(args, p, st)
                                : launch_prefill_dm<128, MODE_AFFINE>(args, p, st);
    case 256:
      return g.mode == MODE_REF ? launch_prefill_dm<256, MODE_REF>(args, p, st)
                                : launch_prefill_dm<256, MODE_AFFINE>(args, p, st);
    case 512:
      return g.mode == MODE_REF ? launch_prefill_dm<512, MODE_REF>(args, p, st)
                                : launch_prefill_dm<512, MODE_AFFINE>(args, p, st);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace krill
