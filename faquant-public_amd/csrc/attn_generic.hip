// General-shape HiF4 flash attention on gfx950: the simulator's recurrence
// (src/faquant/simulated_flash_attention.py:457-909) for the shapes and operand types the
// headline kernel (hif4_attention.hip: head_dim 128, key tiles of 128, bf16 operands) does not
// take: any head_dim up to 256, any key tile up to 1024 keys, and fp32, bf16 or fp16 Q/K/V
// (the reference multiplies unquantized fp32 operands as they are, sfa:723-724, 848-850).
// Quantized operands (sfa:592-619) come in already quantized.
//
// Per query row and key tile [k0, k0 + W), in the reference's order of operations:
//   s = fp32(dot(q, k) * scale)                          sfa:723-724
//   s = tanh(s / softcap) * softcap                      sfa:725-727 (softcap > 0)
//   s = s + mask  |  s = -inf outside the row's keys     sfa:730-776
//   m' = max(m, max_k s);  prev = exp(m - m') (0 for m = -inf)          sfa:778-787
//   P = exp(s - m') (0 for s = -inf)                     sfa:788-792
//   P^ = HiF4 QDQ of P in 64-key groups from the tile start, zero-padded (sfa:793-806,
//        292-338), with the reference's E6M2 scale and micro exponents (pquant8)
//   l = prev l + sum(P^ or P);  acc = prev acc + P^ V   sfa:826-850
// and O = acc / max(l, FLT_MIN) where l > 0, else 0 (sfa:871-876).  The products are exact
// and summed in fp32 by the matrix cores: bf16 and fp16 operands have exact fp32 products,
// P^ has at most six significant bits (exact in bf16, pairs with bf16 V on the bf16 MFMA),
// and everything else (fp32 Q, K or V, unquantized P, mixed types) goes through the fp32
// MFMA.  P^ is the reference quantizer applied to this kernel's P, bit for bit.
//
// Work decomposition: a 256-thread workgroup of four waves, 32 query rows each: hpw query
// heads of one KV head times 4 / hpw blocks of 32 positions, so K and V staged in LDS serve
// 128 rows.  Key tiles are processed in groups of up to 128 keys (two 64-key HiF4 groups);
// a tile of at most 128 keys is one group, whose scores stay in registers between the
// maximum and P.  A longer tile runs over its groups twice: once for the maximum (K only),
// once for P (the scores computed again, the same bits), so that no tile size needs room
// for its scores.
//
// MFMA layout (32x32 shapes; lane l, n = l % 32, half = l / 32): scores are S^T = K Q^T
// with the A row m of key block kb being key 32 ((m >> 2) & 1) + 16 kb + 4 (m >> 3) + (m & 3)
// of its 64-key group, so lane (n, half) holds keys 32 half + 16 kb + i (register i) of
// query row n: every 8-key micro group is lane-local and in order, and the 64-key group is
// the two halves of a row.  PV is O^T = V^T P^T: the B operand slots 8 half + t of k-chunk c
// are keys 32 half + 8 c + t, this lane's own P; the bf16 A operand comes from natural V rows
// by transposing LDS reads (ds_read_b64_tr_b16), the fp32 one by plain reads.  fp32 products
// run v_mfma_f32_32x32x2_f32 with k slot `half` holding dim 8 u + 4 half + e (scores) or key
// 32 half + i (PV).
//
// What bounds it, and what this form measured (MI355X, causal, Qwen3-8B heads, 4096 tokens,
// head_dim 128, bf16 HiF4 operands, HIP events; in brackets the fp32 VALU kernel it replaced,
// which was bound by LDS bandwidth): key tiles of 64 0.297 ms (6.82), 128 0.270 ms (6.53), 256
// 0.348 ms (8.12: the scores twice), 16 1.11 ms (10.9: mostly padding); head_dim 64 / 256 with
// tiles of 128 0.210 / 0.640 ms (4.56 / 18.1).  There the exponent and the P quantizer's
// VALU work and the bf16 MFMAs take turns, as in the headline kernel, and two workgroups per
// CU cover each other's loads and barriers (K/V go through registers into one LDS stage).
// fp32 operands run at the fp32 MFMA's rate (1/16 of bf16's): 16 heads, 2000 tokens, tiles of
// 128: 0.28-0.43 ms (1.13-1.16).
#include <cfloat>

#include "attn_generic.h"
#include "hif4_attention.hip"

namespace faq {
namespace {

// exp(x) for x <= 0, within 2 ulp of e^x: 2^t with t = RN(x log2 e), corrected by the
// rounding error of t.  -inf, NaN (inf - inf: a masked or overflowed score) and anything
// below -200 give 0; exactly 1 at 0.  Results below 2^-126 are flushed to 0.
__device__ __forceinline__ float gen_exp(float x) {
  const float y = fmaxf(x, -200.0f);
  const float t = y * 1.44269502162933349609375f;
  float e = __builtin_fmaf(y, 1.44269502162933349609375f, -t);
  e = __builtin_fmaf(y, 1.92596299e-8f, e);
  const float p = __builtin_amdgcn_exp2f(t);
  return __builtin_fmaf(p, e * 0.693147182464599609375f, p);
}

// Whether e^x rounds to a subnormal, which gen_exp flushes and the probe counts as positive
// (e^x > 2^-150, half the smallest subnormal).
__device__ __forceinline__ bool gen_exp_flushed(float x) { return x > -103.972084f && gen_exp(x) == 0.0f; }

__device__ __forceinline__ float gen_load(const void* p, int dt, int64_t i) {
  if (dt == 0) return static_cast<const float*>(p)[i];
  if (dt == 1) return bf16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
  return __half2float(static_cast<const __half*>(p)[i]);
}

// Four consecutive values from element i (16- or 8-byte aligned, see gen_vec_ok).
__device__ __forceinline__ float4 gen_load4(const void* p, int dt, int64_t i) {
  if (dt == 0) return *reinterpret_cast<const float4*>(static_cast<const float*>(p) + i);
  const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
  if (dt == 1)
    return make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xFFFF0000u), __uint_as_float(w.y << 16),
                       __uint_as_float(w.y & 0xFFFF0000u));
  return make_float4(__half2float(__ushort_as_half(static_cast<unsigned short>(w.x & 0xFFFFu))),
                     __half2float(__ushort_as_half(static_cast<unsigned short>(w.x >> 16))),
                     __half2float(__ushort_as_half(static_cast<unsigned short>(w.y & 0xFFFFu))),
                     __half2float(__ushort_as_half(static_cast<unsigned short>(w.y >> 16))));
}

// Whether rows of D elements at element offset `base` and row stride sl can be read in units
// of `vw` elements of `es` bytes, each unit aligned to its size.
__device__ __forceinline__ bool gen_vec_ok(const void* p, int64_t base, int64_t sl, int D, int vw, int es) {
  return D % vw == 0 && base % vw == 0 && sl % vw == 0 &&
         (reinterpret_cast<uintptr_t>(p) & static_cast<uintptr_t>(vw * es - 1)) == 0;
}

// kRows rows (key j at element base + j sl) into LDS at `pitch` bytes, kDp dims each, dims
// past D and rows past nk as zeros.  16-bit rows are copied as they are (the MFMA takes
// them), fp32 rows are converted from any dtype.
template <int kDp, bool kF32, int kPitch>
__device__ __forceinline__ void gen_stage(uint8_t* dst, const void* src, int dt, int64_t base, int64_t sl, int nk, int D,
                                          bool vec, int tid, int rows) {
  constexpr int vw = kF32 ? 4 : 8;       // values per 16-byte LDS unit
  constexpr int upr = kDp / vw;          // units per row
  constexpr int per = 64 * upr / 256;    // units per thread and 64 rows
  if (vec) {
    for (int r0 = 0; r0 < rows; r0 += 64) {
      uint4 w[per];
#pragma unroll
      for (int i = 0; i < per; ++i) {
        const int u = tid + 256 * i, j = r0 + u / upr, d0 = (u % upr) * vw;
        w[i] = make_uint4(0u, 0u, 0u, 0u);
        if (j < nk && d0 < D) {
          const int64_t at = base + static_cast<int64_t>(j) * sl + d0;
          if constexpr (kF32) {
            const float4 f = gen_load4(src, dt, at);
            w[i] = make_uint4(__float_as_uint(f.x), __float_as_uint(f.y), __float_as_uint(f.z), __float_as_uint(f.w));
          } else {
            w[i] = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(src) + at);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < per; ++i) {
        const int u = tid + 256 * i;
        *reinterpret_cast<uint4*>(dst + (r0 + u / upr) * kPitch + (u % upr) * 16) = w[i];
      }
    }
  } else {
    for (int idx = tid; idx < rows * kDp; idx += 256) {
      const int j = idx / kDp, d = idx % kDp;
      const bool in = j < nk && d < D;
      const int64_t at = base + static_cast<int64_t>(j) * sl + d;
      if constexpr (kF32) {
        *reinterpret_cast<float*>(dst + j * kPitch + 4 * d) = in ? gen_load(src, dt, at) : 0.0f;
      } else {
        *reinterpret_cast<uint16_t*>(dst + j * kPitch + 2 * d) = in ? static_cast<const uint16_t*>(src)[at] : 0;
      }
    }
  }
}

__device__ __forceinline__ floatx16 mfma32_f32(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// pquant_setup and pquant8 (hif4_attention.hip) with the level form as three wave-uniform
// numbers instead of three copies of the code, the same values:
//   123: 4 2^e2 = med3(hm, 4, 8), 4K = med3(x, 4 2^e2, 16)
//   12:  x = the larger x of the two 4-key groups, e2 = 0, 4K = med3(x, 4, 8)
//   13:  e2 = 0, 4K = med3(x, 4, 8)
struct GenLevels {
  float div_rec, e_max, k4_max;
  bool pair;
};

__device__ __forceinline__ GenLevels gen_levels(int lv) {
  return {lv == 123 ? divisor_reciprocal<123>() : divisor_reciprocal<12>(), lv == 123 ? 8.0f : 4.0f,
          lv == 123 ? 16.0f : 8.0f, lv == 12};
}

__device__ __forceinline__ PQuant gen_pquant_setup(float m1, const GenLevels& lv) {
  const float s0 = bf16_round_hw(m1 * lv.div_rec);
  uint32_t b = min(max(__float_as_uint(s0), 0x27800000u), 0x47400000u);
  b = (b + 0x000FFFFFu + ((b >> 21) & 1u)) & 0xFFE00000u;
  const float sc = __uint_as_float(b);
  const float rec = bf16_round_hw(__builtin_amdgcn_rcpf(sc));
  return {rec * 4.0f, sc * 0.0625f};
}

__device__ __forceinline__ void gen_pquant8(float* g, const PQuant& q, const GenLevels& lv) {
#pragma unroll
  for (int j = 0; j < 8; ++j) g[j] = g[j] * q.rec4;
  const uint32_t xa = __float_as_uint(floor2(fmaxf(fmaxf(g[0], g[1]), fmaxf(g[2], g[3]))));
  const uint32_t xb = __float_as_uint(floor2(fmaxf(fmaxf(g[4], g[5]), fmaxf(g[6], g[7]))));
  const uint32_t xm = max(xa, xb);
  const float e2 = __builtin_amdgcn_fmed3f(__uint_as_float(xm - 0x00800000u), 4.0f, lv.e_max);
  const float k4a = __builtin_amdgcn_fmed3f(__uint_as_float(lv.pair ? xm : xa), e2, lv.k4_max);
  const float k4b = __builtin_amdgcn_fmed3f(__uint_as_float(lv.pair ? xm : xb), e2, lv.k4_max);
  const float ika = inv_k_of(k4a), ikb = inv_k_of(k4b);
  const float dqa = k4a * q.s16, dqb = k4b * q.s16;  // K s / 4
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    g[j] = fminf(floorf(__builtin_fmaf(g[j], ika, 0.5f)), 7.0f) * dqa;
    g[4 + j] = fminf(floorf(__builtin_fmaf(g[4 + j], ikb, 0.5f)), 7.0f) * dqb;
  }
}

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

// V^T rows 32 mb + m (m the A row), keys 32 half + 8 c + 0..7 of a 64-key group, from
// natural bf16 rows: within each 16-lane group, lane i of ds_read_b64_tr_b16 receives element
// i % 4 of the 8 bytes addressed by lanes 4k + i / 4, k = 0..3.
template <int kPitch>
__device__ __forceinline__ bf16x8 gen_vt_fragment(const uint8_t* v, int lane, int mb, int c) {
  const int g = lane >> 4, jj = lane & 15;
  const uint8_t* p = v + (32 * (g >> 1) + 8 * c + (jj >> 2)) * kPitch + 2 * (32 * mb + 16 * (g & 1) + 4 * (jj & 3));
  const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p));
  const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(p + 4 * kPitch));
  bf16x8 r;
  __builtin_memcpy(&r, &lo, 8);
  __builtin_memcpy(reinterpret_cast<char*>(&r) + 8, &hi, 8);
  return r;
}

// Sum of 16 values as a tree (shorter and rounding less than a chain).
__device__ __forceinline__ float gen_sum16(const floatx16& v) {
  float t[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = v[i] + v[i + 8];
#pragma unroll
  for (int d = 4; d >= 1; d >>= 1)
#pragma unroll
    for (int i = 0; i < d; ++i) t[i] += t[i + d];
  return t[0];
}

// LDS layout: K rows, then V rows, 128 keys each.  K rows have an odd number of 16-byte units
// (conflict-free operand reads: 16 rows distinct mod 16 per pass); bf16 V rows a pitch of
// 64 bytes mod 128 (the four keys of a transposing read in distinct bank quarters).
// Where both do not leave room for two workgroups per CU, V overwrites K (kShare).
template <int DB, int kQK, int kPV>
struct GenShape {
  static constexpr int kDp = 32 * DB;
  static constexpr int kKPitch = kDp * (kQK == 2 ? 4 : 2) + 16;
  static constexpr int kVPitch = kPV == 2 ? kDp * 4 + 16 : (DB % 2 ? 64 * DB : 64 * DB + 64);
  static constexpr bool kShare = 128 * (kKPitch + kVPitch) > 80 * 1024;
  static constexpr int kVOff = kShare ? 0 : 128 * kKPitch;
  static constexpr int kLds = kShare ? 128 * (kKPitch > kVPitch ? kKPitch : kVPitch) : 128 * (kKPitch + kVPitch);
  // registers: Q (kDp / 4 or / 2), scores 64, accumulators 16 DB; two waves per SIMD have 256
  static constexpr int kWaves = DB <= (kQK == 2 || kPV == 2 ? 2 : 4) ? 2 : 1;
};

// kFull: with the softcap, the dense mask and the probe (a.softcap, a.amask, a.diag), whose code
// would cost the plain form its registers.
template <int DB, int kQK, int kPV, bool kFull>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(GenShape<DB, kQK, kPV>::kWaves,
                                                                     GenShape<DB, kQK, kPV>::kWaves)))
void gen_attention_kernel(GenAttnArgs a) {
  typedef GenShape<DB, kQK, kPV> Sh;
  constexpr int kDp = Sh::kDp;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Sh::kLds];
  __shared__ int sh_lo, sh_hi;
  uint8_t* const ks = lds;
  uint8_t* const vs = lds + Sh::kVOff;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n = lane & 31, half = lane >> 5;
  const int D = a.D, T = a.T;

  // item: (head group, position block) of batch entry z, heads fastest (a multiple of 8 head
  // groups keeps each on one XCD), the longest causal position blocks first
  const int G = a.Hq / a.Hkv;
  const int X = a.Hq / a.hpw;
  const int b = blockIdx.z, x = blockIdx.x % X, y = blockIdx.x / X;
  const int hq = x * a.hpw + w % a.hpw;
  const int kvh = (x * a.hpw) / G;
  const int pb = a.causal ? a.n_pblocks - 1 - y : y;
  const int p0w = (pb * (4 / a.hpw) + w / a.hpw) * 32;
  const int pos = p0w + n;
  const bool live = pos < a.Lq;
  const int off = a.Lk - a.Lq;  // bottom-right causal: position p sees keys <= p + off
  const bool ranges = a.row_lo != nullptr;
  const bool dense = kFull && a.amask != nullptr;

  // this row's keys [lo, hi], and the wave's and the workgroup's union
  int lo = a.Lk, hi = -1;
  if (live) {
    lo = 0;
    hi = a.Lk - 1;
    if (ranges) {
      lo = max(0, a.row_lo[static_cast<int64_t>(b) * a.Lq + pos]);
      hi = min(a.Lk - 1, a.row_hi[static_cast<int64_t>(b) * a.Lq + pos]);
    } else if (a.causal && !dense) {
      hi = min(a.Lk - 1, pos + off);
    }
  }
  const bool any = lo <= hi;
  const int lo_w = wave_min_i32(any ? lo : a.Lk), hi_w = wave_max_i32(any ? hi : -1);
  if (tid == 0) {
    sh_lo = a.Lk;
    sh_hi = -1;
  }
  __syncthreads();
  if (lane == 0) {
    atomicMin(&sh_lo, lo_w);
    atomicMax(&sh_hi, hi_w);
  }
  __syncthreads();
  const int wg_lo = __builtin_amdgcn_readfirstlane(sh_lo), wg_hi = __builtin_amdgcn_readfirstlane(sh_hi);
  const int t_lo = wg_lo <= wg_hi ? wg_lo / T : 1;
  const int t_hi = wg_lo <= wg_hi ? wg_hi / T : 0;

  // Q fragment: 16-bit, dims 16 c + 8 half .. + 7; fp32, dims 8 u + 4 half .. + 3
  constexpr int kQN = kQK == 2 ? kDp / 8 : kDp / 16;
  uint4 qf[kQN];
  {
    const int64_t qb = b * a.q_sb + hq * a.q_sh + static_cast<int64_t>(live ? pos : 0) * a.q_sl;
    constexpr int vw = kQK == 2 ? 4 : 8;
    const bool qvec = gen_vec_ok(a.q, b * a.q_sb + hq * a.q_sh, a.q_sl, D, vw, a.q_dt == 0 ? 4 : 2);
#pragma unroll
    for (int c = 0; c < kQN; ++c) {
      const int d0 = (2 * c + half) * vw;
      uint32_t wv[4] = {0u, 0u, 0u, 0u};
      if (live && d0 < D) {
        if constexpr (kQK == 2) {
          float f[4];
          if (qvec) {
            const float4 f4 = gen_load4(a.q, a.q_dt, qb + d0);
            f[0] = f4.x, f[1] = f4.y, f[2] = f4.z, f[3] = f4.w;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) f[i] = d0 + i < D ? gen_load(a.q, a.q_dt, qb + d0 + i) : 0.0f;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) wv[i] = __float_as_uint(f[i]);
        } else {
          const uint16_t* qp = static_cast<const uint16_t*>(a.q) + qb + d0;
          if (qvec) {
            const uint4 q4 = *reinterpret_cast<const uint4*>(qp);
            wv[0] = q4.x, wv[1] = q4.y, wv[2] = q4.z, wv[3] = q4.w;
          } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
              if (d0 + i < D) wv[i >> 1] |= static_cast<uint32_t>(qp[i]) << (16 * (i & 1));
          }
        }
      }
      qf[c] = make_uint4(wv[0], wv[1], wv[2], wv[3]);
    }
  }

  const int64_t kb0 = b * a.k_sb + kvh * a.k_sh, vb0 = b * a.v_sb + kvh * a.v_sh;
  const bool kvec = gen_vec_ok(a.k, kb0, a.k_sl, D, kQK == 2 ? 4 : 8, a.k_dt == 0 ? 4 : 2);
  const bool vvec = gen_vec_ok(a.v, vb0, a.v_sl, D, kPV == 2 ? 4 : 8, a.v_dt == 0 ? 4 : 2);

  floatx16 acc[DB];
#pragma unroll
  for (int mb = 0; mb < DB; ++mb) acc[mb] = floatx16{};
  float m_run = -INFINITY, l_run = 0.0f;
  float dq_run = 0.0f, dp_run = 0.0f, dg_zero = 0.0f, dg_err = 0.0f, dg_ref = 0.0f;
  const bool sum_ph = a.quant_p && a.norm_same;
  const GenLevels lv = gen_levels(a.p_levels);
  const int krow0 = 32 * ((n >> 2) & 1) + 4 * (n >> 3) + (n & 3);

  // Scores sc of the group's 64-key group `sub` (first key base0): scaled, capped, masked.
  auto scores = [&](floatx16 (&sc)[2], int sub, int base0, int tile_end) __attribute__((always_inline)) {
    const uint8_t* kp = ks + (64 * sub + krow0) * Sh::kKPitch + 16 * half;
    sc[0] = floatx16{};
    sc[1] = floatx16{};
    // step st = (dims c = st / 2, key block kb = st % 2); the K unit of step st + kAhead is read
    // before step st's MFMAs, and the scheduling barrier keeps the reads from piling up
    constexpr int kSteps = 2 * kQN, kAhead = kQK == 2 ? 2 : 4;
    uint4 kf[kAhead + 1];
    auto k_unit = [&](int st) __attribute__((always_inline)) {
      return *reinterpret_cast<const uint4*>(kp + (st & 1) * 16 * Sh::kKPitch + 32 * (st >> 1));
    };
#pragma unroll
    for (int st = 0; st < kAhead; ++st) kf[st] = k_unit(st);
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
      if (st + kAhead < kSteps) kf[(st + kAhead) % (kAhead + 1)] = k_unit(st + kAhead);
      const uint4 ku = kf[st % (kAhead + 1)], qu = qf[st >> 1];
      floatx16& sk = sc[st & 1];
      if constexpr (kQK == 0) {
        bf16x8 k8, q8;
        __builtin_memcpy(&k8, &ku, 16);
        __builtin_memcpy(&q8, &qu, 16);
        sk = mfma32(k8, q8, sk);
      } else if constexpr (kQK == 1) {
        f16x8 k8, q8;
        __builtin_memcpy(&k8, &ku, 16);
        __builtin_memcpy(&q8, &qu, 16);
        sk = __builtin_amdgcn_mfma_f32_32x32x16_f16(k8, q8, sk, 0, 0, 0);
      } else {
        sk = mfma32_f32(__uint_as_float(ku.x), __uint_as_float(qu.x), sk);
        sk = mfma32_f32(__uint_as_float(ku.y), __uint_as_float(qu.y), sk);
        sk = mfma32_f32(__uint_as_float(ku.z), __uint_as_float(qu.z), sk);
        sk = mfma32_f32(__uint_as_float(ku.w), __uint_as_float(qu.w), sk);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[kb][i] = sc[kb][i] * a.scale;
    if (kFull && a.softcap > 0.0f) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          // the quotient by softcap: q0 corrected by one fma step
          const float t = sc[kb][i], q0 = t * a.softcap_rec;
          sc[kb][i] =
              softcap_tanh(__builtin_fmaf(__builtin_fmaf(-q0, a.softcap, t), a.softcap_rec, q0)) * a.softcap;
        }
    }
    // this lane's 32 keys from `base`; bit j: key base + j is seen
    const int base = base0 + 32 * half;
    uint32_t see;
    if (dense) {
      see = bit_range32(0, min(tile_end, a.Lk) - 1 - base);
      // (keys past the tile re-read its last column and are masked below)
      const int last = min(tile_end, a.Lk) - 1;
      const float* mr = a.amask + b * a.am_sb + hq * a.am_sh + static_cast<int64_t>(live ? pos : 0) * a.am_sq;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kb][i] = sc[kb][i] + mr[min(base + 16 * kb + i, last)];
    } else {
      see = bit_range32(lo - base, min(hi, tile_end - 1) - base);
      if (ranges && see) {
        // see != 0: base <= hi < Lk, so word base / 32 exists; the next one only where it does
        const uint32_t* kw = a.key_bits + b * a.key_words;
        const int wi = base >> 5, sh = base & 31;
        uint32_t bits = kw[wi] >> sh;
        if (sh && wi + 1 < a.key_words) bits |= kw[wi + 1] << (32 - sh);
        see &= bits;
      }
    }
    if (__ballot(see != ~0u) != 0) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const uint32_t keep = static_cast<uint32_t>(
              __builtin_amdgcn_sbfe(static_cast<int>(see), static_cast<uint32_t>(16 * kb + i), 1u));
          sc[kb][i] = __uint_as_float((__float_as_uint(sc[kb][i]) & keep) | (0xFF800000u & ~keep));
        }
    }
  };
  auto sub_max = [&](const floatx16 (&sc)[2], float mx) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, sc[kb][i]);
    return mx;
  };

  for (int t = t_lo; t <= t_hi; ++t) {
    const int key0 = t * T;
    const int W = min(T, a.Lk - key0);
    const int groups = (W + 127) / 128;
    // a wave whose rows see none of the tile's keys only stages (the same as a tile of -inf;
    // with kShare the wave's work spans barriers, so there every wave takes every tile)
    const bool mine = Sh::kShare || (lo_w <= hi_w && key0 <= hi_w && key0 + W - 1 >= lo_w);
    float m_new = m_run, prev = 1.0f, rowsum = 0.0f, sq = 0.0f, sp = 0.0f;
    // fp32 products: the tile's PV is summed from zero and added to acc once, as the reference
    // adds its per-tile matmul (128 single additions to a long acc would round more)
    floatx16 pv[kPV == 2 ? DB : 1];
    if constexpr (kPV == 2) {
#pragma unroll
      for (int mb = 0; mb < DB; ++mb) pv[mb] = floatx16{};
    }
    if (groups > 1) {
      float mx = -INFINITY;
      for (int g = 0; g < groups; ++g) {
        const int g0 = key0 + 128 * g, nk = min(128, key0 + W - g0);
        __syncthreads();
        gen_stage<kDp, kQK == 2, Sh::kKPitch>(ks, a.k, a.k_dt, kb0 + static_cast<int64_t>(g0) * a.k_sl, a.k_sl, nk, D,
                                              kvec, tid, nk > 64 ? 128 : 64);
        __syncthreads();
        if (mine) {
          floatx16 sc[2];
          scores(sc, 0, g0, key0 + W);
          mx = sub_max(sc, mx);
          if (nk > 64) {
            scores(sc, 1, g0 + 64, key0 + W);
            mx = sub_max(sc, mx);
          }
        }
      }
      m_new = fmaxf(m_run, halves_max(mx));
    }
    for (int g = 0; g < groups; ++g) {
      const int g0 = key0 + 128 * g, nk = min(128, key0 + W - g0);
      const int rows = nk > 64 ? 128 : 64;
      __syncthreads();
      gen_stage<kDp, kQK == 2, Sh::kKPitch>(ks, a.k, a.k_dt, kb0 + static_cast<int64_t>(g0) * a.k_sl, a.k_sl, nk, D,
                                            kvec, tid, rows);
      if (!Sh::kShare)
        gen_stage<kDp, kPV == 2, Sh::kVPitch>(vs, a.v, a.v_dt, vb0 + static_cast<int64_t>(g0) * a.v_sl, a.v_sl, nk, D,
                                              vvec, tid, rows);
      __syncthreads();
      if (mine) {
        floatx16 s[2][2];
        bf16x8 pf[2][4];
        scores(s[0], 0, g0, key0 + W);
        __builtin_amdgcn_sched_barrier(0);
        if (nk > 64) scores(s[1], 1, g0 + 64, key0 + W);
        __builtin_amdgcn_sched_barrier(0);
        if (groups == 1) {
          float mx = sub_max(s[0], -INFINITY);
          if (nk > 64) mx = sub_max(s[1], mx);
          m_new = fmaxf(m_run, halves_max(mx));
        }
        if (g == 0) {
          prev = gen_exp(m_run - m_new);
          if (kPV == 0 && __ballot(prev != 1.0f) != 0) {
#pragma unroll
            for (int mb = 0; mb < DB; ++mb)
#pragma unroll
              for (int i = 0; i < 16; ++i) acc[mb][i] *= prev;
          }
        }
        // ---- P and P^ of each 64-key group, 8 keys at a time
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
          if (sub == 0 || nk > 64) {
            if (kFull && a.diag) {
              // subnormal P has P^ = 0 (the smallest group scale is 2^-48)
#pragma unroll
              for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i) dg_zero += gen_exp_flushed(s[sub][kb][i] - m_new) ? 1.0f : 0.0f;
            }
            float m1 = 0.0f;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                s[sub][kb][i] = gen_exp(s[sub][kb][i] - m_new);
                m1 = fmaxf(m1, s[sub][kb][i]);
              }
            if (!sum_ph) rowsum += gen_sum16(s[sub][0]) + gen_sum16(s[sub][1]);
            if (a.quant_p) {
              const PQuant pq = gen_pquant_setup(halves_max(m1), lv);
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                float pc[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) pc[j] = s[sub][c >> 1][8 * (c & 1) + j];
                gen_pquant8(pc, pq, lv);
                if (kFull && a.diag) {
#pragma unroll
                  for (int j = 0; j < 8; ++j) {
                    const float p = s[sub][c >> 1][8 * (c & 1) + j], d = pc[j] - p;
                    sq += pc[j];
                    sp += p;
                    dg_err = __builtin_fmaf(d, d, dg_err);
                    dg_ref = __builtin_fmaf(p, p, dg_ref);
                    dg_zero += (pc[j] == 0.0f && p > 0.0f) ? 1.0f : 0.0f;
                  }
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) s[sub][c >> 1][8 * (c & 1) + j] = pc[j];
              }
            }
            if (sum_ph) rowsum += gen_sum16(s[sub][0]) + gen_sum16(s[sub][1]);
            if constexpr (kPV == 0) {
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                float pc[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) pc[j] = s[sub][c >> 1][8 * (c & 1) + j];
                pf[sub][c] = pack8<true>(pc);
              }
            }
          }
        }
      if (Sh::kShare) {
        __syncthreads();
        gen_stage<kDp, kPV == 2, Sh::kVPitch>(vs, a.v, a.v_dt, vb0 + static_cast<int64_t>(g0) * a.v_sl, a.v_sl, nk, D,
                                              vvec, tid, rows);
        __syncthreads();
      }
        // ---- O^T += V^T P^T
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
          if (sub == 0 || nk > 64) {
            const uint8_t* vp = vs + 64 * sub * Sh::kVPitch;
            constexpr int kSteps = (kPV == 0 ? 4 : 32) * DB, kAhead = 4;
            if constexpr (kPV == 0) {
              bf16x8 va[kAhead + 1];
#pragma unroll
              for (int st = 0; st < kAhead; ++st) va[st] = gen_vt_fragment<Sh::kVPitch>(vp, lane, st % DB, st / DB);
#pragma unroll
              for (int st = 0; st < kSteps; ++st) {
                if (st + kAhead < kSteps)
                  va[(st + kAhead) % (kAhead + 1)] =
                      gen_vt_fragment<Sh::kVPitch>(vp, lane, (st + kAhead) % DB, (st + kAhead) / DB);
                acc[st % DB] = mfma32(va[st % (kAhead + 1)], pf[sub][st / DB], acc[st % DB]);
                __builtin_amdgcn_sched_barrier(0);
              }
            } else {
              const uint8_t* vl = vp + 32 * half * Sh::kVPitch + 4 * n;
              auto v_at = [&](int st) __attribute__((always_inline)) {
                return *reinterpret_cast<const float*>(vl + (st / DB) * Sh::kVPitch + 128 * (st % DB));
              };
              float va[kAhead + 1];
#pragma unroll
              for (int st = 0; st < kAhead; ++st) va[st] = v_at(st);
#pragma unroll
              for (int st = 0; st < kSteps; ++st) {
                if (st + kAhead < kSteps) va[(st + kAhead) % (kAhead + 1)] = v_at(st + kAhead);
                const int i = st / DB;
                pv[st % DB] = mfma32_f32(va[st % (kAhead + 1)], s[sub][i >> 4][i & 15], pv[st % DB]);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
          }
        }
      }
    }
    if (mine) {
      if constexpr (kPV == 2) {
#pragma unroll
        for (int mb = 0; mb < DB; ++mb)
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[mb][i] = __builtin_fmaf(prev, acc[mb][i], pv[mb][i]);
      }
      l_run = prev * l_run + halves_sum(rowsum);
      if (kFull && a.diag) {
        dq_run = prev * dq_run + halves_sum(sq);
        dp_run = prev * dp_run + halves_sum(sp);
      }
      m_run = m_new;
    }
  }

  if (kFull && a.diag) {
    dg_zero = halves_sum(dg_zero);
    dg_err = halves_sum(dg_err);
    dg_ref = halves_sum(dg_ref);
  }
  if (!live) return;
  const int64_t row = (static_cast<int64_t>(b) * a.Hq + hq) * a.Lq + pos;
  const int64_t ob = b * a.o_sb + hq * a.o_sh + static_cast<int64_t>(pos) * a.o_sl;
  const bool ovec = gen_vec_ok(a.o, b * a.o_sb + hq * a.o_sh, a.o_sl, D, 4, a.o_dt == 0 ? 4 : 2);
  const bool pos_l = l_run > 0.0f;
  const float den = fmaxf(l_run, FLT_MIN);
#pragma unroll
  for (int mb = 0; mb < DB; ++mb)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d0 = 32 * mb + 8 * j + 4 * half;
      if (d0 >= D) continue;
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = pos_l ? acc[mb][4 * j + r] / den : 0.0f;
      if (a.o_dt == 0) {
        float* o = static_cast<float*>(a.o) + ob + d0;
        if (ovec) {
          *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (d0 + r < D) o[r] = v[r];
        }
      } else {
        uint16_t h[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (a.o_dt == 1) {
            const __bf16 hb = static_cast<__bf16>(v[r]);
            __builtin_memcpy(&h[r], &hb, 2);
          } else {
            h[r] = __half_as_ushort(__float2half_rn(v[r]));
          }
        }
        uint16_t* o = static_cast<uint16_t*>(a.o) + ob + d0;
        if (ovec) {
          uint2 w2;
          __builtin_memcpy(&w2, h, 8);
          *reinterpret_cast<uint2*>(o) = w2;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (d0 + r < D) o[r] = h[r];
        }
      }
    }
  if (half == 0) {
    if (a.row_den) a.row_den[row] = l_run;
    if (kFull && a.diag) {
      float* dg = a.diag + row * 5;
      dg[0] = dq_run;
      dg[1] = dp_run;
      dg[2] = dg_zero;
      dg[3] = dg_err;
      dg[4] = dg_ref;
    }
  }
}

}  // namespace

#ifdef FAQ_GEN_FORM  // this object's instantiations: 10 kQK + kPV

template <int DB, int kQK, int kPV>
static void launch_gen_db(const GenAttnArgs& a, dim3 grid, hipStream_t st) {
  if (a.softcap > 0.0f || a.amask || a.diag)
    hipLaunchKernelGGL((gen_attention_kernel<DB, kQK, kPV, true>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((gen_attention_kernel<DB, kQK, kPV, false>), grid, dim3(256), 0, st, a);
}

template <int kQK, int kPV>
void launch_gen_form(const GenAttnArgs& a, dim3 grid, hipStream_t st) {
  if (a.D <= 64) launch_gen_db<2, kQK, kPV>(a, grid, st);
  else if (a.D <= 96) launch_gen_db<3, kQK, kPV>(a, grid, st);
  else if (a.D <= 128) launch_gen_db<4, kQK, kPV>(a, grid, st);
  else if (a.D <= 192) launch_gen_db<6, kQK, kPV>(a, grid, st);
  else launch_gen_db<8, kQK, kPV>(a, grid, st);
}

template void launch_gen_form<FAQ_GEN_FORM / 10, FAQ_GEN_FORM % 10>(const GenAttnArgs&, dim3, hipStream_t);

#else  // the launcher

static void gen_geometry(const GenAttnArgs& a, int& hpw, int64_t& pblocks) {
  const int G = a.Hq / a.Hkv;
  hpw = G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1;
  const int pos = 32 * (4 / hpw);
  pblocks = (static_cast<int64_t>(a.Lq) + pos - 1) / pos;
}

int64_t gen_attention_blocks(const GenAttnArgs& a) {
  int hpw;
  int64_t pblocks;
  gen_geometry(a, hpw, pblocks);
  const int64_t n = pblocks * (a.Hq / hpw);
  return n <= INT32_MAX ? n : -1;
}

void launch_gen_attention(const GenAttnArgs& args, hipStream_t st) {
  GenAttnArgs a = args;
  int64_t pblocks;
  gen_geometry(a, a.hpw, pblocks);
  a.n_pblocks = static_cast<int>(pblocks);
  const dim3 grid(static_cast<unsigned>(gen_attention_blocks(a)), 1, a.B);
  // 16-bit operands of one type have exact products on that type's MFMA; P^ is exact in bf16
  const int qk = a.q_dt == 1 && a.k_dt == 1 ? 0 : a.q_dt == 2 && a.k_dt == 2 ? 1 : 2;
  const int pv = a.quant_p && a.v_dt == 1 ? 0 : 2;
  if (qk == 0 && pv == 0) launch_gen_form<0, 0>(a, grid, st);
  else if (qk == 0) launch_gen_form<0, 2>(a, grid, st);
  else if (qk == 1 && pv == 0) launch_gen_form<1, 0>(a, grid, st);
  else if (qk == 1) launch_gen_form<1, 2>(a, grid, st);
  else if (pv == 0) launch_gen_form<2, 0>(a, grid, st);
  else launch_gen_form<2, 2>(a, grid, st);
}

#endif

}  // namespace faq
