// vkv_fdecode.hip -- decode attention (one query token per row) over dense
// float K/V: the MLXFast SDPA of KVCacheSimple / RotatingKVCache decode
// steps (sdpa_vector.h:15-177, MLXFast.swift:173-218).
//
// Semantics as the generic attention kernel's MLXFast mode: queries scaled
// in fp32, scores and the probability-weighted sum in fp32, masked keys
// skipped (a bool mask) or offset (an additive f32 mask), an empty row
// yields zeros; split partials are merged by attn_combine_kernel as
// sdpa_vector_2pass_2 merges them (sdpa_vector.h:320-394).
//
// bf16 / f16 K/V (fdecode16_kernel).  A workgroup of 8 waves owns a (row, kv
// head, head group, token part) and deals its part to the waves in steps of
// 16 tokens:
//   * scores on matrix cores, S^T (16 tokens x 16 columns, the group's REP <=
//     8 heads) = K (A operands: lane (m, g) loads dims 32 s + 8 g .. + 7 of
//     token m, 16 bytes straight from memory) . Q^T (B operands: the raw
//     queries in registers), one 16x16x32 MFMA per 32 dims; the fp32 scores
//     are then scaled (the reference scales the queries first: the same fp32
//     arithmetic up to summation order);
//   * online softmax in the lanes that hold a head's scores, the running max
//     refreshed only when a score exceeds it by kTau (one ballot a step), the
//     sum kept per lane until the end, the probabilities through LDS;
//   * values on the vector ALUs (at REP <= 8 heads about one FMA a byte):
//     lanes own 16-byte runs of a value row, D / 8 lanes a row, so every load
//     instruction reads whole rows; the lanes that share a run sum their
//     tokens at the end.
// A step's keys are loaded while the step before is in its softmax and
// values, its values while it is in its scores: the operand registers are
// reloaded as soon as they are used, so a wave always has loads in flight
// and still fits 128 registers (four waves a SIMD).  Loads are buffer loads
// with the step's base in scalar registers and the rows that exist as the
// bound: rows past the end read as zeros without traffic, and a lane's
// addresses are two 32-bit offsets.  K/V may be dense (strided slices of a
// cache) or float pages behind a block table, rows of unequal length.
//
// Bound: HBM on large launches, the chain launch -> queries and first rows ->
// merge on small ones.  Measured against one-wave workgroups that loaded a
// 32-token step and then computed on it, with a merge launch behind (us a
// call): 8 x 6001 tokens, 8/32 heads x 128 (197 MB) 52.1 -> 37.7 (5.2 TB/s);
// 4 x 1024 tokens, 8/16 heads x 256 (34 MB) 15.8 -> 11.8; one row of 512 tokens
// 10.0 -> 9.3; pages of 16 rows of 128-4096 tokens (159 MB, the generic kernel
// before) 214 -> 39.
//
// Split merge.  The waves merge in LDS (sdpa_vector.h:320-394).  Parts
// merge inside the launch: the workgroup stores its (o, max, sum) with
// device-coherent stores (relaxed agent-scope atomics, which write through to
// the level every XCD reads), waits for them and counts itself in on a
// per-(row, kv head, head group) counter; the workgroup that counts last
// reads the parts back with device-coherent loads, merges them, writes the
// output and zeroes the counter for the next launch.  No fence writes back
// or invalidates an L2.  Without counters (the no-allocation entry point) the
// partials go to attn_combine_kernel.
//
// f32 K/V (fdecode_kernel): one wave per workgroup and token part, steps of
// 32 tokens, lanes t and t + 32 on token t, each scoring half of its row
// against the queries in LDS; parts merge as above or in
// attn_combine_kernel.
#include <algorithm>
#include <type_traits>

#include "vkv_device.h"
#include <hip/hip_ext.h>
#include "vkv_internal.h"

namespace vkv {

namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(1))) const u32x4_t g_u32x4_t;

// 16x16x32 MFMA on 16-bit operands of the cache dtype
template <int DT>
__device__ __forceinline__ f32x4_t mfma16(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
  if constexpr (DT == kF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Tokens per step: two lanes per token, each scoring half of the dims.
constexpr int kStep = 32;

// 16 loaded bytes -> VEC floats
template <int DT>
__device__ __forceinline__ void unpack16(const u32x4_t& w, float* out) {
  if constexpr (DT == kF32) {
#pragma unroll
    for (int e = 0; e < 4; e++) out[e] = __uint_as_float(w[e]);
  } else if constexpr (DT == kBF16) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      out[2 * e] = __uint_as_float(w[e] << 16);
      out[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      out[2 * e] = f16_to_f32(static_cast<uint16_t>(w[e] & 0xFFFFu));
      out[2 * e + 1] = f16_to_f32(static_cast<uint16_t>(w[e] >> 16));
    }
  }
}

// Cross-lane moves without an LDS round trip where one exists: DPP inside
// rows of 16 lanes, the swizzle for partners 8 and 16 lanes away (within
// 32), the half swap for partners 32 lanes away.
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, true));
}
template <int M>  // the value of lane (lane ^ M), M = 8 or 16
__device__ __forceinline__ float swz_xor(float x) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x1F | (M << 10)));
}
// v + the value of lane (lane ^ 32), added in that order
__device__ __forceinline__ float add_xor32(float v) {
  float lo = v, hi = v;
  // lo's upper half <- hi's lower half: lo = the lower half's values in both
  // halves, hi = the upper half's
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
  return lo + hi;
}

// Maximum / sum within each half-wave of 32 lanes: pairs 1 and 2 apart
// (quad permutes), then each lane with its mirror in 8 and in 16 lanes (the
// partners hold equal values by then, so the mirror acts as a butterfly),
// then 16 apart.
__device__ __forceinline__ float half_maxf(float x) {
  x = fmaxf(x, dpp_mov<0xB1>(x));
  x = fmaxf(x, dpp_mov<0x4E>(x));
  x = fmaxf(x, dpp_mov<0x141>(x));
  x = fmaxf(x, dpp_mov<0x140>(x));
  return fmaxf(x, swz_xor<16>(x));
}
__device__ __forceinline__ float half_sumf(float x) {
  x += dpp_mov<0xB1>(x);
  x += dpp_mov<0x4E>(x);
  x += dpp_mov<0x141>(x);
  x += dpp_mov<0x140>(x);
  return x + swz_xor<16>(x);
}

// Orders a wave's LDS writes before its other lanes' reads (the LDS data
// of a workgroup of several waves is per wave, so no workgroup barrier).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// The in-launch merge of a (row, kv head, head group)'s parts
// (sdpa_vector.h:320-394), by the part that counted in last: the partials
// come back through device-coherent loads; all 64 lanes take D / 64 dims of
// a head each and issue every part's loads of the head together, one round
// trip per head.
template <int D, int REP>
__device__ __forceinline__ void fdecode_merge_rows(const AttnArgs& a, int64_t b, int h0, int nh,
                                                   int lane) {
  using E = Elem<kF32>;
  constexpr int DPL = D / 64;  // dims per lane: 1, 2 or 4
  constexpr int kMaxP = 32;    // parts per round trip
  for (int r = 0; r < nh; r++) {
    const int h = h0 + r;
    const int64_t rh = b * a.Hq + h;
    const float* mlp = a.ws_ml + rh * a.n_parts * 2;
    const float* wo = a.ws_o + rh * a.n_parts * D + DPL * lane;
    float M = -3.402823466e38f, den = 0.0f, acc[DPL];
#pragma unroll
    for (int e = 0; e < DPL; e++) acc[e] = 0.0f;
    for (int c = 0; c < a.n_parts; c += kMaxP) {
      float mj[kMaxP], lj[kMaxP], vj[kMaxP][DPL];
#pragma unroll
      for (int j = 0; j < kMaxP; j++) {
        const int pp = min(c + j, a.n_parts - 1);  // (clamped slots are selected away)
        const uint64_t w = __hip_atomic_load(reinterpret_cast<const uint64_t*>(mlp) + pp,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        mj[j] = __uint_as_float(static_cast<uint32_t>(w));
        lj[j] = __uint_as_float(static_cast<uint32_t>(w >> 32));
        const float* src = wo + static_cast<int64_t>(pp) * D;
        if constexpr (DPL == 1) {
          vj[j][0] = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
#pragma unroll
          for (int e = 0; e < DPL / 2; e++) {
            const uint64_t x = __hip_atomic_load(reinterpret_cast<const uint64_t*>(src) + e,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            vj[j][2 * e] = __uint_as_float(static_cast<uint32_t>(x));
            vj[j][2 * e + 1] = __uint_as_float(static_cast<uint32_t>(x >> 32));
          }
        }
      }
      float Mc = M;
#pragma unroll
      for (int j = 0; j < kMaxP; j++)
        if (c + j < a.n_parts) Mc = fmaxf(Mc, mj[j]);
      const float rsc = __expf(M - Mc);
      den *= rsc;
#pragma unroll
      for (int e = 0; e < DPL; e++) acc[e] *= rsc;
      M = Mc;
#pragma unroll
      for (int j = 0; j < kMaxP; j++) {
        if (c + j < a.n_parts) {
          const float w = __expf(mj[j] - M);
          den += w * lj[j];
#pragma unroll
          for (int e = 0; e < DPL; e++) acc[e] = fmaf(w, vj[j][e], acc[e]);
        }
      }
    }
    typename E::T* out = static_cast<typename E::T*>(a.out) + b * a.o_sb + h * a.o_sh + DPL * lane;
#pragma unroll
    for (int e = 0; e < DPL; e++) out[e] = E::from_f32(den > 0.0f ? acc[e] / den : 0.0f);
  }
}

template <int D, int REP>
__global__ void __launch_bounds__(64) fdecode_kernel(AttnArgs a, int rep_total) {
  constexpr int DT = kF32;  // 16-bit K/V take fdecode16_kernel
  using E = Elem<DT>;
  constexpr int VEC = 16 / E::kBytes;  // elements per 16-byte load
  constexpr int KL = D / VEC;          // loads per key row
  constexpr int LPR = D / VEC;         // lanes per value row
  constexpr int RPI = 64 / LPR;        // value rows per load instruction
  static_assert(LPR <= 64 && 64 % LPR == 0, "value rows must tile a wave");
  static_assert(KL % 2 == 0 && kStep % RPI == 0, "key rows split in two halves, value rows tile a step");
  __shared__ float qs[REP][D];
  __shared__ float ps[REP][kStep];
  const int lane = threadIdx.x & 63;
  const int part = static_cast<int>(blockIdx.x);
  const int n_hg = (rep_total + REP - 1) / REP;
  const int hk = blockIdx.y / n_hg, hg = blockIdx.y % n_hg;
  const int64_t b = blockIdx.z;
  const int h0 = hk * rep_total + hg * REP;
  const int nh = min(REP, rep_total - hg * REP);
  const int64_t T = a.kv.T;
  const int64_t t_begin = static_cast<int64_t>(part) * a.part_tokens;
  const int64_t t_end = min<int64_t>(T, t_begin + a.part_tokens);

  const uint8_t* kbase = a.kv.kc.ptr + b * a.kv.kc.sb + hk * a.kv.kc.sh;
  const uint8_t* vbase = a.kv.vc.ptr + b * a.kv.vc.sb + hk * a.kv.vc.sh;
  const int64_t kst = a.kv.kc.st, vst = a.kv.vc.st;
  const int rs = lane / LPR, dg = lane % LPR;  // value phase: row slot, 16-byte run
  const int tok = lane & (kStep - 1), half = lane / kStep;
  // Loads of a step (t0): lanes tok and tok + 32 read half of key row
  // t0 + tok each; value row slot rs takes tokens t0 + rs, t0 + rs + RPI, ...
  // (rows past the end read the range's first row; their scores are masked
  // and their probabilities are 0).  All of a step's loads go out before
  // its first use, so a step waits for one memory round trip, not one per
  // group of loads; f32 at 256 dims would need more than 160 registers for
  // both sets, so there the value loads go out after the scores.  (Loading
  // the next step during this one's arithmetic keeps both sets live across
  // the loop: measured slower, fewer waves fit.)
  constexpr int NV = kStep / RPI;
  constexpr bool kVEarly = (KL / 2 + NV) * 4 <= 160;
  u32x4_t kw[KL / 2], vw[NV];
  // a cache update's deferred token: row new_t comes from its source rows,
  // and the range that holds it writes it into the cache (one head group)
  const int64_t new_t = a.has_new ? a.new_t : -1;
  const bool writes_new = new_t >= t_begin && new_t < t_end && hg == 0;
  const uint8_t* nkrow = a.has_new ? a.nk_ptr + b * a.nk_sb + hk * a.nk_sh : kbase;
  const uint8_t* nvrow = a.has_new ? a.nv_ptr + b * a.nv_sb + hk * a.nv_sh : vbase;
  auto load_k = [&](int64_t t0) __attribute__((always_inline)) {
    const int64_t t = t0 + tok < t_end ? t0 + tok : t_begin;
    const uint8_t* krow = (t == new_t ? nkrow : kbase + t * kst) + 16 * (KL / 2) * half;
#pragma unroll
    for (int c = 0; c < KL / 2; c++) kw[c] = *(g_u32x4_t*)(krow + 16 * c);
  };
  auto load_v = [&](int64_t t0) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int64_t tv = t0 + rs + RPI * k < t_end ? t0 + rs + RPI * k : t_begin;
      vw[k] = *(g_u32x4_t*)((tv == new_t ? nvrow : vbase + tv * vst) + 16 * dg);
    }
  };

  // the queries (times the scale) go to LDS; their loads go out first,
  // then the first step's key and value loads, so both latencies overlap
  constexpr int NQ = REP * D / 64;
  float qv[NQ];
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    const int i = lane + 64 * j, r = i / D, d = i % D;
    qv[j] = r < nh ? E::load(static_cast<const typename E::T*>(a.q) + b * a.q_sb + (h0 + r) * a.q_sh + d)
                   : 0.0f;
  }
  if (t_begin < t_end) {
    load_k(t_begin);
    if constexpr (kVEarly) load_v(t_begin);
  }
#pragma unroll
  for (int j = 0; j < NQ; j++) {
    const int i = lane + 64 * j;
    qs[i / D][i % D] = qv[j] * a.scale;
  }
  __syncthreads();
  float m[REP], l[REP], o[REP][VEC];
#pragma unroll
  for (int r = 0; r < REP; r++) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
    // an attention sink is one more logit with a zero value row, counted
    // once per row: the running max starts at it with sum 1
    // (sdpa_vector.h:93-96, :257-260)
    if (a.sinks && part == 0 && r < nh) {
      m[r] = load_as<DT>(a.sinks, a.sinks_dtype, h0 + r);
      l[r] = 1.0f;
    }
#pragma unroll
    for (int e = 0; e < VEC; e++) o[r][e] = 0.0f;
  }

  for (int64_t t0 = t_begin; t0 < t_end; t0 += kStep) {
    // ---- scores: lanes tok and tok + 32 own token t0 + tok, each half of
    // its dims
    const int64_t t = t0 + tok;
    const bool valid = t < t_end;
    if (t0 != t_begin) {
      load_k(t0);
      if constexpr (kVEarly) load_v(t0);
    }
    float s[REP];
#pragma unroll
    for (int r = 0; r < REP; r++) s[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < KL / 2; c++) {
      float kv[VEC];
      unpack16<DT>(kw[c], kv);
      const int q0 = VEC * (c + (KL / 2) * half);
#pragma unroll
      for (int r = 0; r < REP; r++)
#pragma unroll
        for (int e = 0; e < VEC; e++) s[r] = fmaf(qs[r][q0 + e], kv[e], s[r]);
    }
    if constexpr (!kVEarly) load_v(t0);
    if (writes_new && t == new_t) {  // the new token's key row into the cache
      uint8_t* dst = const_cast<uint8_t*>(kbase) + new_t * kst + 16 * (KL / 2) * half;
#pragma unroll
      for (int c = 0; c < KL / 2; c++) *reinterpret_cast<u32x4_t*>(dst + 16 * c) = kw[c];
    }

#pragma unroll
    for (int r = 0; r < REP; r++) s[r] = add_xor32(s[r]);
#pragma unroll
    for (int r = 0; r < REP; r++) {
      bool vis = valid && r < nh;
      if (vis && a.mask_mode >= 2) {
        const int64_t mo = b * a.m_sb + (h0 + r) * a.m_sh + t * a.m_st;
        if (a.mask_mode == 2) {
          vis = static_cast<const uint8_t*>(a.mask)[mo] != 0;
        } else {
          // the mask in the query dtype; keys below its lowest finite
          // value are skipped (sdpa_vector.h:105-121)
          const float add = load_as<DT>(a.mask, a.mask_dtype, mo);
          vis = add >= -E::kMax;
          s[r] += add;
        }
      }
      s[r] = vis ? s[r] : -INFINITY;
    }
    // ---- online softmax per head (sdpa_vector.h:116-131)
#pragma unroll
    for (int r = 0; r < REP; r++) {
      const float mn = fmaxf(m[r], half_maxf(s[r]));
      float p = 0.0f, alpha = 1.0f;
      if (mn != -INFINITY) {
        p = s[r] == -INFINITY ? 0.0f : __expf(s[r] - mn);
        alpha = m[r] == -INFINITY ? 0.0f : __expf(m[r] - mn);
      }
      l[r] = l[r] * alpha + half_sumf(p);
      m[r] = mn;
      if (half == 0) ps[r][tok] = p;
#pragma unroll
      for (int e = 0; e < VEC; e++) o[r][e] *= alpha;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const int tt = rs + RPI * k;
      if (writes_new && t0 + tt == new_t)  // the new token's value row into the cache
        *reinterpret_cast<u32x4_t*>(const_cast<uint8_t*>(vbase) + new_t * vst + 16 * dg) = vw[k];
      float vv[VEC];
      unpack16<DT>(vw[k], vv);
#pragma unroll
      for (int r = 0; r < REP; r++) {
        const float p = ps[r][tt];
#pragma unroll
        for (int e = 0; e < VEC; e++) o[r][e] = fmaf(p, vv[e], o[r][e]);
      }
    }
    __syncthreads();
  }

  // the row slots of a run hold disjoint tokens: sum them
#pragma unroll
  for (int r = 0; r < REP; r++)
#pragma unroll
    for (int e = 0; e < VEC; e++) {
      if constexpr (LPR <= 8) o[r][e] += swz_xor<8>(o[r][e]);
      if constexpr (LPR <= 16) o[r][e] += swz_xor<16>(o[r][e]);
      if constexpr (LPR <= 32) o[r][e] = add_xor32(o[r][e]);
    }
  const bool merge_here = a.n_parts > 1 && a.counters;
  if (rs == 0) {
#pragma unroll
    for (int r = 0; r < REP; r++) {
      if (r >= nh) break;
      const int h = h0 + r;
      const int d0 = VEC * dg;
      if (a.n_parts == 1) {
        const float inv = l[r] > 0.0f ? 1.0f / l[r] : 0.0f;
        typename E::T* out = static_cast<typename E::T*>(a.out) + b * a.o_sb + h * a.o_sh + d0;
#pragma unroll
        for (int e = 0; e < VEC; e++) out[e] = E::from_f32(o[r][e] * inv);
      } else if (merge_here) {
        const int64_t base = (b * a.Hq + h) * a.n_parts + part;
        uint64_t* wo = reinterpret_cast<uint64_t*>(a.ws_o + base * D + d0);
#pragma unroll
        for (int e = 0; e < VEC / 2; e++)
          __hip_atomic_store(wo + e, pack_f2(o[r][2 * e], o[r][2 * e + 1]), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        if (dg == 0)
          __hip_atomic_store(reinterpret_cast<uint64_t*>(a.ws_ml + base * 2), pack_f2(m[r], l[r]),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        const int64_t base = (b * a.Hq + h) * a.n_parts + part;
        float* wo = a.ws_o + base * D + d0;
#pragma unroll
        for (int e = 0; e < VEC; e++) wo[e] = o[r][e];
        if (dg == 0) {
          a.ws_ml[base * 2] = m[r];
          a.ws_ml[base * 2 + 1] = l[r];
        }
      }
    }
  }
  if (!merge_here) return;
  // this part's partial stores are complete before it counts itself in
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  uint32_t* cnt = a.counters + (b * a.Hkv + hk) * n_hg + hg;
  uint32_t before = 0;
  if (lane == 0) before = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  before = __builtin_amdgcn_readfirstlane(before);
  if (before != static_cast<uint32_t>(a.n_parts - 1)) return;
  // the last part merges every part of the group's heads, then zeroes the
  // counter for the next launch
  if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  fdecode_merge_rows<D, REP>(a, b, h0, nh, lane);
}

// ------------------------------------------------------ 16-bit K/V

constexpr int kWaves16 = 8;    // waves of a workgroup
constexpr int kStep16 = 16;    // tokens of a wave's step
constexpr float kTau = 8.0f;   // the running max lags a score by at most this
constexpr float kLowest = -3.402823466e38f;
constexpr int kCus = 256;            // compute units of the device
constexpr int kOnePart = 32768;      // tokens x dims of a row that is one part
constexpr int kShortRow = 768;       // tokens of a row whose heads may be split

typedef __attribute__((address_space(4))) const int32_t c_i32_t;

// Registers a wave: 128 (four waves a SIMD, two workgroups a CU) where the
// operands of a step (D / 4 registers), the queries and the accumulators
// (8 a head) leave room for the rest; else two waves a SIMD.
template <int D, int REP>
constexpr int fd16_waves_per_simd() {
  return D / 4 + D / 8 + 9 * REP <= 92 ? 4 : 2;
}

// Dense rows, dense rows under an array mask (its loads and 64-bit offsets
// would cost the plain loop registers), or float pages.
enum { kDense = 0, kMasked = 1, kPages = 2 };

template <int DT, int D, int REP, int MODE>
__global__ void __launch_bounds__(64 * kWaves16)
    __attribute__((amdgpu_waves_per_eu(fd16_waves_per_simd<D, REP>())))
    fdecode16_kernel(const AttnArgs a, int rep_total) {
  using E = Elem<DT>;
  constexpr bool PAGED = MODE == kPages;
  constexpr int KS = D / 32;         // 32-dim K steps of a key row
  constexpr int LPR = D / 8;         // lanes per value row
  constexpr int NV = LPR / 4;        // value rows a lane reads a step (16 rows over 64 / LPR slots)
  constexpr int NW = kWaves16;
  __shared__ __attribute__((aligned(16))) float ps_g[NW][REP][kStep16];
  __shared__ __attribute__((aligned(16))) float mo_g[NW][REP][D];
  __shared__ float ml_g[NW][REP][2];
  __shared__ int last_s;

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = blockIdx.x;
  const int n_hg = (rep_total + REP - 1) / REP;
  const int hk = blockIdx.y / n_hg, hg = blockIdx.y - hk * n_hg;
  const int64_t b = blockIdx.z;
  const int h0 = hk * rep_total + hg * REP;
  const int nh = min(REP, rep_total - hg * REP);
  const int T = a.kv.seq_lens ? min(a.kv.seq_lens[b], a.kv.T) : a.kv.T;
  const int t_begin = part * a.part_tokens;
  const int t_end = min(T, t_begin + a.part_tokens);
  // parts of this row (its own length's); the others have nothing to add
  const int np = T > 0 ? (T + a.part_tokens - 1) / a.part_tokens : 1;
  const bool merge_here = a.counters != nullptr;
  if (part >= np && (merge_here || a.n_parts == 1)) return;
  const int nsteps = t_end > t_begin ? (t_end - t_begin + kStep16 - 1) / kStep16 : 0;

  const int mrow = lane & 15, kgrp = lane >> 4;  // scores: token / head column, dims 8 kgrp
  const int rs = lane / LPR, dg = lane % LPR;    // values: row slot (tokens NV rs ..), run
  const uint8_t* kbase = a.kv.kc.ptr + hk * a.kv.kc.sh + (PAGED ? 0 : b * a.kv.kc.sb);
  const uint8_t* vbase = a.kv.vc.ptr + hk * a.kv.vc.sh + (PAGED ? 0 : b * a.kv.vc.sb);
  const int kst = static_cast<int>(a.kv.kc.st), vst = static_cast<int>(a.kv.vc.st);
  // (the whole offset in the vector operand: the bound is checked against
  // it less the scalar offset, which would wrap on an empty buffer)
  const int koff = mrow * kst + 16 * kgrp, voff = NV * rs * vst + 16 * dg;
  const int bs = a.kv.block_size;
  // page of token t: the quotient by multiplication, in scalar registers (a
  // division would hold vector registers through the loop)
  auto page = [&](int t) __attribute__((always_inline)) {
    return static_cast<int>(__umulhi(static_cast<uint32_t>(t), a.bs_mul) >> a.bs_sh);
  };
  c_i32_t* table = (c_i32_t*)(a.kv.table + (PAGED ? b * a.kv.table_stride : 0));
  // step i of the part: its first token and (paged) block; steps past the
  // end read nothing
  auto block_of = [&](int i) __attribute__((always_inline)) {
    const int t = t_begin + kStep16 * min(i, max(nsteps - 1, 0));
    return nsteps > 0 ? table[page(t)] : 0;
  };
  u32x4_t kw[KS], vw[NV];
  // non-temporal where one workgroup reads a long row (at REP = 8 further head
  // groups may; below, only those of short rows): 8 x 6001 bf16 tokens 40.2 ->
  // 37.6 us
  constexpr int kNt = REP < 8 ? 2 : 0;
  // K (or V) rows of step i, as a buffer whose end is the last row's
  auto rows_of = [&](const uint8_t* base, const Comp& c, int st, int i, int blk) __attribute__((always_inline)) {
    const int t0 = t_begin + kStep16 * i;
    const int n = min(t_end - t0, kStep16);
    const uint8_t* p = base;
    if constexpr (PAGED)
      p += blk * c.sb + static_cast<int64_t>(t0 - page(t0) * bs) * st;
    else
      p += static_cast<int64_t>(t0) * st;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0,
                                             n > 0 ? (n - 1) * st + 2 * D : 0, 0x00020000);
  };
  auto load_k = [&](int i, int blk) __attribute__((always_inline)) {
    const auto r = rows_of(kbase, a.kv.kc, kst, i, blk);
#pragma unroll
    for (int s = 0; s < KS; s++) kw[s] = __builtin_amdgcn_raw_buffer_load_b128(r, koff + 64 * s, 0, kNt);
  };
  auto load_v = [&](int i, int blk) __attribute__((always_inline)) {
    const auto r = rows_of(vbase, a.kv.vc, vst, i, blk);
#pragma unroll
    for (int k = 0; k < NV; k++) vw[k] = __builtin_amdgcn_raw_buffer_load_b128(r, voff + k * vst, 0, kNt);
  };

  int blk = 0, blk_next = 0;
  if constexpr (PAGED) {
    blk = block_of(wv);
    blk_next = block_of(wv + NW);
  }
  // the queries, B operands: head mrow, dims 32 s + 8 kgrp .. + 7
  u32x4_t qb[KS];
  {
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + b * a.q_sb +
                         static_cast<int64_t>(h0 + min(mrow, nh - 1)) * a.q_sh + 8 * kgrp;
    if (((reinterpret_cast<uintptr_t>(a.q) >> 1 | a.q_sb | a.q_sh) & 7) == 0) {
#pragma unroll
      for (int s = 0; s < KS; s++) qb[s] = *(g_u32x4_t*)(qp + 32 * s);
    } else {
#pragma unroll 1
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int s = 0; s < KS; s++) {
          const uint32_t w = qp[32 * s + 2 * e] | static_cast<uint32_t>(qp[32 * s + 2 * e + 1]) << 16;
#pragma unroll
          for (int x = 0; x < 4; x++) qb[s][x] = x == e ? w : qb[s][x];
        }
    }
  }
  load_k(wv, blk);
  load_v(wv, blk);
#pragma unroll
  for (int s = 0; s < KS; s++)
#pragma unroll
    for (int e = 0; e < 4; e++) qb[s][e] = mrow < nh ? qb[s][e] : 0u;

  float m_own = kLowest, l_own = 0.0f;  // this lane's head: running max, its share of the sum
  // an attention sink is one more logit with a zero value row, counted once
  // per row: the running max starts at it with sum 1 (sdpa_vector.h:93-96)
  if (a.sinks && part == 0 && wv == 0 && mrow < nh) {
    m_own = sink_start(load_as<DT>(a.sinks, a.sinks_dtype, h0 + mrow), kLowest);
    l_own = kgrp == 0 ? 1.0f : 0.0f;
  }
  float o[REP][8];
#pragma unroll
  for (int r = 0; r < REP; r++)
#pragma unroll
    for (int e = 0; e < 8; e++) o[r][e] = 0.0f;

  for (int i = wv; i < nsteps; i += NW) {
    const int t0 = t_begin + kStep16 * i;
    if (!PAGED && a.has_new && a.new_t >= t0 && a.new_t < t0 + kStep16) {
      // a cache update's deferred token: its rows come from the caller's
      // arrays, and the first head group writes them into the cache
      const int at = static_cast<int>(a.new_t) - t0;
      const uint8_t* nk = a.nk_ptr + b * a.nk_sb + hk * a.nk_sh + 16 * kgrp;
      const uint8_t* nv = a.nv_ptr + b * a.nv_sb + hk * a.nv_sh + 16 * dg;
      uint8_t* ck = const_cast<uint8_t*>(kbase) + a.new_t * kst + 16 * kgrp;
      uint8_t* cv = const_cast<uint8_t*>(vbase) + a.new_t * vst + 16 * dg;
      if (mrow == at) {
#pragma unroll
        for (int s = 0; s < KS; s++) {
          kw[s] = *(g_u32x4_t*)(nk + 64 * s);
          if (hg == 0) *reinterpret_cast<u32x4_t*>(ck + 64 * s) = kw[s];
        }
      }
#pragma unroll
      for (int k = 0; k < NV; k++) {
        if (NV * rs + k == at) {
          vw[k] = *(g_u32x4_t*)nv;
          if (hg == 0) *reinterpret_cast<u32x4_t*>(cv) = vw[k];
        }
      }
    }
    // ---- scores: lane (mrow, kgrp) ends with head mrow, tokens t0 + 4 kgrp + j
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; s++) acc = mfma16<DT>(kw[s], qb[s], acc);
    load_k(i + NW, blk_next);
    float x[4], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int t = t0 + 4 * kgrp + j;
      float v = acc[j] * a.scale;
      bool vis = t < t_end && mrow < nh;
      if (MODE == kMasked && vis) {
        const int64_t mo = b * a.m_sb + (h0 + mrow) * a.m_sh + t * a.m_st;
        if (a.mask_mode == 2) {
          vis = static_cast<const uint8_t*>(a.mask)[mo] != 0;
        } else {
          // the mask in the query dtype; keys below its lowest finite value
          // are skipped (sdpa_vector.h:105-121)
          const float add = load_as<DT>(a.mask, a.mask_dtype, mo);
          vis = add >= -E::kMax;
          v += add;
        }
      }
      x[j] = vis ? v : -INFINITY;
      mx = fmaxf(mx, x[j]);
    }
    if (__builtin_amdgcn_ballot_w64(mx > m_own + kTau)) {
      // the head's new max over its four lanes, the accumulators rescaled
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mn = fmaxf(m_own, mx);
      const float al = __expf(m_own - mn);
      m_own = mn;
      l_own *= al;
#pragma unroll
      for (int r = 0; r < REP; r++) {
        const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(al), r));
#pragma unroll
        for (int e = 0; e < 8; e++) o[r][e] *= f;
      }
    }
    f32x4_t p;
#pragma unroll
    for (int j = 0; j < 4; j++) p[j] = __expf(x[j] - m_own);
    l_own += (p[0] + p[1]) + (p[2] + p[3]);
    if (mrow < REP) *reinterpret_cast<f32x4_t*>(&ps_g[wv][mrow][4 * kgrp]) = p;
    wave_lds_sync();
    // ---- values: this lane's rows are tokens t0 + NV rs .. + NV
    float pr[REP][NV];
#pragma unroll
    for (int r = 0; r < REP; r++)
#pragma unroll
      for (int k = 0; k < NV; k++) pr[r][k] = ps_g[wv][r][NV * rs + k];
#pragma unroll
    for (int k = 0; k < NV; k++) {
      float vv[8];
      unpack16<DT>(vw[k], vv);
#pragma unroll
      for (int r = 0; r < REP; r++)
#pragma unroll
        for (int e = 0; e < 8; e++) o[r][e] = fmaf(pr[r][k], vv[e], o[r][e]);
    }
    load_v(i + NW, blk_next);
    if constexpr (PAGED) blk_next = block_of(i + 2 * NW);
    wave_lds_sync();
  }

  // ---- the row slots of a run hold disjoint tokens: sum them
#pragma unroll
  for (int r = 0; r < REP; r++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      if constexpr (LPR <= 8) o[r][e] += swz_xor<8>(o[r][e]);
      if constexpr (LPR <= 16) o[r][e] += swz_xor<16>(o[r][e]);
      if constexpr (LPR <= 32) o[r][e] = add_xor32(o[r][e]);
    }
  l_own += __shfl_xor(l_own, 16);
  l_own += __shfl_xor(l_own, 32);
  // ---- the waves merge in LDS, then every thread takes two dims of a head
  if (rs == 0) {
#pragma unroll
    for (int r = 0; r < REP; r++)
#pragma unroll
      for (int e = 0; e < 8; e += 4)
        *reinterpret_cast<f32x4_t*>(&mo_g[wv][r][8 * dg + e]) =
            f32x4_t{o[r][e], o[r][e + 1], o[r][e + 2], o[r][e + 3]};
  }
  if (lane < REP) {
    ml_g[wv][lane][0] = m_own;
    ml_g[wv][lane][1] = l_own;
  }
  __syncthreads();
  const int pairs = nh * (D / 2);
  for (int idx = threadIdx.x; idx < pairs; idx += 64 * NW) {
    const int r = idx / (D / 2), d = 2 * (idx % (D / 2)), h = h0 + r;
    float M = kLowest;
#pragma unroll
    for (int w = 0; w < NW; w++) M = fmaxf(M, ml_g[w][r][0]);
    float den = 0.0f, a0 = 0.0f, a1 = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const float f = __expf(ml_g[w][r][0] - M);
      den = fmaf(f, ml_g[w][r][1], den);
      a0 = fmaf(f, mo_g[w][r][d], a0);
      a1 = fmaf(f, mo_g[w][r][d + 1], a1);
    }
    if (a.n_parts == 1 || (merge_here && np == 1)) {
      // (an empty row's sum is 0; a NaN one is NaN in the output)
      typename E::T* out = static_cast<typename E::T*>(a.out) + b * a.o_sb + h * a.o_sh + d;
      out[0] = E::from_f32(den != 0.0f ? a0 / den : 0.0f);
      out[1] = E::from_f32(den != 0.0f ? a1 / den : 0.0f);
    } else {
      const int64_t slot = (b * a.Hq + h) * a.n_parts + part;
      uint64_t* wo = reinterpret_cast<uint64_t*>(a.ws_o + slot * D + d);
      uint64_t* wm = reinterpret_cast<uint64_t*>(a.ws_ml + slot * 2);
      __hip_atomic_store(wo, pack_f2(a0, a1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0)
        __hip_atomic_store(wm, pack_f2(M, den), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (a.n_parts == 1 || !merge_here || np == 1) return;
  // ---- the parts merge in the workgroup that counts in last; every wave's
  // partial stores are complete before the count
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint32_t* cnt = a.counters + (b * a.Hkv + hk) * n_hg + hg;
  if (threadIdx.x == 0)
    last_s = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             static_cast<uint32_t>(np - 1);
  __syncthreads();
  if (!last_s) return;
  if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int idx = threadIdx.x; idx < pairs; idx += 64 * NW) {
    const int r = idx / (D / 2), d = 2 * (idx % (D / 2)), h = h0 + r;
    const int64_t slot = (b * a.Hq + h) * a.n_parts;
    const uint64_t* wo = reinterpret_cast<const uint64_t*>(a.ws_o + slot * D + d);
    const uint64_t* wm = reinterpret_cast<const uint64_t*>(a.ws_ml + slot * 2);
    float M = kLowest, den = 0.0f, a0 = 0.0f, a1 = 0.0f;
    constexpr int kP = 8;  // parts a round trip
    for (int c = 0; c < np; c += kP) {
      uint64_t ml[kP], ov[kP];
#pragma unroll
      for (int j = 0; j < kP; j++) {
        const int q = min(c + j, np - 1);  // (clamped parts are selected away)
        ml[j] = __hip_atomic_load(wm + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ov[j] = __hip_atomic_load(wo + static_cast<int64_t>(q) * (D / 2), __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT);
      }
      float Mc = M;
#pragma unroll
      for (int j = 0; j < kP; j++)
        if (c + j < np) Mc = fmaxf(Mc, __uint_as_float(static_cast<uint32_t>(ml[j])));
      const float f0 = __expf(M - Mc);
      den *= f0;
      a0 *= f0;
      a1 *= f0;
      M = Mc;
#pragma unroll
      for (int j = 0; j < kP; j++) {
        if (c + j < np) {
          const float f = __expf(__uint_as_float(static_cast<uint32_t>(ml[j])) - M);
          den = fmaf(f, __uint_as_float(static_cast<uint32_t>(ml[j] >> 32)), den);
          a0 = fmaf(f, __uint_as_float(static_cast<uint32_t>(ov[j])), a0);
          a1 = fmaf(f, __uint_as_float(static_cast<uint32_t>(ov[j] >> 32)), a1);
        }
      }
    }
    typename E::T* out = static_cast<typename E::T*>(a.out) + b * a.o_sb + h * a.o_sh + d;
    out[0] = E::from_f32(den != 0.0f ? a0 / den : 0.0f);
    out[1] = E::from_f32(den != 0.0f ? a1 / den : 0.0f);
  }
}

// All of a kv head's query heads, up to 8, so that each key row is read once
// for them; of the sizes 1, 2, 4 and 8 that the kernels are built for.
int fd_most_heads(int Hq, int Hkv) {
  const int rep = Hq / Hkv;
  return rep <= 1 ? 1 : rep <= 2 ? 2 : rep <= 4 ? 4 : 8;
}

template <int DT, int D, int R>
void launch_r(const AttnArgs& a, int64_t rows, int rep, int n_hg, hipStream_t st) {
  const TimedLaunch tl = timing_prepare(kTimeFDecode);
  const dim3 grid(a.n_parts, a.Hkv * n_hg, static_cast<unsigned>(rows));
  if constexpr (DT == kF32) {
    hipExtLaunchKernelGGL((fdecode_kernel<D, R>), grid, dim3(64), 0, st, tl.start, tl.stop, 0, a,
                          rep);
  } else {
    auto run = [&](auto M_) {
      hipExtLaunchKernelGGL((fdecode16_kernel<DT, D, R, decltype(M_)::value>), grid,
                            dim3(64 * kWaves16), 0, st, tl.start, tl.stop, 0, a, rep);
    };
    if (a.kv.table) run(std::integral_constant<int, kPages>{});
    else if (a.mask_mode >= 2) run(std::integral_constant<int, kMasked>{});
    else run(std::integral_constant<int, kDense>{});
  }
  VKV_HIP(hipGetLastError());
  timing_commit(tl);
}

template <int DT, int D>
void launch_d(const AttnArgs& a, int64_t rows, hipStream_t st) {
  const int rep = a.Hq / a.Hkv, R = a.group_heads;
  const int n_hg = (rep + R - 1) / R;
  if (R == 1) launch_r<DT, D, 1>(a, rows, rep, n_hg, st);
  else if (R == 2) launch_r<DT, D, 2>(a, rows, rep, n_hg, st);
  else if (R == 4) launch_r<DT, D, 4>(a, rows, rep, n_hg, st);
  else launch_r<DT, D, 8>(a, rows, rep, n_hg, st);
}

template <int DT>
void launch_dt(const AttnArgs& a, int64_t rows, hipStream_t st) {
  if (a.D == 64) launch_d<DT, 64>(a, rows, st);
  else if (a.D == 128) launch_d<DT, 128>(a, rows, st);
  else launch_d<DT, 256>(a, rows, st);
}

}  // namespace

bool fdecode_supported(int dtype, int bits, bool qsem, const AttnArgs& a) {
  if (bits != 0 || qsem || a.L != 1 || a.kv.qfmt) return false;
  if (a.D != a.Dv || (a.D != 64 && a.D != 128 && a.D != 256)) return false;
  if (a.Hq % a.Hkv) return false;
  if (a.mask_mode < 0 || a.mask_mode > 3) return false;
  const int rep = a.Hq / a.Hkv;
  if (dtype == kF32) {
    // dense rows of one length; f32 rows at 128 dims with more than 4 query
    // heads a kv head, or at 256 dims with more than 2, need more registers
    // than a wave has (the step's f32 key and value rows beside the group's
    // accumulators): those variants spill hundreds of registers to scratch
    // and ran 1.9-4.7x slower than the generic kernel, which therefore takes
    // them
    if (a.kv.table || a.kv.seq_lens) return false;
    if ((a.D == 128 && rep > 4) || (a.D == 256 && rep > 2)) return false;
  } else {
    // a step's rows lie in one page, and within a 32-bit buffer
    if (a.kv.table && (a.kv.block_size < kStep16 || a.kv.block_size % kStep16 || a.mask_mode >= 2))
      return false;
    for (const Comp* c : {&a.kv.kc, &a.kv.vc})
      if (c->st < 2 * a.D || c->st >= (int64_t{1} << 26)) return false;
    if (static_cast<int64_t>(a.Hkv) * rep > 65535) return false;
  }
  // 16-byte loads of key and value rows
  auto al = [](const void* p, int64_t s0, int64_t s1, int64_t s2) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0 && s0 % 16 == 0 && s1 % 16 == 0 && s2 % 16 == 0;
  };
  return al(a.kv.kc.ptr, a.kv.kc.sb, a.kv.kc.sh, a.kv.kc.st) &&
         al(a.kv.vc.ptr, a.kv.vc.sb, a.kv.vc.sh, a.kv.vc.st);
}

FdecodePlan fdecode_plan(int dtype, int64_t rows, int Hq, int Hkv, int64_t T, int D, int waves) {
  FdecodePlan p;
  p.heads = fd_most_heads(Hq, Hkv);
  int64_t parts, step;
  if (dtype == kF32) {
    // about `waves` (default 2048) one-wave workgroups
    step = kStep;
    parts = (waves > 0 ? waves : 2048) / std::max<int64_t>(1, rows * Hkv);
    parts = std::min<int64_t>(parts, (T + step - 1) / step);
  } else {
    step = kStep16;
    constexpr int kRound = kStep16 * kWaves16;  // tokens of one step of every wave
    auto groups = [&](int R) { return rows * Hkv * ((Hq / Hkv + R - 1) / R); };
    if (waves > 0) {
      parts = std::min<int64_t>(waves / kWaves16 / std::max<int64_t>(1, groups(p.heads)),
                                (T + kRound - 1) / kRound);
    } else {
      // Rows up to 64 KB of keys are one part: the merge of parts through
      // device memory costs ~2 us, more than a wave's second and third step
      // (us of GPU a call in a graph, one part / parts of 128 tokens: 32/8
      // heads x 128, 200 tokens 6.3 / 7.3, 300 6.7 / 7.4, 512 9.1 / 7.6; x 64,
      // 512 tokens 6.9 / 6.9; 8 rows of 256 x 64 6.1 / 7.5).
      const bool one = T * D <= kOnePart;
      const int64_t most = one ? 1 : (T + kRound - 1) / kRound;
      // Heads are dealt to more workgroups while that leaves the launch
      // within a workgroup a CU: each then holds fewer accumulators and ends
      // sooner, and the rows it reads again come from the L2 (64/8 heads x
      // 128, in two or more heads a workgroup / the rule's: 100 tokens 7.3 / 4.5,
      // 300 9.8 / 7.1, 512 9.9 / 7.6; 32/8 x 64, 100 tokens 5.2 / 3.9).  At
      // 1500 tokens (32/8 x 64: 8.2 with four heads, 8.6 with two) and at 256
      // dims (16/8 heads, 700 tokens 8.7 / 9.0) it does not pay.
      if (T <= kShortRow && D <= 128)
        for (int R = 1; R < p.heads; R *= 2)
          if (groups(R) * most <= kCus) {
            p.heads = R;
            break;
          }
      // Two workgroups a CU, each of at least one step a wave: 1024 and 2048
      // workgroups are slower, a workgroup's fixed chain being ~5 us.  256 are
      // as fast or faster on long rows (us a call at 256, 512, 1024, 2048
      // workgroups: 8 x 6001 tokens, 32/8 heads x 128, 35.8, 38.3, 43.4, 54.2; 8
      // x 2000 of 64/8 heads 17.3, 23.6, 41.2, 41.2; pages of 16 rows to 4096
      // tokens 39.3, 39.6, 44.4, 55.1); rows of very unequal length were not
      // measured at 256.
      parts = std::min<int64_t>(512 / std::max<int64_t>(1, groups(p.heads)), most);
    }
  }
  parts = std::max<int64_t>(1, parts);
  int64_t pt = (T + parts - 1) / parts;
  pt = std::max<int64_t>(step, (pt + step - 1) / step * step);
  p.part_tokens = static_cast<int32_t>(pt);
  p.n_parts = static_cast<int32_t>(std::max<int64_t>(1, (T + pt - 1) / pt));
  return p;
}

void launch_fdecode(int dtype, const AttnArgs& a, int64_t rows, hipStream_t st) {
  if (rows <= 0) return;
  // a causal mask leaves one query token every key
  AttnArgs b = a;
  if (b.mask_mode == 1) b.mask_mode = 0;
  if (b.kv.table) {
    // t / block_size = mulhi(t, bs_mul) >> bs_sh for t < 2^31
    int sh = 0;
    while ((int64_t{1} << sh) < b.kv.block_size) sh++;
    b.bs_mul = static_cast<uint32_t>((uint64_t{1} << (31 + sh)) / b.kv.block_size + 1);
    b.bs_sh = sh - 1;
  }
  switch (dtype) {
    case kF32: launch_dt<kF32>(b, rows, st); break;
    case kF16: launch_dt<kF16>(b, rows, st); break;
    case kBF16: launch_dt<kBF16>(b, rows, st); break;
    default: throw Error("unsupported dtype");
  }
  if (b.n_parts > 1 && !b.counters) launch_attn_combine(dtype, b, rows, st);
}

int fdecode_counter_count(int Hq, int Hkv, int heads) {
  return Hkv * ((Hq / Hkv + heads - 1) / heads);
}

bool fdecode_merge_here(int dtype, int n_parts, int Dv, int heads) {
  if (dtype != kF32) return true;  // the whole workgroup merges
  // partial floats the last part of a head group reads back
  constexpr int64_t kMaxMergeFloats = 12288;
  return static_cast<int64_t>(n_parts) * Dv * heads <= kMaxMergeFloats;
}

}  // namespace vkv
