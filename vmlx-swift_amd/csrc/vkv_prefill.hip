// vkv_prefill.hip -- multi-query attention (L >= 2 query tokens per row:
// chunked prefill) over dense float K/V on gfx950 matrix cores.
//
// Semantics: MLXFast.scaledDotProductAttention with no mask, a causal or a
// bool array mask (MLXFast.swift:173-218; causal = query l of L sees keys 0 .. T - L + l,
// with T each row's own length when the rows are ragged: the chunk of a
// continuous batch over a paged pool),
// and quantizedScaledDotProductAttention (KVCache.swift:1909-1997) of the
// quantized caches after their pages are gathered to bf16 (the dequantized
// values the reference's dequantize produces).  Scores and the weighted sum
// accumulate in fp32; the probabilities enter the second contraction as the
// input dtype (bf16 / f16).  Split partials are merged by
// attn_combine_kernel as sdpa_vector_2pass_2 merges them
// (sdpa_vector.h:320-394).
//
// Work layout.  A workgroup of 8 waves (two per SIMD, one workgroup per
// CU) owns a block of 256 query rows of one (row of the batch, kv head) and
// one key range; a query row is one (query head of the group, position),
// position-major.  Wave w owns rows 32w .. 32w + 31.  Each 32-token key tile
// takes two phases: a matrix phase (the scores of the tile, the P.V of the
// tile before) and a softmax phase.  Waves 4..7 run one phase behind waves
// 0..3, so the two waves of a SIMD are in different phases: one wave's MFMAs
// overlap the other's softmax (ping-pong), and the wave in its matrix phase
// issues at the higher priority.  At 256 dims a workgroup barrier ends every
// phase; up to 128 dims a wave reads the tile's V operands in the softmax
// phase before, and one barrier a tile is enough (see the tile loop).
//
// Bound: the matrix rate the card sustains on non-zero data (1.85 PFLOP/s
// dense bf16: 18 ns a 32x32x16 MFMA and SIMD) and the softmax's vector
// instructions, which overlap it in part.  Measured (512-token chunk over
// 4608 4-bit keys, 32 / 8 heads x 128: 24 MFMAs a tile and wave, 36 tiles):
// 67 -> 60 us, of which 31 are the matrix cores', 9 the launch and the
// prologue, 5 the 33 MB of partials; per tile 1.30 us, where the MFMAs alone
// take 0.86 and the softmax alone 0.9.  No variant spills: with the masked
// and the open softmax as two copies in the tail loop it did (24 to 60
// registers), and a scratch reload waits for the tile loads in flight.
//
// Per tile:
//   * K and V tiles (32 rows of D elements each) go HBM -> LDS with
//     global_load_lds_dwordx4 two tiles ahead into four stages (each wave
//     loads one 1 KB piece of each); the per-lane source offsets place each
//     16-byte piece at its swizzled slot, so the tiles are bank-conflict
//     free with no register staging;
//   * scores S^T = K Q^T on v_mfma_f32_32x32x16 (A = key rows from LDS,
//     B = the wave's queries, in registers): lane l holds query row l % 32
//     of its block for tokens 8 (j / 4) + 4 (l / 32) + j % 4, j = 0..15;
//   * online softmax per row in the lane that owns it (the other token half
//     is lane l ^ 32); a rescale of the accumulators only when a row's max
//     grows by more than 2^kTau;
//   * O^T += V^T P^T: B = the lane's own probabilities, which are exactly
//     the B operand of the k-steps of 16 tokens, A = value columns read with
//     the transposing LDS load ds_read_b64_tr_b16.  O^T keeps one query row
//     per lane, so the rescale and the final 1 / sum need no exchange.
//
// LDS tiles (D = 128: 256-byte rows, 16 slots of 16 bytes): key row t holds
// its piece s at slot s ^ (t & 15) (the score reads of 16 consecutive rows
// hit 16 distinct slots); value row t holds piece s at slot s ^ (4 (t & 3))
// (the transposing reads: 4 rows x 32 bytes per 16 lanes, 16 distinct
// slots per 256 bytes).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <utility>

#include "vkv_device.h"
#include "vkv_internal.h"

namespace vkv {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const u32x4_t g_u32x4_t;

constexpr int kTok = 32;      // tokens per key tile
constexpr int kStages = 4;    // K+V tiles in LDS; the open-tile loop is unrolled by it
constexpr int kWaves = 8;     // two per SIMD, one workgroup per CU
constexpr int kThreads = 64 * kWaves;
constexpr float kTau = 8.0f;  // rescale threshold (log2)
constexpr int kMaskChunk = 256;     // tokens a mask-packing workgroup takes
constexpr int kMaxMaskTiles = 2048; // key tiles of one part under an array mask
constexpr float kLog2e = 1.4426950408889634f;

// Layout for head dim D (keys and values).  Every wave owns 32 query rows.
// Up to 128 dims a wave holds all D output dims, so a workgroup covers 8
// row blocks; at 256 dims the two waves of a SIMD own the same 32 rows and
// split the output dims (each computes the full scores), so a workgroup
// covers 4 row blocks.
template <int D>
struct PfCfg {
  static constexpr int kChunks = D / 16;            // K steps of the score MFMA
  static constexpr int kSplit = D == 256 ? 2 : 1;   // waves sharing a row block
  static constexpr int kDBw = D / 32 / kSplit;      // 32-dim output blocks per wave
  static constexpr int kRB = kWaves / kSplit;       // row blocks per workgroup
  static constexpr int kRows = 32 * kRB;            // query rows per workgroup
  static constexpr int kRowB = 2 * D;               // bytes per K / V row
  static constexpr int kTileB = kTok * kRowB;       // bytes per K (or V) tile
  static constexpr int kSlots = D / 8;              // 16-byte pieces per row
  static constexpr int kKLoads = kTileB / 1024;     // 1 KB loads of a K (or V) tile
  static constexpr int kLoads = 2 * kKLoads / kWaves;  // 1 KB loads per wave per tile
  static constexpr bool kAhead = D <= 128;  // V operands read a phase ahead, one barrier a tile
  static_assert(D == 64 || D == 128 || D == 256, "head dims 64, 128, 256");
  static_assert(kLoads >= 1 && kLoads * kWaves == 2 * kKLoads, "loads split evenly");
};
// LDS slot of piece p of key row t is p ^ kswz(t): a score read of 16
// consecutive rows at one piece hits 16 distinct 16-byte bank groups (rows
// of 256 or 512 bytes: t & 15; of 128 bytes, where rows t and t + 1 already
// differ by half the banks: (t / 2) & 7).
template <int D>
__device__ __forceinline__ int kswz(int t) {
  return D == 64 ? (t >> 1) & 7 : t & 15;
}
// value rows: piece p at slot p ^ vswz(t & 3), for the transposing reads
// (4 rows x 32 bytes per 16 lanes)
template <int D>
__device__ __forceinline__ int vswz(int t) {
  return D == 64 ? 2 * ((t >> 1) & 1) : 4 * (t & 3);
}

template <int... Is, class F>
__device__ __forceinline__ void sfor_impl(std::integer_sequence<int, Is...>, F&& f) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void sfor(F&& f) {
  sfor_impl(std::make_integer_sequence<int, N>{}, f);
}

template <int DT>
__device__ __forceinline__ f32x16_t mfma(const u32x4_t& a, const u32x4_t& b, const f32x16_t& c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (DT == kBF16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, f16x2_t));
}

__device__ __forceinline__ float fast_exp2f(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) void*)p));
}
template <class T>
__device__ __forceinline__ __attribute__((address_space(3))) T* lds_ptr(uint32_t a) {
  return reinterpret_cast<__attribute__((address_space(3))) T*>(static_cast<uintptr_t>(a));
}
// 16 bytes per lane from base + voff to LDS lds + 16 * lane; waited for by
// the kernel itself (vmcnt), so the compiler inserts no waits for it.
__device__ __forceinline__ void dma16(const uint8_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, %2" ::"v"(voff), "s"(lds),
               "s"(base)
               : "memory", "m0");
}
// Before every barrier a wave waits for all of its tile loads but the last
// tile's (LOADS), and for its LDS reads.  The scheduling barriers
// keep the compiler from moving any instruction from one phase into the
// other.
// A wave enters a matrix phase at issue priority 1 and a softmax phase at
// 0, so that on a SIMD the MFMAs of the one wave issue back to back and the
// softmax of the other fills the cycles between them.
template <int PRIO, int LOADS>
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_waitcnt lgkmcnt(0)\n\ts_barrier" ::"n"(LOADS) : "memory");
  __builtin_amdgcn_s_setprio(PRIO);
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void tile_wait_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// A value a phase produces is complete before the phase's closing barrier:
// the compiler may otherwise move pure arithmetic (the exponentials, the
// MFMAs) across the barrier into the other phase.
__device__ __forceinline__ void pin(float v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void pin(const u32x4_t& v) { asm volatile("" ::"v"(v)); }
__device__ __forceinline__ void pin(const f32x16_t& v) { asm volatile("" ::"v"(v)); }
// last visible key of a tile relative to its first, clamped to -1 .. kTok
__device__ __forceinline__ int tile_limit(int64_t last) {
  return static_cast<int>(last < -1 ? -1 : (last > kTok ? kTok : last));
}
// max of a value over the two 32-lane halves of the wave
__device__ __forceinline__ float halves_max(float v) {
  float lo = v, hi = v;
  // lo's upper half <- hi's lower half: lo = the lower half's values in both
  // halves, hi = the upper half's
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(lo), "+v"(hi));
  return fmaxf(lo, hi);
}

// 4 bytes per lane from base + voff to LDS lds + 4 * lane, as dma16.
__device__ __forceinline__ void dma4(const void* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, %2" ::"v"(voff), "s"(lds), "s"(base)
               : "memory", "m0");
}

// 16 mask bytes (any non-zero value is true) as 16 bits, byte i in bit i.
__device__ __forceinline__ uint32_t mask_bits16(const u32x4_t& x) {
  uint32_t b = 0;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    // bit 7 of every non-zero byte, then the four gathered by one product
    // (byte k's bit lands at 24 + k; no two partial products share a bit)
    const uint32_t t = ((((x[w] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x[w]) >> 7) & 0x01010101u;
    b |= (t * 0x01020408u >> 24 & 15u) << (4 * w);
  }
  return b;
}

// A bool array mask as one bit per (query row, key), before the attention:
// words[row][T / 32] with the bits past the row's length clear, the class of
// every (row block of the attention kernel, 32-key tile) -- 0: no row sees
// any of it, 2: every row sees all of it, 1: else -- and per (row, 256 keys)
// whether any key is seen.  The attention kernel then skips class-0 tiles,
// runs class-2 tiles without mask work and reads one word per row and tile
// of the others, where the bytes would be 16 loads a lane in the softmax
// phase.  A workgroup takes the rows of one row block x 256 keys, 16 lanes a
// row, 16 bytes a lane.  Latency bound: a [512, 1535] mask (0.8 MB) is 64
// workgroups of two loads a wave and takes 4.7 us; one row a wave with byte
// loads unrolled eight deep (1800 instructions, each fetched once) took 14 us.
__global__ void __launch_bounds__(512) mask_pack_kernel(const AttnArgs a, int rep, int rows_per_wg) {
  __shared__ uint32_t s_or[8], s_and[8];
  const int c = blockIdx.x, rblk = blockIdx.y;
  const int lane = threadIdx.x & 63, sub = threadIdx.x & 15;
  const int nh = a.m_sh ? a.Hkv : 1;
  const int zb = blockIdx.z / nh, zh = blockIdx.z - zb * nh;
  const int T = a.kv.seq_lens ? min(a.kv.seq_lens[zb], a.kv.T) : a.kv.T;
  // the block's positions (rows are position-major), and the heads of each
  const int row0 = rblk * rows_per_wg, row1 = min(a.L * rep, row0 + rows_per_wg) - 1;
  const int p0 = row0 / rep, heads = a.m_sh ? rep : 1;
  const int items = (row1 / rep - p0 + 1) * heads;
  if (threadIdx.x < 8) {
    s_or[threadIdx.x] = 0;
    s_and[threadIdx.x] = ~0u;
  }
  __syncthreads();
  const int t0 = c * kMaskChunk + 16 * sub;  // this lane's 16 keys
  const int left = T - t0;                   // keys of them that exist
  const uint8_t* mz = static_cast<const uint8_t*>(a.mask) + zb * a.m_sb;
#pragma unroll 2
  for (int it = threadIdx.x >> 4; it < items; it += 32) {
    const int dl = heads == 1 ? it : it / heads;
    const int h = zh * rep + it - dl * heads, l = p0 + dl;
    const uint8_t* m = mz + h * a.m_sh + l * a.m_sl;
    uint32_t w = 0;
    if (a.m_st == 1 && T >= 16) {
      // a lane at the row's end reads its last 16 bytes and shifts
      u32x4_t x;
      __builtin_memcpy(&x, m + min(t0, T - 16), 16);
      w = left > 0 ? mask_bits16(x) >> max(16 - left, 0) : 0;
    } else if (left > 0) {
      for (int k = 0; k < min(left, 16); k++) w |= (m[(t0 + k) * a.m_st] ? 1u : 0u) << k;
    }
    // even lanes hold 32 keys: their own 16 and the next lane's
    w |= static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(w, 0xB1, 0xF, 0xF, false)) << 16;
    const int64_t row = zb * a.mw_b + h * a.mw_h + l;
    const uint64_t any = __builtin_amdgcn_ballot_w64(w != 0) >> (lane & 48) & 0xFFFF;
    if (sub == 0) a.mrow[row * (a.mw_words / 8) + c] = any != 0;
    if (!(sub & 1)) {
      a.mw[row * a.mw_words + 8 * c + sub / 2] = w;
      atomicOr(&s_or[sub / 2], w);
      atomicAnd(&s_and[sub / 2], w);
    }
  }
  __syncthreads();
  if (threadIdx.x < 8)
    a.mcls[(static_cast<int64_t>(blockIdx.z) * gridDim.y + rblk) * a.mw_words + 8 * c + threadIdx.x] =
        s_or[threadIdx.x] == 0 ? 0 : s_and[threadIdx.x] == ~0u ? 2 : 1;
}

// QSEM: the quantized-SDPA arithmetic (KVCache.swift:1909-1997): queries
// times the scale rounded to the dtype, rounded again, instead of fp32 scores
// times the scale; scores rounded to the dtype before the softmax.
// ARR: a bool array mask, packed by mask_pack_kernel: the workgroup runs the
// tiles some row of it sees, the wholly visible ones first (the order of the
// keys does not matter to the online softmax), and each wave loads its rows'
// words of a tile beside the tile.  Measured (512-token chunk on a 1024-token
// window, 16/8 heads x 256, 1535 keys): 40 us and 4.3 us for the packing, where
// the generic kernel took 1780 us.
template <int DT, bool QSEM, int D, bool ARR>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
prefill_kernel(const AttnArgs a, int rep) {
  using Cfg = PfCfg<D>;
  constexpr int kChunks = Cfg::kChunks, kDBw = Cfg::kDBw, kRows = Cfg::kRows;
  constexpr int kRowB = Cfg::kRowB, kTileB = Cfg::kTileB;
  constexpr int kLoads = Cfg::kLoads + (ARR ? 1 : 0);  // loads per wave per tile
  constexpr bool HL = QSEM || ARR;  // P as hi + lo
  __shared__ __attribute__((aligned(16))) uint8_t kv[kStages][2][kTileB];  // [stage][K/V]
  // ARR: the mask words of each wave's rows per stage, and the tiles to run
  __shared__ uint32_t mwords[ARR ? kStages : 1][ARR ? kWaves : 1][ARR ? 64 : 1];
  __shared__ uint16_t tlist[ARR ? kMaxMaskTiles : 1];
  __shared__ int tcount[2];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // waves w and w + 4 share a SIMD; group 1 runs one phase behind group 0
  const int grp = wave >> 2;
  // the wave's 32-row block and (at 256 dims) half of the output dims
  const int rb = wave % Cfg::kRB, dh = wave / Cfg::kRB;
  const int lane = tid & 63, l32 = lane & 31, kg = lane >> 5;
  // workgroup id -> (kv head, part, row block, row of the batch), kv head
  // fastest: workgroups are dealt to the 8 XCDs in id order, so with 8 kv
  // heads each XCD serves one head, and that head's K/V, re-read by every
  // row block and part, stays in the XCD's L2
  const int L = a.L;
  const int rblocks = static_cast<int>((static_cast<uint32_t>(L) * rep + kRows - 1) / kRows);
  // parts of this launch: all, or a window part0 .. part0 + parts_run - 1
  const int prun = a.parts_run > 0 ? a.parts_run : a.n_parts;
  int id = blockIdx.x;
  const int hk = id % a.Hkv;
  id /= a.Hkv;
  const int part = a.part0 + id % prun;
  id /= prun;
  const int rblk = id % rblocks;
  const int64_t b = id / rblocks;
  // keys of this row of the batch: its own length when the rows are ragged
  // (query l of a row of length T sees keys up to T - L + l when causal)
  const int64_t T = a.kv.seq_lens ? min<int64_t>(a.kv.seq_lens[b], a.kv.T) : a.kv.T;
  // query rows of (b, hk): below 2^30 (prefill_supported), so that the row
  // arithmetic is 32-bit
  const int nrows = L * rep;
  const int row0 = rblk * kRows;
  // keys of this workgroup: the part's range, and for a causal mask the
  // range its last position can see
  const int rlast = min(nrows, row0 + kRows) - 1;
  int64_t k_end = min<int64_t>(T, static_cast<int64_t>(part + 1) * a.part_tokens);
  // QSEM: a query that sees no key (a ragged row shorter than the chunk)
  // has every score at T's lowest value in the reference (where(mask, s,
  // finfo.min)), i.e. uniform weights over all of the row's keys; a
  // workgroup holding such a query scans them all
  bool some_none = QSEM && a.mask_mode == 1 && T - L + row0 / rep < 0;
  if (a.mask_mode == 1 && !some_none) k_end = min<int64_t>(k_end, T - L + rlast / rep + 1);
  const int64_t k_begin = static_cast<int64_t>(part) * a.part_tokens;
  int ntiles = k_end > k_begin ? static_cast<int>((k_end - k_begin + kTok - 1) / kTok) : 0;
  // tiles that every row of the workgroup sees whole (no mask work)
  int n_open = 0;
  if (!some_none) {
    const int64_t kmin = a.mask_mode == 1 ? T - L + row0 / rep : T - 1;
    const int64_t open = min<int64_t>(kmin, k_end - 1) - k_begin + 1;
    n_open = open > 0 ? static_cast<int>(min<int64_t>(open / kTok, ntiles)) : 0;
  }

  // ---- this lane's query row and its queries: B operand of score step c
  // = dims 16c + 8 kg .. +8
  using E = Elem<DT>;
  const int qrow = row0 + 32 * rb + l32;
  const int qr = min(qrow, nrows - 1);  // (rows past the end repeat the last)
  const int qpos = static_cast<uint32_t>(qr) / static_cast<uint32_t>(rep);
  const int qhead = hk * rep + (qr - qpos * rep);
  bool none = false;   // ARR: the row sees no key at all (QSEM averages V then)
  uint32_t mrow_off = 0;  // ARR: byte offset of the row's mask words
  if constexpr (ARR) {
    const int64_t mr = b * a.mw_b + qhead * a.mw_h + qpos;
    mrow_off = static_cast<uint32_t>(4 * mr * a.mw_words);
    if constexpr (QSEM) {
      // (whole 32-bit words: the row's bytes are padded to 4)
      const int nc = a.mw_words / 8;
      const uint32_t* ra = reinterpret_cast<const uint32_t*>(a.mrow + mr * nc);
      uint32_t any = 0;
      for (int c = 0; c < nc / 4; c++) any |= ra[c];
      none = any == 0;
      some_none = __syncthreads_or(none);
    }
    // the tiles some row sees, the wholly visible ones first
    const int nh = a.m_sh ? a.Hkv : 1;
    const int64_t z = (a.mw_b ? b : 0) * nh + (a.m_sh ? hk : 0);
    const uint8_t* cls = a.mcls + (z * rblocks + rblk) * a.mw_words + k_begin / kTok;
    if (wave == 0) {
      auto cls_at = [&](int t) -> int {
        if (t >= ntiles) return 0;
        const int x = cls[t];
        return QSEM && some_none ? 1 : x;
      };
      int open = 0;
      for (int t0 = 0; t0 < ntiles; t0 += 64)
        open += __popcll(__builtin_amdgcn_ballot_w64(cls_at(t0 + lane) == 2));
      int io = 0, ip = open;
      for (int t0 = 0; t0 < ntiles; t0 += 64) {
        const int x = cls_at(t0 + lane);
        const uint64_t bo = __builtin_amdgcn_ballot_w64(x == 2);
        const uint64_t bp = __builtin_amdgcn_ballot_w64(x == 1);
        const uint64_t below = (uint64_t{1} << lane) - 1;
        if (x == 2) tlist[io + __popcll(bo & below)] = static_cast<uint16_t>(t0 + lane);
        if (x == 1) tlist[ip + __popcll(bp & below)] = static_cast<uint16_t>(t0 + lane);
        io += __popcll(bo);
        ip += __popcll(bp);
      }
      if (lane == 0) {
        tcount[0] = ip;
        tcount[1] = open;
      }
    }
    __syncthreads();
    ntiles = __builtin_amdgcn_readfirstlane(tcount[0]);
    n_open = __builtin_amdgcn_readfirstlane(tcount[1]);
  }
  int64_t kmax;  // last key the row may see
  u32x4_t qf[kChunks];
  {
    kmax = a.mask_mode == 1 ? T - L + qpos : T - 1;
    const typename E::T* qp = static_cast<const typename E::T*>(a.q) + b * a.q_sb +
                              static_cast<int64_t>(qhead) * a.q_sh + qpos * a.q_sl + 8 * kg;
#pragma unroll
    for (int c = 0; c < kChunks; c++) qf[c] = *(const g_u32x4_t*)(qp + 16 * c);
  }
  if constexpr (QSEM) {
    const float st = round_to<DT>(a.scale);
#pragma unroll
    for (int c = 0; c < kChunks; c++)
#pragma unroll
      for (int w = 0; w < 4; w++) {
        const uint32_t x = qf[c][w];
        qf[c][w] = pack2<DT>(E::to_f32(static_cast<typename E::T>(x & 0xFFFFu)) * st,
                             E::to_f32(static_cast<typename E::T>(x >> 16)) * st);
      }
  }
  // the query loads complete before the tile loads start (a compiler wait
  // for them inside the tile loop would also wait for every tile load)
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  const float cl = QSEM ? kLog2e : a.scale * kLog2e;

  f32x16_t o[kDBw];  // output dims 32 (dh kDBw + db) ..
  float m_run = -1e30f;  // finite: a masked score (-inf) gives p = 0
  float l_run = 0.f;
  // an attention sink (MLXFast semantics only) is one more logit with a
  // zero value row, counted once per row (sdpa_vector.h:93-96): the running
  // max (log2 units) starts at it with sum 1
  if (!QSEM && a.sinks && part == 0) {
    m_run = sink_start(load_as<DT>(a.sinks, a.sinks_dtype, qhead) * kLog2e, m_run);
    l_run = kg == 0 ? 1.f : 0.f;  // the two lane halves' sums are added at the end
  }
#pragma unroll
  for (int db = 0; db < kDBw; db++) o[db] = f32x16_t{};

  if (ntiles > 0) {
    // ---- tile loads.  A tile is 2 kKLoads loads of 1 KB (the K tile's,
    // then the V tile's); wave w issues loads w + 8 x.  Lane lam of a load
    // fills LDS slot lam % kSlots of its row (the load covers 1024 / kRowB
    // consecutive rows) with the row's piece (lam % kSlots) ^ swizzle(row).
    // row 0 of the K / V views is token t_base (a window of the keys)
    const uint8_t* kbase = a.kv.kc.ptr + b * a.kv.kc.sb + hk * a.kv.kc.sh;
    const uint8_t* vbase = a.kv.vc.ptr + b * a.kv.vc.sb + hk * a.kv.vc.sh;
    const int64_t kst = a.kv.kc.st, vst = a.kv.vc.st;
    // the lane's row and piece in load x (recomputed where needed: at 256
    // dims four loads' worth would hold registers through the loop)
    auto lrow = [&](int x) __attribute__((always_inline)) {
      return ((wave + kWaves * x) % Cfg::kKLoads) * (1024 / kRowB) + lane / Cfg::kSlots;
    };
    auto lpiece = [&](int x) __attribute__((always_inline)) {
      const int slot = lane % Cfg::kSlots, r = lrow(x);
      return wave + kWaves * x >= Cfg::kKLoads ? slot ^ vswz<D>(r & 3) : slot ^ kswz<D>(r);
    };
    uint32_t loff[Cfg::kLoads];  // offsets within a whole tile (T * stride < 2^31, host-checked)
#pragma unroll
    for (int x = 0; x < Cfg::kLoads; x++) {
      const bool is_v = wave + kWaves * x >= Cfg::kKLoads;  // wave-uniform
      loff[x] = static_cast<uint32_t>(lrow(x) * (is_v ? vst : kst)) + 16 * lpiece(x);
    }
    auto load_tile = [&](int i, int s) __attribute__((always_inline)) {
      const int ti = min(i, ntiles - 1);  // clamped: every wave issues the same loads
      const int64_t t0 =
          k_begin + static_cast<int64_t>(kTok) *
                        (ARR ? __builtin_amdgcn_readfirstlane(tlist[ti]) : ti);
      if constexpr (ARR)
        dma4(a.mw, mrow_off + static_cast<uint32_t>(4 * (t0 / kTok)),
             __builtin_amdgcn_readfirstlane(lds_addr(&mwords[s][wave][0])));
#pragma unroll
      for (int x = 0; x < Cfg::kLoads; x++) {
        const int n = wave + kWaves * x, pn = n % Cfg::kKLoads;
        const bool is_v = n >= Cfg::kKLoads;
        const int64_t st = is_v ? vst : kst;
        uint32_t off = loff[x];
        if (t0 + kTok > T) {
          // rows past the end repeat the last row (masked); t0 < T here
          const int t = min<int64_t>(lrow(x), T - 1 - t0);
          off = static_cast<uint32_t>(t * st) + 16 * lpiece(x);
        }
        // wave-uniform (M0), which the compiler does not see through the select
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_addr(&kv[s][is_v][0]) + 1024 * pn);
        dma16((is_v ? vbase : kbase) + (t0 - a.t_base) * st, off, dst);
      }
    };

    // ---- per-lane LDS addresses
    // score A operand, step c: K row l32, piece 2c + kg at slot (2c + kg) ^ kswz(l32)
    const uint32_t ka = lds_addr(&kv[0][0][0]) + l32 * kRowB;
    const int kx = kswz<D>(l32);
    // value A operand (dim block db, k-step ks, token half hf): lane
    // 16 a4 + 4 e + jj reads V row 16 ks + 8 hf + 4 (a4 / 2) + e, dims
    // 32 db + 16 (a4 % 2) + 4 jj .. +4 = piece 4 db + 2 (a4 % 2) + jj / 2
    const int a4 = lane >> 4, e4 = (lane >> 2) & 3, jj = lane & 3;
    const uint32_t va = lds_addr(&kv[0][1][0]) + (4 * (a4 >> 1) + e4) * kRowB + 8 * (jj & 1);
    const int vpc = 2 * (a4 & 1) + (jj >> 1);  // piece within the 4-piece group
    const int vx = vswz<D>(e4);                // swizzle of rows 4 (a4 / 2) + e (+ 8 hf + 16 ks)

    // HL: P carried as hi + lo (two operands of the dtype, ~16 significant
    // bits in bf16), so the weighted sum keeps fp32-like accuracy (on large
    // value channels of quantized caches; under array masks, whose calls held
    // the probabilities in fp32 on the generic kernel: relative error against
    // 64 bits 1.654e-3 to 1.663e-3 over chunks of 22-512 tokens in bf16, 2.07e-4
    // in f16, the generic kernel's to five digits; 2.3e-3 with one bf16
    // operand); otherwise one operand
    u32x4_t pb[2], pl[2];
    f32x16_t x;
    // the matrix phase: scores of the tile at LDS base kb (K rows) into x
    // and, with PV, O^T += V^T P^T for the tile at LDS base vb (V rows).
    // Every LDS read is issued before the first MFMA, so the MFMAs run
    // back to back instead of each waiting for its operand's read.
    u32x4_t kf[kChunks], vf[kDBw][2];
    auto read_k = [&](uint32_t kb) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < kChunks; c++)
        kf[c] = *lds_ptr<const u32x4_t>(kb + 16 * ((2 * c + kg) ^ kx));
    };
    auto read_v = [&](uint32_t vb) __attribute__((always_inline)) {
#pragma unroll
      for (int db = 0; db < kDBw; db++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          // rows 16 ks + 8 hf + 4 (a4 / 2) + e (row & 3 = e): piece
          // 4 gdb + vpc (gdb = the global dim block) at slot (4 gdb + vpc) ^ vswz(e)
          const uint32_t slot = 16 * ((4 * (dh * kDBw + db) + vpc) ^ vx);
          const uint32_t off0 = (16 * ks) * kRowB + slot;
          const uint32_t off1 = (16 * ks + 8) * kRowB + slot;
          const i16x4_t x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_ptr<i16x4_t>(vb + off0));
          const i16x4_t x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_ptr<i16x4_t>(vb + off1));
          const u32x2_t w0 = __builtin_bit_cast(u32x2_t, x0), w1 = __builtin_bit_cast(u32x2_t, x1);
          vf[db][ks] = u32x4_t{w0[0], w0[1], w1[0], w1[1]};
        }
    };
    auto matrix = [&](uint32_t kb, uint32_t vb, auto PV_) __attribute__((always_inline)) {
      constexpr bool PV = decltype(PV_)::value;
      read_k(kb);
      if constexpr (!Cfg::kAhead && PV) read_v(vb);
      x = f32x16_t{};
      if constexpr (PV) {
        // the score chain (8 dependent MFMAs) interleaved with the P.V
        // MFMAs (one chain per 32-dim block)
        constexpr int kPv = (HL ? 4 : 2) * kDBw;  // P.V MFMAs
        auto pv = [&](auto J) __attribute__((always_inline)) {  // n-th P.V MFMA
          constexpr int n = decltype(J)::value, db = n % kDBw, q = n / kDBw;
          constexpr int ks = HL ? q / 2 : q;  // HL: ks hi, ks lo; else ks
          if constexpr (HL && q % 2 == 1)
            o[db] = mfma<DT>(vf[db][ks], pl[ks], o[db]);
          else
            o[db] = mfma<DT>(vf[db][ks], pb[ks], o[db]);
        };
        // operands read ahead: the first kFirst P.V MFMAs run while the key
        // reads arrive
        constexpr int kFirst = Cfg::kAhead ? kPv / 2 : 0, kRest = kPv - kFirst;
        sfor<kFirst>(pv);
        if constexpr (Cfg::kAhead) __builtin_amdgcn_sched_barrier(0);
        sfor<kChunks>([&](auto C) {
          constexpr int c = decltype(C)::value;
          x = mfma<DT>(kf[c], qf[c], x);
          // the P.V MFMAs spread evenly over the score steps
          sfor<kRest>([&](auto J) {
            constexpr int n = decltype(J)::value;
            if constexpr (n >= c * kRest / kChunks && n < (c + 1) * kRest / kChunks)
              pv(std::integral_constant<int, kFirst + n>{});
          });
        });
        if constexpr (!Cfg::kAhead) {
          // at 256 dims every read at once would not fit the registers:
          // eight rounds of reads, each followed by its share of MFMAs
          sfor<8>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, (kChunks + 4 * kDBw) / 8, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, (kChunks + kPv) / 8, 0);
          });
        }
#pragma unroll
        for (int db = 0; db < kDBw; db++) pin(o[db]);
      } else {
#pragma unroll
        for (int c = 0; c < kChunks; c++) x = mfma<DT>(kf[c], qf[c], x);
        if constexpr (D <= 128) {
          __builtin_amdgcn_sched_group_barrier(0x100, kChunks, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, kChunks, 0);
        } else {
          sfor<4>([&](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, kChunks / 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, kChunks / 4, 0);
          });
        }
      }
      pin(x);
    };
    // softmax of the row over tile i's scores x: the running max and sum,
    // the rescale of o, and the P operands.  EDGE and `masked`: keys past the
    // range or the causal limit of some row are masked
    // (ARR: the mask words of the tile, in its stage)
    auto softmax = [&](int i, bool masked, auto EDGE_) __attribute__((always_inline)) {
      constexpr bool EDGE = decltype(EDGE_)::value;
      const int64_t t0 = k_begin + static_cast<int64_t>(kTok) * i;
      if constexpr (QSEM) {
        // the scores are stored in the dtype (quantizedMM returns T,
        // KVCache.swift:1945-1949) before the mask and the softmax: the
        // packed hardware conversion (round to nearest even), then back
#pragma unroll
        for (int j = 0; j < 16; j += 2) {
          const uint32_t w = pack2<DT>(x[j], x[j + 1]);
          x[j] = E::to_f32(static_cast<typename E::T>(w & 0xFFFFu));
          x[j + 1] = E::to_f32(static_cast<typename E::T>(w >> 16));
        }
      }
      if (EDGE && !masked) {
        // a tile of the tail loop that every row sees whole
      } else if constexpr (EDGE && ARR) {
        uint32_t w = mwords[i % kStages][wave][lane];
        if (QSEM && some_none) {
          // rows that see no key: equal scores (0) on the row's keys
          const int64_t left =
              k_end - k_begin - kTok * static_cast<int64_t>(tlist[i]);  // >= 1
          const uint32_t all = left >= kTok ? ~0u : (1u << left) - 1;
          w = none ? all : w;
#pragma unroll
          for (int j = 0; j < 16; j++) x[j] = none ? 0.0f : x[j];
        }
        w >>= 4 * kg;
#pragma unroll
        for (int j = 0; j < 16; j++) {
          const uint32_t m =
              static_cast<uint32_t>(__builtin_amdgcn_sbfe(w, 8 * (j >> 2) + (j & 3), 1));
          x[j] = __uint_as_float((__float_as_uint(x[j]) & m) | (0xff800000u & ~m));
        }
      } else if constexpr (EDGE) {
        if (QSEM && some_none && __builtin_amdgcn_ballot_w64(kmax < 0)) {
          // rows that see no key: equal scores (0) on the row's keys
          const bool none = kmax < 0;
          const int lim = tile_limit((none ? k_end - 1 : min<int64_t>(kmax, k_end - 1)) - t0);
#pragma unroll
          for (int j = 0; j < 16; j++) {
            if (none) x[j] = 0.0f;
            if (8 * (j >> 2) + 4 * kg + (j & 3) > lim) x[j] = -INFINITY;
          }
        } else {
          const int lim = tile_limit(min<int64_t>(kmax, k_end - 1) - t0);
#pragma unroll
          for (int j = 0; j < 16; j++)
            if (8 * (j >> 2) + 4 * kg + (j & 3) > lim) x[j] = -INFINITY;
        }
      }
      float mx = x[0];
#pragma unroll
      for (int j = 1; j < 16; j++) mx = fmaxf(mx, x[j]);
      mx = halves_max(mx) * cl;  // scale > 0
      if (__builtin_amdgcn_ballot_w64(mx > m_run + kTau)) {
        const float mn = fmaxf(m_run, mx);
        const float al = fast_exp2f(m_run - mn);
        l_run *= al;
#pragma unroll
        for (int db = 0; db < kDBw; db++) o[db] *= al;
        m_run = mn;
      }
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; e++) p[e] = fast_exp2f(fmaf(x[8 * ks + e], cl, -m_run));
        // a sum tree instead of a chain of dependent adds
        l_run += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        pb[ks] = u32x4_t{pack2<DT>(p[0], p[1]), pack2<DT>(p[2], p[3]), pack2<DT>(p[4], p[5]),
                         pack2<DT>(p[6], p[7])};
        if constexpr (HL) {
          float r[8];
#pragma unroll
          for (int w = 0; w < 4; w++) {
            const uint32_t hw = pb[ks][w];
            r[2 * w] = p[2 * w] - E::to_f32(static_cast<typename E::T>(hw & 0xFFFFu));
            r[2 * w + 1] = p[2 * w + 1] - E::to_f32(static_cast<typename E::T>(hw >> 16));
          }
          pl[ks] = u32x4_t{pack2<DT>(r[0], r[1]), pack2<DT>(r[2], r[3]), pack2<DT>(r[4], r[5]),
                           pack2<DT>(r[6], r[7])};
          pin(pl[ks]);
        }
        pin(pb[ks]);
      }
      pin(l_run);
    };

    // ---- the tile loop, in two phases per tile: a matrix phase (scores of
    // tile i, O += V P of tile i - 1) and a softmax phase (tile i).  Group 1
    // runs one phase behind group 0, so on each SIMD one wave's MFMAs overlap
    // the other wave's softmax.  Tile i lives in stage i % 4.
    //   Two barriers a tile (256 dims): tile i's K is read in the matrix
    // phases of i, its V in those of i + 1; the matrix phase of tile i + 1
    // loads tile i + 3 (the last read of the stage, by group 1, ended at the
    // barrier before).
    //   One barrier a tile (up to 128): step i of group 0 is softmax i, matrix
    // i + 1; of group 1 matrix i, softmax i; a barrier ends each step.  V of
    // tile i is read into registers in softmax i, so step i reads K of tiles
    // i and i + 1 and V of tile i: it may load tile i + 3 over tile i - 1, and
    // tile i + 1 is whole when it begins (its loads were issued in step i - 2,
    // and the barrier of step i - 1 waits for all loads but the newest
    // tile's).
    // The first tiles that every row sees whole run unrolled by the stage
    // count, so every LDS address is a per-lane base plus an immediate offset;
    // the rest run with the stage computed and mask what is to be masked (all
    // tiles under an array mask at 256 dims, which has few).
    const uint32_t stage_b = 2 * kTileB;
    constexpr bool kOne = Cfg::kAhead;
    // tile that the matrix phase of tile 1 loads
    const int lead = kOne ? 3 + grp : 3;
    // the barrier after group g's phase, entering one of priority PRIO
    auto phase_end = [&](int g, auto PRIO_) __attribute__((always_inline)) {
      constexpr int PRIO = decltype(PRIO_)::value;
      if (!kOne || grp == g) {
        phase_barrier<PRIO, kLoads>();
      } else {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(PRIO);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    constexpr auto kToMatrix = std::integral_constant<int, 1>{};
    constexpr auto kToSoftmax = std::integral_constant<int, 0>{};
    load_tile(0, 0);
    load_tile(1, 1);
    phase_barrier<1, kLoads>();
    if constexpr (kOne) load_tile(2, 2);
    if (grp) phase_barrier<1, kLoads>();
    if (!kOne || grp) load_tile(lead - 1, lead - 1);
    matrix(ka, 0, std::false_type{});
    phase_end(0, kToSoftmax);
    auto ahead = [&](int s) __attribute__((always_inline)) {
      if constexpr (Cfg::kAhead) {
        read_v(va + s * stage_b);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // softmax of tile i, then the matrix phase of tile i + 1
    auto open_tile = [&](int i, auto S_) __attribute__((always_inline)) {
      constexpr int S = decltype(S_)::value;
      ahead(S);
      softmax(i, false, std::false_type{});
      phase_end(1, kToMatrix);
      load_tile(i + lead, (S + lead) % kStages);
      // past the last tile this scores the clamped copy of the last tile
      // (loaded and complete like any other): unused, but no branch
      matrix(ka + ((S + 1) % kStages) * stage_b, va + S * stage_b, std::true_type{});
      phase_end(0, kToSoftmax);
    };
    int i = 0;
    if constexpr (!(ARR && D == 256)) {
      for (; i + kStages <= n_open; i += kStages) {
        open_tile(i, std::integral_constant<int, 0>{});
        open_tile(i + 1, std::integral_constant<int, 1>{});
        open_tile(i + 2, std::integral_constant<int, 2>{});
        open_tile(i + 3, std::integral_constant<int, 3>{});
      }
    }
    for (; i < ntiles; i++) {
      const int s = i % kStages;
      ahead(s);
      softmax(i, i >= n_open, std::true_type{});
      phase_end(1, kToMatrix);
      load_tile(i + lead, (s + lead) % kStages);
      matrix(ka + ((s + 1) % kStages) * stage_b, va + s * stage_b, std::true_type{});
      phase_end(0, kToSoftmax);
    }
    // group 0 has one barrier fewer: it meets group 1's last one here
    if (!kOne && !grp) phase_barrier<0, kLoads>();
    tile_wait_all();  // the clamped loads issued past the end
  }

  // ---- output: lane (l32, kg) holds, in o[db][j], query row qrow and dim
  // 32 db + 8 (j / 4) + 4 kg + j % 4
  const float lt = l_run + __shfl_xor(l_run, 32);
  if (qrow >= nrows) return;
  const int64_t grow = b * L + qpos;  // row of the batch x L
  if (a.n_parts == 1) {
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    typename E::T* op = static_cast<typename E::T*>(a.out) + b * a.o_sb + qhead * a.o_sh + qpos * a.o_sl;
#pragma unroll
    for (int db = 0; db < kDBw; db++)
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int d = 32 * (dh * kDBw + db) + 8 * m + 4 * kg;
        u32x2_t w;
        w[0] = pack2<DT>(o[db][4 * m] * inv, o[db][4 * m + 1] * inv);
        w[1] = pack2<DT>(o[db][4 * m + 2] * inv, o[db][4 * m + 3] * inv);
        *reinterpret_cast<u32x2_t*>(op + d) = w;
      }
  } else {
    // unnormalized partial; (max, sum) with the max in natural-log units
    const int64_t base = (grow * a.Hq + qhead) * a.n_parts + part;
    float* wo = a.ws_o + base * D + 32 * dh * kDBw;
#pragma unroll
    for (int db = 0; db < kDBw; db++)
#pragma unroll
      for (int j = 0; j < 16; j++) wo[32 * db + 8 * (j >> 2) + 4 * kg + (j & 3)] = o[db][j];
    if (kg == 0 && dh == 0) {  // the two dim halves hold the same (max, sum)
      a.ws_ml[base * 2] = lt > 0.f ? m_run * (1.0f / kLog2e) : -INFINITY;
      a.ws_ml[base * 2 + 1] = lt;
    }
  }
}

}  // namespace

bool prefill_supported(int dtype, int bits, const AttnArgs& a) {
  if (bits != 0 || a.kv.table || a.kv.qfmt) return false;
  if (dtype != kBF16 && dtype != kF16) return false;
  if (a.L < 2 || a.Dv != a.D || a.Hq % a.Hkv) return false;
  // 32-bit query rows
  if (static_cast<int64_t>(a.L) * (a.Hq / a.Hkv) >= (int64_t{1} << 30)) return false;
  if (a.D != 64 && a.D != 128 && a.D != 256) return false;
  // none, causal, or a bool array (additive arrays are the generic kernel's);
  // an array's scores are compared before the scale, so scale > 0, and its
  // word offsets are 32-bit
  if (a.mask_mode != 0 && a.mask_mode != 1 && a.mask_mode != 2) return false;
  if (a.mask_mode == 2 && (!(a.scale > 0.0f) || !a.mask)) return false;
  // uniform rows: a causal chunk longer than the keys is the generic
  // kernel's; ragged rows (seq_lens) shorter than the chunk see no keys for
  // their first queries, as there
  if (a.mask_mode == 1 && !a.kv.seq_lens && a.L > a.kv.T) return false;
  // 16-byte loads of query rows and of K / V rows
  auto al = [](const void* p, int64_t s0, int64_t s1, int64_t s2) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0 && s0 % 16 == 0 && s1 % 16 == 0 && s2 % 16 == 0;
  };
  if (!al(a.kv.kc.ptr, a.kv.kc.sb, a.kv.kc.sh, a.kv.kc.st) ||
      !al(a.kv.vc.ptr, a.kv.vc.sb, a.kv.vc.sh, a.kv.vc.st))
    return false;
  const int64_t es = 2;
  if (reinterpret_cast<uintptr_t>(a.q) % 16 || (a.q_sb * es) % 16 || (a.q_sh * es) % 16 ||
      (a.q_sl * es) % 16)
    return false;
  // 8-byte output stores
  if (reinterpret_cast<uintptr_t>(a.out) % 8 || (a.o_sb * es) % 8 || (a.o_sh * es) % 8 ||
      (a.o_sl * es) % 8)
    return false;
  // 32-bit per-lane offsets within a (row, head) of K / V
  if (a.kv.T * std::max(a.kv.kc.st, a.kv.vc.st) >= (int64_t(1) << 31)) return false;
  return true;
}

static int prefill_rows_per_wg(int D) { return D == 256 ? PfCfg<256>::kRows : PfCfg<128>::kRows; }

int prefill_parts(int64_t rows, int Hkv, int64_t L, int rep, int64_t T, int D, int32_t* part_tokens) {
  const int64_t rpw = prefill_rows_per_wg(D);
  const int64_t rblocks = (L * rep + rpw - 1) / rpw;
  const int64_t wgs = rows * Hkv * rblocks;  // rows = batch rows here
  // one workgroup per CU
  int64_t parts = std::max<int64_t>(1, 256 / std::max<int64_t>(1, wgs));
  parts = std::min<int64_t>(parts, std::max<int64_t>(1, (T + 255) / 256));
  int64_t pt = (T + parts - 1) / parts;
  pt = (pt + kTok - 1) / kTok * kTok;
  *part_tokens = static_cast<int32_t>(std::max<int64_t>(kTok, pt));
  return static_cast<int>((T + *part_tokens - 1) / *part_tokens);
}

namespace {
// Extents of a packed mask: batch rows and heads it distinguishes.
struct MaskPlan {
  int64_t nb, nz, rows, words, rblocks;
};
MaskPlan mask_plan(const AttnArgs& a, int64_t batch) {
  MaskPlan p;
  // (rows of unequal length differ even under one mask)
  p.nb = a.m_sb || a.kv.seq_lens ? batch : 1;
  p.nz = p.nb * (a.m_sh ? a.Hkv : 1);
  p.rows = p.nb * (a.m_sh ? a.Hq : 1) * a.L;
  // whole 1024-key groups, so that a row's per-256-key bytes fill 32-bit words
  p.words = (static_cast<int64_t>(a.kv.T) + 1023) / 1024 * 32;
  const int64_t rpw = prefill_rows_per_wg(a.D);
  p.rblocks = (static_cast<int64_t>(a.L) * (a.Hq / a.Hkv) + rpw - 1) / rpw;
  return p;
}
}  // namespace

bool prefill_mask_fits(const AttnArgs& a, int64_t batch) {
  if (a.mask_mode != 2) return true;
  const MaskPlan p = mask_plan(a, batch);
  return 4 * p.rows * p.words < (int64_t{1} << 32) && p.rblocks < 65536 && p.nz < 65536;
}

size_t prefill_mask_floats(const AttnArgs& a, int64_t batch) {
  if (a.mask_mode != 2) return 0;
  const MaskPlan p = mask_plan(a, batch);
  const int64_t bytes = 4 * p.rows * p.words + p.rows * p.words / 8 + p.nz * p.rblocks * p.words;
  return static_cast<size_t>((bytes + 255) / 256 * 64);
}

void prefill_mask_parts(const AttnArgs& a, int64_t T, int32_t* part_tokens, int32_t* n_parts) {
  if (a.mask_mode != 2 || *part_tokens <= kMaxMaskTiles * kTok) return;
  *part_tokens = kMaxMaskTiles * kTok;
  *n_parts = static_cast<int32_t>((T + *part_tokens - 1) / *part_tokens);
}

void launch_prefill_mask(AttnArgs& a, int64_t batch, float* ws, hipStream_t st) {
  if (a.mask_mode != 2 || batch <= 0 || a.L <= 0) return;
  const MaskPlan p = mask_plan(a, batch);
  a.mw = reinterpret_cast<uint32_t*>(ws);
  a.mrow = reinterpret_cast<uint8_t*>(a.mw + p.rows * p.words);
  a.mcls = a.mrow + p.rows * p.words / 8;
  a.mw_words = p.words;
  a.mw_h = a.m_sh ? a.L : 0;
  a.mw_b = p.nb > 1 ? (a.m_sh ? static_cast<int64_t>(a.Hq) : 1) * a.L : 0;
  const dim3 grid(static_cast<unsigned>(p.words / 8), static_cast<unsigned>(p.rblocks),
                  static_cast<unsigned>(p.nz));
  hipLaunchKernelGGL(mask_pack_kernel, grid, dim3(512), 0, st, a, a.Hq / a.Hkv,
                     static_cast<int>(prefill_rows_per_wg(a.D)));
  VKV_HIP(hipGetLastError());
}

template <int D, bool ARR>
static void launch_prefill_d(int dtype, bool qsem, const AttnArgs& a, const dim3& grid, int rep,
                             hipStream_t st) {
  if (dtype == kBF16 && qsem)
    hipLaunchKernelGGL((prefill_kernel<kBF16, true, D, ARR>), grid, dim3(kThreads), 0, st, a, rep);
  else if (dtype == kBF16)
    hipLaunchKernelGGL((prefill_kernel<kBF16, false, D, ARR>), grid, dim3(kThreads), 0, st, a, rep);
  else if (qsem)
    hipLaunchKernelGGL((prefill_kernel<kF16, true, D, ARR>), grid, dim3(kThreads), 0, st, a, rep);
  else
    hipLaunchKernelGGL((prefill_kernel<kF16, false, D, ARR>), grid, dim3(kThreads), 0, st, a, rep);
}

void launch_prefill(int dtype, bool qsem, const AttnArgs& a, int64_t batch, hipStream_t st,
                    bool combine) {
  if (batch <= 0 || a.L <= 0) return;
  VKV_CHECK(a.D == 64 || a.D == 128 || a.D == 256, "prefill kernel head dim");
  const int prun = a.parts_run > 0 ? a.parts_run : a.n_parts;
  VKV_CHECK(a.part0 >= 0 && a.part0 + prun <= a.n_parts, "prefill part window");
  const int rep = a.Hq / a.Hkv;
  const int64_t rpw = prefill_rows_per_wg(a.D);
  const int64_t rblocks = (static_cast<int64_t>(a.L) * rep + rpw - 1) / rpw;
  const int64_t wgs = rblocks * prun * a.Hkv * batch;
  VKV_CHECK(wgs < (int64_t{1} << 31), "too many prefill workgroups for one launch");
  const dim3 grid(static_cast<unsigned>(wgs));
  VKV_CHECK(a.mask_mode != 2 || (a.mw && a.part_tokens <= kMaxMaskTiles * kTok),
            "prefill mask not packed");
  auto run = [&](auto D_) {
    constexpr int D = decltype(D_)::value;
    if (a.mask_mode == 2)
      launch_prefill_d<D, true>(dtype, qsem, a, grid, rep, st);
    else
      launch_prefill_d<D, false>(dtype, qsem, a, grid, rep, st);
  };
  if (a.D == 64)
    run(std::integral_constant<int, 64>{});
  else if (a.D == 128)
    run(std::integral_constant<int, 128>{});
  else
    run(std::integral_constant<int, 256>{});
  VKV_HIP(hipGetLastError());
  if (combine && a.n_parts > 1) launch_attn_combine(dtype, a, batch * a.L, st);
}

}  // namespace vkv
