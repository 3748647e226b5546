// vkv_kernels.hip -- gfx950 kernels of the KV-cache engine: affine
// quantize-on-append (dense and paged, bit-exact with the reference
// quantizer), scatter/gather, dequant-on-read, strided copies, and the
// generic split-K decode attention used for float and quantized caches.
//
// Reference arithmetic: Source/Cmlx/mlx-generated/metal/quantized.h:2393-2560
// (affine quantize / dequantize) and sdpa_vector.h:15-394 (decode SDPA and
// its two-pass combine); Libraries/MLXLMCommon/KVCache.swift:1909-1997
// (quantized SDPA semantics).
#include "vkv_device.h"
#include "vkv_internal.h"
#include "vkv_kvread.h"
#include <hip/hip_ext.h>

#include <algorithm>
#include <type_traits>

namespace vkv {

// ----------------------------------------------------------------- helpers

__device__ __forceinline__ const uint8_t* row_ptr(const RowSrc& s, int64_t row, int esize) {
  const int64_t r1 = index_div(row, s.e2), i0 = index_div(r1, s.e1);
  const int64_t i2 = row - r1 * s.e2, i1 = r1 - i0 * s.e1;
  return static_cast<const uint8_t*>(s.ptr) + (i0 * s.s0 + i1 * s.s1 + i2 * s.s2) * esize;
}

// Quotients by a fixed divisor: x / n = mulhi(x, mul) >> (sh - 1) for x <
// 2^31, with mul = 2^(31 + sh) / n + 1 and 2^sh >= n.
struct FastDiv {
  uint32_t n, mul, sh;
  __device__ __forceinline__ uint32_t quot(uint32_t x) const {
    return n == 1 ? x : __umulhi(x, mul) >> (sh - 1);
  }
};
static FastDiv fast_div(int64_t n) {
  FastDiv f{};
  f.n = static_cast<uint32_t>(n);
  while ((int64_t{1} << f.sh) < n) f.sh++;
  f.mul = static_cast<uint32_t>((uint64_t{1} << (31 + f.sh)) / static_cast<uint64_t>(n) + 1);
  return f;
}

// Slot (block * block_size + offset) of paged token n; < 0 means skip (so
// does an explicit slot past the pool, which would write outside it).
__device__ __forceinline__ int64_t token_slot(const RowDst& d, int64_t n) {
  if (d.slots) {
    const int64_t s = d.slots[n];
    return (d.slot_limit > 0 && s >= d.slot_limit) ? -1 : s;
  }
  const int64_t b = index_div(n, d.seq_S);
  const int64_t pos = d.start + (n - b * d.seq_S), pb = index_div(pos, d.block_size);
  const int32_t blk = d.table[b * d.table_stride + pb];
  if (blk < 0) return -1;
  return static_cast<int64_t>(blk) * d.block_size + (pos - pb * d.block_size);
}

template <int DT>
__device__ __forceinline__ void load8(const uint8_t* p, float* v) {
  using E = Elem<DT>;
  typename E::T q[8];  // (16-byte loads at any element alignment)
  __builtin_memcpy(q, p, sizeof(q));
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = E::to_f32(q[i]);
}

// Store the 8 codes of dims [8j, 8j+8) of token `tib` into a paged chunk
// (format in vkv_device.h).  V codes of one word belong to 8 different
// tokens, so a 4-bit V store is a read-modify-write done with two atomics on
// the containing word (other tokens' nibbles may be written concurrently).
template <int BITS>
__device__ __forceinline__ void store_chunk_codes(uint8_t* chunk, const RowDst& dst, int tib, int j,
                                                  int D, const uint32_t* code) {
  uint8_t* c = chunk + dst.c_off;
  if (!dst.is_v) {
    if constexpr (BITS == 4) {
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < 8; i++) w |= code[i] << (4 * i);
      *reinterpret_cast<uint32_t*>(c + qk_word_off(tib, j, D, 4)) = w;
    } else {
      const uint32_t w0 = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
      const uint32_t w1 = code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24);
      *reinterpret_cast<uint32_t*>(c + qk_word_off(tib, 2 * j, D, 8)) = w0;
      *reinterpret_cast<uint32_t*>(c + qk_word_off(tib, 2 * j + 1, D, 8)) = w1;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      int sh;
      const int64_t off = qv_word_off(tib, j * 8 + i, D, BITS, &sh);
      if constexpr (BITS == 8) {
        c[off + sh / 8] = static_cast<uint8_t>(code[i]);
      } else {
        uint32_t* word = reinterpret_cast<uint32_t*>(c + off);
        atomicAnd(word, ~(0xFu << sh));
        atomicOr(word, code[i] << sh);
      }
    }
  }
}

// ------------------------------------------------------- affine quantize
//
// One thread owns 8 consecutive values of a row; GROUP/8 neighbouring lanes
// form one quantization group and reduce min/max with xor-shuffles; the
// arithmetic is the reference's (affine_quantize8, quantized.h:2422-2458),
// scale/bias stored rounded to T (:2447-2450).
// mode 0 writes the reference layout; mode 1 writes a paged chunk (K rows
// token-major, V rows dim-major).
template <int DT, int BITS, int GROUP, int MODE>
__global__ void __launch_bounds__(256) quantize_rows_kernel(RowSrc src, RowDst dst, int64_t rows,
                                                            int D) {
  using E = Elem<DT>;
  constexpr int TEAM = GROUP / 8;
  const int tpr = D / 8;
  const int64_t gtid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t row = index_div(gtid, tpr);
  const int j = static_cast<int>(gtid - row * tpr);
  const bool active = row < rows;

  float v[8];
  if (active) {
    load8<DT>(row_ptr(src, row, E::kBytes) + static_cast<int64_t>(j) * 8 * E::kBytes, v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = 0.0f;
  }
  uint32_t code[8];
  float scale, bias;
  affine_quantize8<DT, BITS, GROUP>(v, code, scale, bias);
  if (!active) return;
  const int G = D / GROUP;
  const int g = (j * 8) / GROUP;
  const bool group_leader = (j % TEAM) == 0;
  const typename E::T s_t = E::from_f32(scale);
  const typename E::T b_t = E::from_f32(bias);

  if constexpr (MODE == 0) {
    uint32_t* wq = static_cast<uint32_t*>(dst.wq) + row * (D * BITS / 32);
    if constexpr (BITS == 4) {
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < 8; i++) w |= code[i] << (4 * i);
      wq[j] = w;
    } else {
      uint32_t w0 = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
      uint32_t w1 = code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24);
      wq[2 * j] = w0;
      wq[2 * j + 1] = w1;
    }
    if (group_leader) {
      static_cast<typename E::T*>(dst.scales)[row * G + g] = s_t;
      static_cast<typename E::T*>(dst.biases)[row * G + g] = b_t;
    }
  } else {
    const int64_t n = index_div(row, src.e2);
    const int64_t h = row - n * src.e2;
    const int64_t slot = token_slot(dst, n);
    if (slot < 0) return;
    const int64_t blk = index_div(slot, dst.block_size);
    const int tib = static_cast<int>(slot - blk * dst.block_size);
    uint8_t* chunk = dst.base + blk * dst.block_bytes + h * dst.head_bytes;
    store_chunk_codes<BITS>(chunk, dst, tib, j, D, code);
    if (group_leader) {
      typename E::T* sbp = reinterpret_cast<typename E::T*>(chunk + dst.s_off);
      sbp[qsb_index(tib, dst.is_v, g, 0, dst.G, dst.keys_only)] = s_t;
      sbp[qsb_index(tib, dst.is_v, g, 1, dst.G, dst.keys_only)] = b_t;
    }
  }
}

// Paged append of K and V in one launch (Pool::append): block = 8
// consecutive tokens x HB heads x the D/8 threads of a row (256 threads);
// blockIdx.z selects K (0) or V (1).  The arithmetic is that of
// quantize_rows_kernel.  V words hold 8 (4-bit) or 4 (8-bit) tokens of one
// dim; they are assembled from the block's 8 tokens in LDS: whole aligned
// 8-token groups (a prefill chunk) are plain stores, and of a 4-bit group
// that the block holds part of, each run of tokens is merged into the word
// with one pair of atomics (8-bit codes are then stored byte by byte).
// Bound by the vector ALUs on large appends (affine_quantize8), by the
// chain slot -> page -> stores on a step's few tokens.  Measured (8 x 4096
// bf16 tokens x 8 heads x 128, K and V, 172 MB moved): 130 -> 61 us from the
// divisions by multiplication (values: affine_quantize8; indexes: AppendDiv);
// 246K tokens of which no group of 8 starts on a page boundary, 5.2 -> 0.7 ms
// from one atomic pair a run instead of one a nibble.
// Tokens and positions are below 2^31 and divide by multiplication (dv).
struct AppendDiv {
  FastDiv e1;   // tokens of a batch row (the source's, and the table's seq_S)
  FastDiv bs;   // tokens of a block
};

template <int DT, int BITS, int GROUP>
__global__ void __launch_bounds__(256) append_affine_kernel(RowSrc sk, RowSrc sv, RowDst dk, RowDst dv,
                                                            uint32_t ntok, int H, int D, AppendDiv dq) {
  using E = Elem<DT>;
  constexpr int TEAM = GROUP / 8;
  const int which = blockIdx.z;
  const RowSrc& src = which ? sv : sk;
  const RowDst& dst = which ? dv : dk;
  const int lt = 31 - __builtin_clz(D / 8);  // D = 32 .. 256, a power of two
  const int tpr = 1 << lt, hb = 32 >> lt;
  const int tid = threadIdx.x;
  const int i = tid >> 5, hl = (tid >> lt) & (hb - 1), j = tid & (tpr - 1);
  const uint32_t n = blockIdx.x * 8 + i;
  const int h = blockIdx.y * hb + hl;
  const bool active = n < ntok && h < H;
  const uint32_t i0 = dq.e1.quot(n), i1 = n - i0 * static_cast<uint32_t>(src.e1);

  // the token's block and place in it (-1: skipped); its read goes out with
  // the row's load
  int blk = -1, tib = 0;
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = 0.0f;
  if (active) {
    uint32_t pos;
    int32_t at;
    if (dst.slots) {
      at = dst.slots[n];
    } else {
      pos = dst.start + i1;
      const uint32_t pb = dq.bs.quot(pos);
      tib = static_cast<int>(pos - pb * static_cast<uint32_t>(dst.block_size));
      at = dst.table[static_cast<int64_t>(i0) * dst.table_stride + pb];
    }
    load8<DT>(static_cast<const uint8_t*>(src.ptr) +
                  (i0 * src.s0 + i1 * src.s1 + h * src.s2 + 8 * j) * E::kBytes,
              v);
    blk = at;
    if (dst.slots && at >= 0) {
      blk = static_cast<int>(dq.bs.quot(at));
      tib = at - blk * dst.block_size;
      if (dst.slot_limit > 0 && at >= dst.slot_limit) blk = -1;
    }
  }
  uint32_t code[8];
  float scale, bias;
  affine_quantize8<DT, BITS, GROUP>(v, code, scale, bias);
  uint8_t* chunk = dst.base + blk * dst.block_bytes + h * dst.head_bytes;
  if (blk >= 0 && (j % TEAM) == 0) {
    const int g = (j * 8) / GROUP;
    typename E::T* sbp = reinterpret_cast<typename E::T*>(chunk + dst.s_off);
    sbp[qsb_index(tib, dst.is_v, g, 0, dst.G, dst.keys_only)] = E::from_f32(scale);
    sbp[qsb_index(tib, dst.is_v, g, 1, dst.G, dst.keys_only)] = E::from_f32(bias);
  }
  if (which == 0) {  // K words are whole stores
    if (blk >= 0) store_chunk_codes<BITS>(chunk, dst, tib, j, D, code);
    return;
  }
  // ---- V
  __shared__ int2 tok[8];  // block and place of each token
  __shared__ __attribute__((aligned(8))) uint8_t vcode[8][256];  // [token][head * D + dim], hb * D = 256
  if (hl == 0 && j == 0) tok[i] = make_int2(blk, tib);  // hl 0: a head below H
  uint2 c8;
  c8.x = code[0] | code[1] << 8 | code[2] << 16 | code[3] << 24;
  c8.y = code[4] | code[5] << 8 | code[6] << 16 | code[7] << 24;
  *reinterpret_cast<uint2*>(&vcode[i][hl * D + 8 * j]) = c8;
  __syncthreads();
  // the 8 tokens are one aligned 8-token group (its block's size is a
  // multiple of 8)
  const int2 t0 = tok[0];
  bool whole = t0.x >= 0 && t0.y % 8 == 0;
#pragma unroll
  for (int t = 1; t < 8; t++) whole = whole && tok[t].x == t0.x && tok[t].y == t0.y + t;
  if (BITS == 8 && !whole) {  // bytes are whole stores
    if (blk >= 0) store_chunk_codes<BITS>(chunk, dst, tib, j, D, code);
    return;
  }
  // thread (head hh, dim d) writes the words of its dim
  const int hh = tid >> (lt + 3), d = tid & (D - 1);
  if (blockIdx.y * hb + hh >= H) return;
  uint8_t* vbase = dst.base + static_cast<int64_t>(blockIdx.y * hb + hh) * dst.head_bytes + dst.c_off;
  auto word_at = [&](const int2& p) {
    int sh;
    return vbase + p.x * dst.block_bytes + qv_word_off(p.y, d, D, BITS, &sh);
  };
  if (whole) {
    uint2 w = {0, 0};
#pragma unroll
    for (int t = 0; t < 8; t++) {
      if constexpr (BITS == 4)
        w.x |= static_cast<uint32_t>(vcode[t][tid]) << (4 * t);
      else
        (t < 4 ? w.x : w.y) |= static_cast<uint32_t>(vcode[t][tid]) << (8 * (t & 3));
    }
    if constexpr (BITS == 4)
      *reinterpret_cast<uint32_t*>(word_at(t0)) = w.x;
    else
      *reinterpret_cast<uint2*>(word_at(t0)) = w;
    return;
  }
  if constexpr (BITS == 4) {
    // runs of tokens of one group: other tokens' nibbles of a word may be
    // written concurrently
    uint32_t w = 0, m = 0;
    int2 cur = make_int2(-1, 0);
#pragma unroll 1
    for (int t = 0; t <= 8; t++) {
      const int2 p = t < 8 ? tok[t] : make_int2(-1, 0);
      if (m && (p.x != cur.x || p.y >> 3 != cur.y >> 3)) {
        uint32_t* at = reinterpret_cast<uint32_t*>(word_at(cur));
        atomicAnd(at, ~m);
        atomicOr(at, w);
        w = m = 0;
      }
      if (p.x < 0) continue;
      cur = p;
      const int sh = 4 * (p.y & 7);
      w = (w & ~(15u << sh)) | static_cast<uint32_t>(vcode[t][tid]) << sh;
      m |= 15u << sh;
    }
  }
}

// Float rows of K and V (blockIdx.y) into the pages of their tokens' slots,
// token-major, 16 bytes a thread where rows and pages are aligned to them.  A
// decode step's few rows are latency bound (the slot, then the row's store):
// one launch for both matrices and 32-bit index arithmetic, 9.4 -> 4.7 us for
// the two of a step of 16 tokens x 8 heads.
template <int ESIZE, bool VEC>
__global__ void __launch_bounds__(256) append_rows_kernel(RowSrc sk, RowSrc sv, RowDst dk, RowDst dv,
                                                          int64_t t0, uint32_t rows, int Dk, int Dv) {
  const RowSrc& src = blockIdx.y ? sv : sk;
  const RowDst& dst = blockIdx.y ? dv : dk;
  const int D = blockIdx.y ? Dv : Dk;
  const uint32_t tpr = (D * ESIZE + 15) / 16;  // 16-byte pieces of a row
  const uint32_t gtid = blockIdx.x * 256u + threadIdx.x;
  const uint32_t row = gtid / tpr;
  if (row >= rows) return;
  const uint32_t j = gtid - row * tpr;
  const uint32_t heads = static_cast<uint32_t>(src.e2);
  const uint32_t n = row / heads, h = row - n * heads;
  const int64_t slot = token_slot(dst, t0 + n);
  const uint8_t* s = static_cast<const uint8_t*>(src.ptr) +
                     ((t0 + n) * src.s1 + h * src.s2) * ESIZE + 16 * j;
  if (slot < 0) return;
  const uint32_t blk = static_cast<uint32_t>(slot) / static_cast<uint32_t>(dst.block_size);
  const uint32_t tib = static_cast<uint32_t>(slot) - blk * dst.block_size;
  uint8_t* o = dst.base + static_cast<int64_t>(blk) * dst.block_bytes + h * dst.head_bytes + dst.c_off +
               static_cast<int64_t>(tib) * D * ESIZE + 16 * j;
  if constexpr (VEC) {
    *reinterpret_cast<uint4*>(o) = *reinterpret_cast<const uint4*>(s);
  } else {
    using U = std::conditional_t<ESIZE == 2, uint16_t, uint32_t>;
    const int cnt = min(16 / ESIZE, D - static_cast<int>(j) * (16 / ESIZE));
    for (int i = 0; i < cnt; i++) reinterpret_cast<U*>(o)[i] = reinterpret_cast<const U*>(s)[i];
  }
}

// quantized.h:2498-2560: out = scale * q + bias, here one fp32 fma rounded
// once to T.  Thread per 8 values, contiguous operands.
template <int DT, int BITS>
__global__ void __launch_bounds__(256) dequantize_kernel(const uint32_t* wq, const void* scales,
                                                         const void* biases, void* out, int64_t rows,
                                                         int D, int group) {
  using E = Elem<DT>;
  const int tpr = D / 8;
  const int64_t gtid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t row = gtid / tpr;
  const int j = static_cast<int>(gtid % tpr);
  if (row >= rows) return;
  const int G = D / group;
  const int g = j * 8 / group;
  const float s = E::load(static_cast<const typename E::T*>(scales) + row * G + g);
  const float b = E::load(static_cast<const typename E::T*>(biases) + row * G + g);
  const uint32_t* w = wq + row * (D * BITS / 32);
  typename E::T* o = static_cast<typename E::T*>(out) + row * D + j * 8;
  if constexpr (BITS == 4) {
    uint32_t x = w[j];
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = E::from_f32(fmaf(s, static_cast<float>((x >> (4 * i)) & 15u), b));
  } else {
    uint32_t x0 = w[2 * j], x1 = w[2 * j + 1];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      o[i] = E::from_f32(fmaf(s, static_cast<float>((x0 >> (8 * i)) & 255u), b));
      o[4 + i] = E::from_f32(fmaf(s, static_cast<float>((x1 >> (8 * i)) & 255u), b));
    }
  }
}

// --------------------------------------------------------------- gather
//
// Thread per (seq, head, token, 8 dims).  out_kind 0: values (dequantized
// when bits > 0) into [n,H,T,D] of dtype; out_kind 1: reference-layout codes.
template <int DT, int BITS, int KIND>
__global__ void __launch_bounds__(256) gather_kernel(GatherArgs g) {
  using E = Elem<DT>;
  const int tpr = (g.D + 7) / 8;
  const int64_t gtid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t row = gtid / tpr;  // (s, h, t)
  const int j = static_cast<int>(gtid % tpr);
  const int64_t total = static_cast<int64_t>(g.n_seqs) * g.H * g.T;
  if (row >= total) return;
  const int64_t t = row % g.T;
  const int64_t h = (row / g.T) % g.H;
  const int64_t s = row / (static_cast<int64_t>(g.T) * g.H);
  const int64_t len = g.kv.seq_lens ? g.kv.seq_lens[s] : g.kv.T;
  if (t + g.t_begin >= len) return;
  const TokLoc l = locate(g.kv, s, t + g.t_begin);
  const int d0 = j * 8;
  const int cnt = min(8, g.D - d0);
  if constexpr (KIND == 0) {
    typename E::T* o = static_cast<typename E::T*>(g.out) + row * g.D + d0;
    for (int i = 0; i < cnt; i++) o[i] = E::from_f32(kv_at<DT, BITS>(g.kv, l, h, d0 + i, g.which, g.group));
  } else {
    // codes of dims [d0, d0+8) re-packed little-endian into the reference layout
    uint32_t code[8];
    float s = 0.0f, b = 0.0f;
    for (int i = 0; i < 8; i++) code[i] = qcode<DT, BITS>(g.kv, l, h, d0 + i, g.which, g.group, &s, &b);
    // (the output row: token out_t0 + t of rows out_cap tokens long)
    const int64_t orow = (row / g.T) * (g.out_cap ? g.out_cap : g.T) + g.out_t0 + t;
    uint32_t* wq = static_cast<uint32_t*>(g.out) + orow * (g.D * BITS / 32);
    if constexpr (BITS == 4) {
      uint32_t w = 0;
      for (int i = 0; i < 8; i++) w |= code[i] << (4 * i);
      wq[j] = w;
    } else {
      wq[2 * j] = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
      wq[2 * j + 1] = code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24);
    }
    if (d0 % g.group == 0) {
      // s and b of the group holding dims [d0, d0+8) (exact stored values)
      const int G = g.D / g.group;
      const int gi = d0 / g.group;
      static_cast<typename E::T*>(g.out_s)[orow * G + gi] = E::from_f32(s);
      static_cast<typename E::T*>(g.out_b)[orow * G + gi] = E::from_f32(b);
    }
  }
}

// Two floats rounded to bf16 / f16 (nearest even), the first in the low half.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
template <int DT>
__device__ __forceinline__ uint32_t pack_pair(float a, float b) {
  if constexpr (DT == kBF16)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
  else
    return static_cast<uint32_t>(Elem<DT>::from_f32(a)) | (static_cast<uint32_t>(Elem<DT>::from_f32(b)) << 16);
}

// Dequantizing gather, 8 dims a thread: one code word (4-bit) or two (8-bit)
// and one scale/bias pair (a group spans a multiple of 8 dims), then one
// 16-byte store of bf16/f16 (two of f32); paged values hold a dim's 8 tokens a
// word (two at 8 bits), so they take 8 words.  The values are those of
// gather_kernel<.., 0>: the fp32 scale * code + bias rounded to the dtype.
// blockIdx.y is the (seq, head) plane; with gridDim.z == 2, blockIdx.z picks
// K (into out) or V (into out_v) in one launch.  One piece a thread: more
// workgroups keep more loads in flight.  Needs D and group multiples of 8,
// 4-byte aligned code rows, a 16-byte aligned output and (row, head) chunks
// below 2^31 bytes (gather8_ok).
//
// Bound: one chain table -> codes -> store a thread, behind the launch (HBM
// would take 5 us of the example), and the index arithmetic before it.
// Indices are divided by multiplication, chunk offsets are 32-bit and bf16
// pairs are converted by the packed instruction: 4608 tokens of 8 heads x 128,
// 4 bits, K and V (24 MB) 10.7 -> 9.6 us.
template <int DT, int BITS>
__global__ void __launch_bounds__(256) gather_dequant8_kernel(GatherArgs g, FastDiv tpr, FastDiv bs,
                                                              FastDiv grp) {
  using E = Elem<DT>;
  constexpr uint32_t kMask = (1u << BITS) - 1u;
  const int plane = blockIdx.y, s = plane / g.H, h = plane - s * g.H;
  // tokens of this row in the window [t_begin, t_begin + T)
  const int len =
      min(g.T, static_cast<int>(g.kv.seq_lens ? g.kv.seq_lens[s] : g.kv.T) - g.t_begin);
  const KVSrc& kv = g.kv;
  const bool ko = kv.keys_only != 0;
  const int which = gridDim.z > 1 ? static_cast<int>(blockIdx.z) : g.which;
  void* const out = which && gridDim.z > 1 ? g.out_v : g.out;
  const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
  const int ti = static_cast<int>(tpr.quot(idx)), u = static_cast<int>(idx) - ti * static_cast<int>(tpr.n);
  if (ti >= len) return;
  const int t = g.t_begin + ti, gi = static_cast<int>(grp.quot(u));
  int blk = s, tib = t;
  if (kv.table) {
    const int b = static_cast<int>(bs.quot(t));
    blk = kv.table[static_cast<int64_t>(s) * kv.table_stride + b];
    tib = t - b * static_cast<int>(bs.n);
  }
  uint32_t c[8];
  float sc, bi;
  if (kv.qfmt) {
    const uint8_t* chunk = kv.base + blk * kv.block_bytes + h * kv.head_bytes;
    const int w = (which && !ko) ? 1 : 0;
    const typename E::T* sb = reinterpret_cast<const typename E::T*>(chunk + kv.sb_off) +
                              (tib * (ko ? 2 : 4) + 2 * w) * kv.G + 2 * gi;
    sc = E::load(sb);
    bi = E::load(sb + 1);
    if (w == 0) {
      // the unit's original word(s) (one at 4 bits, two at 8), which the
      // chunk keeps side by side (qk_word_off)
      const uint32_t* p = reinterpret_cast<const uint32_t*>(chunk + kv.kc_off) +
                          (tib * (kv.D >> 3) + (u & 3) * (kv.D >> 5) + (u >> 2)) * (BITS / 4);
#pragma unroll
      for (int i = 0; i < 8; i++) c[i] = (p[i * BITS / 32] >> (i * BITS % 32)) & kMask;
    } else {
      // dims 8 u .. + 7: m = 8 (u & 1) + i of tile u / 2 (qv_word_off)
      const int NT = kv.D >> 4, q = tib & 7;
      const uint32_t* p = reinterpret_cast<const uint32_t*>(chunk + kv.vc_off) + (tib >> 5) * kv.D * BITS +
                          ((((tib >> 3) & 3) * 16 + 8 * (u & 1)) * NT + (u >> 1)) * (BITS / 4) +
                          (BITS == 8 ? q >> 2 : 0);
      const int sh = BITS == 4 ? 4 * q : 8 * (q & 3);
#pragma unroll
      for (int i = 0; i < 8; i++) c[i] = (p[i * NT * (BITS / 4)] >> sh) & kMask;
    }
  } else {
    const TokLoc l{blk, tib};
    const Comp& cc = which ? kv.vc : kv.kc;
    const Comp& scp = which ? kv.vs : kv.ks;
    const Comp& bcp = which ? kv.vb : kv.kb;
    sc = E::load(reinterpret_cast<const typename E::T*>(at(scp, l, h)) + gi);
    bi = E::load(reinterpret_cast<const typename E::T*>(at(bcp, l, h)) + gi);
    const uint32_t* p = reinterpret_cast<const uint32_t*>(at(cc, l, h) + u * BITS);
#pragma unroll
    for (int i = 0; i < 8; i++) c[i] = (p[i * BITS / 32] >> (i * BITS % 32)) & kMask;
  }
  float f[8];
#pragma unroll
  for (int i = 0; i < 8; i++) f[i] = fmaf(sc, static_cast<float>(c[i]), bi);
  typename E::T* o =
      static_cast<typename E::T*>(out) + (static_cast<int64_t>(plane) * g.T + ti) * g.D + 8 * u;
  if constexpr (E::kBytes == 2) {
    uint32_t pk[4];
#pragma unroll
    for (int i = 0; i < 4; i++) pk[i] = pack_pair<DT>(f[2 * i], f[2 * i + 1]);
    *reinterpret_cast<uint4*>(o) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
  } else {
    reinterpret_cast<float4*>(o)[0] = make_float4(f[0], f[1], f[2], f[3]);
    reinterpret_cast<float4*>(o)[1] = make_float4(f[4], f[5], f[6], f[7]);
  }
}

// Codes, scales and biases of paged affine chunks in the reference layout.
// blockIdx.y is the (seq, head) plane.  Keys: a thread writes 4 words of a
// token's row (the chunk keeps a row's words permuted).  Values: a thread
// reads the words of 8 dims of an aligned 8-token group (dim-major in the
// chunk) and transposes them in registers, so every word is read once; lanes
// take neighbouring words of the chunk, then the two halves of a 16-dim tile.
// HBM bound: 8 x 4096 tokens x 8 heads x 128 at 4 bits (19 MB read, 19
// written a matrix) take 8.6 us for the keys and 8.9 for the values, 48 with a
// thread per (token, 8 dims) that read 8 words for 8 nibbles and divided in 64
// bits.
template <int DT, int BITS>
__global__ void __launch_bounds__(256) gather_codes_kernel(GatherArgs g) {
  using T = typename Elem<DT>::T;
  const KVSrc& kv = g.kv;
  const int plane = blockIdx.y, s = plane / g.H, h = plane - s * g.H;
  // tokens [t_begin, t_end) of this row
  const int t_end =
      min(g.t_begin + g.T, static_cast<int>(kv.seq_lens ? kv.seq_lens[s] : kv.T));
  const int D = g.D, G = D / g.group, W = D * BITS / 32;
  const int64_t row0 = static_cast<int64_t>(plane) * (g.out_cap ? g.out_cap : g.T) + g.out_t0 - g.t_begin;
  uint32_t* wq = static_cast<uint32_t*>(g.out);
  const int which = g.which, idx = blockIdx.x * 256 + static_cast<int>(threadIdx.x);
  auto chunk_of = [&](int t, int& tib) {
    const int b = t / kv.block_size;
    tib = t - b * kv.block_size;
    const int64_t blk = kv.table[static_cast<int64_t>(s) * kv.table_stride + b];
    return kv.base + blk * kv.block_bytes + h * kv.head_bytes;
  };
  auto scales = [&](const uint8_t* chunk, int tib, int t, int gi) {
    const T* sb = reinterpret_cast<const T*>(chunk + kv.sb_off);
    static_cast<T*>(g.out_s)[(row0 + t) * G + gi] = sb[qsb_index(tib, which, gi, 0, kv.G, kv.keys_only)];
    static_cast<T*>(g.out_b)[(row0 + t) * G + gi] = sb[qsb_index(tib, which, gi, 1, kv.G, kv.keys_only)];
  };
  if (which == 0) {
    const int per = W / 4, ti = idx / per, q = idx - ti * per, t = g.t_begin + ti;
    if (t >= t_end) return;
    int tib;
    const uint8_t* chunk = chunk_of(t, tib);
    const uint32_t* row = reinterpret_cast<const uint32_t*>(chunk + kv.kc_off) + static_cast<int64_t>(tib) * W;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int o = 4 * q + e, p = BITS == 4 ? o : o >> 1;  // original word; its 8-dim unit
      const int pos = (p & 3) * (D / 32) + (p >> 2);
      w[e] = row[BITS == 4 ? pos : 2 * pos + (o & 1)];
    }
    uint32_t* o = wq + (row0 + t) * W + 4 * q;
    *reinterpret_cast<uint4*>(o) = make_uint4(w[0], w[1], w[2], w[3]);
    for (int gi = q; gi < G; gi += per) scales(chunk, tib, t, gi);
    return;
  }
  // values: 8-token groups counted from the aligned one holding t_begin; a
  // thread takes dims 16 mt + 8 hf .. + 8, mt fastest
  const int NT = D / 16, per = D / 8;
  const int gq = idx / per, r = idx - gq * per, hf = r / NT, mt = r - hf * NT;
  const int t8 = (g.t_begin & ~7) + 8 * gq;
  if (t8 >= t_end) return;
  int tib;
  const uint8_t* chunk = chunk_of(t8, tib);
  const uint32_t* vb = reinterpret_cast<const uint32_t*>(chunk + kv.vc_off) +
                       static_cast<int64_t>(tib >> 5) * (D * BITS / 4);
  const int kg = (tib & 31) >> 3;
  uint32_t w[8][BITS / 4];
#pragma unroll
  for (int e = 0; e < 8; e++)
#pragma unroll
    for (int x = 0; x < BITS / 4; x++)
      w[e][x] = vb[((kg * 16 + 8 * hf + e) * NT + mt) * (BITS / 4) + x];
  // w[dim e]: codes of 8 tokens -> token k: codes of 8 dims
  auto swap = [](uint32_t& a, uint32_t& b, int sh, uint32_t m) __attribute__((always_inline)) {
    const uint32_t t = ((a >> sh) ^ b) & m;
    b ^= t;
    a ^= t << sh;
  };
  uint32_t out[8][BITS / 4];
  if constexpr (BITS == 4) {
#pragma unroll
    for (int e = 0; e < 4; e++) swap(w[e][0], w[e + 4][0], 16, 0x0000FFFFu);
#pragma unroll
    for (int e = 0; e < 8; e += (e & 1) ? 3 : 1) swap(w[e][0], w[e + 2][0], 8, 0x00FF00FFu);
#pragma unroll
    for (int e = 0; e < 8; e += 2) swap(w[e][0], w[e + 1][0], 4, 0x0F0F0F0Fu);
#pragma unroll
    for (int k = 0; k < 8; k++) out[k][0] = w[k][0];
  } else {
    // two 4 x 4 byte transposes per half of the tokens
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 2; y++) {
        uint32_t a = w[4 * y][x], b = w[4 * y + 1][x], c = w[4 * y + 2][x], d = w[4 * y + 3][x];
        swap(a, c, 16, 0x0000FFFFu);
        swap(b, d, 16, 0x0000FFFFu);
        swap(a, b, 8, 0x00FF00FFu);
        swap(c, d, 8, 0x00FF00FFu);
        out[4 * x][y] = a;
        out[4 * x + 1][y] = b;
        out[4 * x + 2][y] = c;
        out[4 * x + 3][y] = d;
      }
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int t = t8 + k;
    if (t < g.t_begin || t >= t_end) continue;
    uint32_t* o = wq + (row0 + t) * W + (2 * mt + hf) * (BITS / 4);
    if constexpr (BITS == 4) *o = out[k][0];
    else *reinterpret_cast<uint2*>(o) = make_uint2(out[k][0], out[k][1]);
  }
  for (int x = r; x < 8 * G; x += per) {
    const int k = x / G, t = t8 + k;
    if (t >= g.t_begin && t < t_end) scales(chunk, tib + k, t, x - k * G);
  }
}

// Reference-layout affine rows -> paged chunks (inverse of the code gather).
template <int ESIZE, int BITS>
__global__ void __launch_bounds__(256) scatter_codes_kernel(ScatterCodesArgs a) {
  const int tpr = a.D / 8;
  const int64_t gtid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t row = gtid / tpr;  // (s, h, t)
  const int j = static_cast<int>(gtid % tpr);
  const int64_t total = static_cast<int64_t>(a.n_seqs) * a.H * a.T;
  if (row >= total) return;
  const int64_t t = row % a.T;
  const int64_t h = (row / a.T) % a.H;
  const int64_t s = row / (static_cast<int64_t>(a.T) * a.H);
  const RowDst& d = a.dst;
  const int32_t blk = d.table[s * d.table_stride + t / d.block_size];
  if (blk < 0) return;
  const int tib = static_cast<int>(t % d.block_size);
  uint8_t* chunk = d.base + static_cast<int64_t>(blk) * d.block_bytes + h * d.head_bytes;
  const uint32_t* w = a.wq + row * (a.D * BITS / 32);
  uint32_t code[8];
  if constexpr (BITS == 4) {
    const uint32_t x = w[j];
    for (int i = 0; i < 8; i++) code[i] = (x >> (4 * i)) & 15u;
  } else {
    const uint32_t x0 = w[2 * j], x1 = w[2 * j + 1];
    for (int i = 0; i < 4; i++) {
      code[i] = (x0 >> (8 * i)) & 255u;
      code[4 + i] = (x1 >> (8 * i)) & 255u;
    }
  }
  store_chunk_codes<BITS>(chunk, d, tib, j, a.D, code);
  if ((j * 8) % a.group == 0) {
    const int G = a.D / a.group;
    const int g = j * 8 / a.group;
    const uint8_t* sp = static_cast<const uint8_t*>(a.scales) + (row * G + g) * ESIZE;
    const uint8_t* bp = static_cast<const uint8_t*>(a.biases) + (row * G + g) * ESIZE;
    uint8_t* so = chunk + d.s_off + qsb_index(tib, d.is_v, g, 0, d.G, d.keys_only) * ESIZE;
    uint8_t* bo = chunk + d.s_off + qsb_index(tib, d.is_v, g, 1, d.G, d.keys_only) * ESIZE;
    for (int i = 0; i < ESIZE; i++) {
      so[i] = sp[i];
      bo[i] = bp[i];
    }
  }
}

// ------------------------------------------------------------ copy4d

// A strided 4-D copy in units of the widest aligned run (1 to 16 bytes):
// extents (as divisors that turn a unit's index, below 2^31, into its
// coordinates) and unit strides, outermost first.
struct CopyPlan {
  const void* src;
  void* dst;
  uint32_t total;
  FastDiv n[4];
  int64_t s[4], d[4];
};

// Up to two copies in one launch (blockIdx.y picks one: a cache update
// writes its K and V tokens with one launch), N units a thread, all loaded
// before any is stored.  HBM bound: the copy moves whole 16-byte units where
// runs and strides allow it, with 32-bit index arithmetic, and keeps N loads
// in flight a thread.  Measured against one element a thread with 64-bit
// divisions: 134 MB of f32 rows 126 -> 58 us, 8 x 1023 bf16 rows of 256 dims
// (8.4 MB moved) 9.3 -> 3.7 us.
template <typename U, int N>
__global__ void __launch_bounds__(256) copy_units_kernel(CopyPlan p0, CopyPlan p1) {
  const CopyPlan& p = blockIdx.y ? p1 : p0;
  const U* src = static_cast<const U*>(p.src);
  U* dst = static_cast<U*>(p.dst);
  const uint32_t i0 = blockIdx.x * (256u * N) + threadIdx.x;
  if (i0 >= p.total) return;
  U v[N];
  int64_t to[N];
#pragma unroll
  for (int j = 0; j < N; j++) {
    const uint32_t i = min(i0 + 256u * j, p.total - 1);  // (clamped copies are not stored)
    const uint32_t r3 = p.n[3].quot(i), r2 = p.n[2].quot(r3), r1 = p.n[1].quot(r2);
    const int64_t c3 = i - r3 * p.n[3].n, c2 = r3 - r2 * p.n[2].n, c1 = r2 - r1 * p.n[1].n, c0 = r1;
    to[j] = c0 * p.d[0] + c1 * p.d[1] + c2 * p.d[2] + c3 * p.d[3];
    v[j] = src[c0 * p.s[0] + c1 * p.s[1] + c2 * p.s[2] + c3 * p.s[3]];
  }
#pragma unroll
  for (int j = 0; j < N; j++)
    if (i0 + 256u * j < p.total) dst[to[j]] = v[j];
}

// Whole-block copy across all layers (copy-on-write, prefix store).  The
// (src, dst) pairs travel in the kernel arguments, so no device staging
// buffer has to outlive the launch.
__global__ void __launch_bounds__(256) copy_blocks_kernel(uint8_t* base, int64_t layer_bytes,
                                                          int64_t block_bytes, BlockPairs pairs) {
  const int pair = blockIdx.y;
  const int layer = blockIdx.z;
  const int64_t words = block_bytes / 16;
  const uint4* s = reinterpret_cast<const uint4*>(base + layer * layer_bytes +
                                                  static_cast<int64_t>(pairs.src[pair]) * block_bytes);
  uint4* d = reinterpret_cast<uint4*>(base + layer * layer_bytes +
                                      static_cast<int64_t>(pairs.dst[pair]) * block_bytes);
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < words;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    d[i] = s[i];
}

__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    p[i] = v;
}

// ------------------------------------------------------------ synthetic

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

template <int DT>
__global__ void __launch_bounds__(256) fill_normal_kernel(void* data, int64_t n, uint64_t seed,
                                                          float std) {
  using E = Elem<DT>;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const uint64_t r = splitmix64(seed * 0x100000001B3ull + static_cast<uint64_t>(i));
    const float u1 = (static_cast<float>(r >> 40) + 1.0f) * (1.0f / 16777216.0f);
    const float u2 = static_cast<float>((r >> 16) & 0xFFFFFFu) * (1.0f / 16777216.0f);
    const float z = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
    static_cast<typename E::T*>(data)[i] = E::from_f32(z * std);
  }
}

// ------------------------------------------------------------ attention
//
// Split-K decode attention, one workgroup (256 threads) per (partition,
// kv head, query row).  A workgroup walks its partition in tiles of 32
// tokens: 8 lanes per token form scores for the REP query heads that share
// the kv head (one K read serves all of them), one wave updates the running
// max / sum (online softmax, sdpa_vector.h:116-131), and each thread then
// accumulates P.V for one value dim.  Partials (unnormalised o, max, sum)
// are combined by attn_combine_kernel exactly as sdpa_vector_2pass_2 does
// (sdpa_vector.h:320-394); a single-partition launch normalises in place.
//
// QSEM selects the quantized-SDPA semantics of KVCache.swift:1909-1997:
// queries scaled in T, scores rounded to T, masked scores set to T's lowest
// value (so a fully masked row averages V).  Otherwise MLXFast semantics: queries scaled in
// fp32, masked keys skipped, an empty row yields zeros.
constexpr int kTile = 32;
constexpr int kMaxD = 256;

template <int DT, int BITS, int REP, bool QSEM>
__global__ void __launch_bounds__(256) attn_partial_kernel(AttnArgs a, int h_off, int rep_total) {
  using E = Elem<DT>;
  __shared__ float qs[REP][kMaxD];
  __shared__ float sc[REP][kTile];
  __shared__ float alpha_s[REP];
  __shared__ float red[256 * REP];

  const int tid = threadIdx.x;
  const int part = blockIdx.x;
  const int hk = blockIdx.y;
  const int64_t row = blockIdx.z;  // b * L + l
  const int64_t b = row / a.L;
  const int l = static_cast<int>(row % a.L);
  const int D = a.D, Dv = a.Dv;
  const int64_t T = a.kv.seq_lens ? a.kv.seq_lens[b] : a.kv.T;
  const int64_t t_begin = static_cast<int64_t>(part) * a.part_tokens;
  const int64_t t_end = min<int64_t>(T, t_begin + a.part_tokens);
  const float lowest = -E::kMax;
  const int group = a.group > 0 ? a.group : 64;

  // queries of the REP heads sharing kv head hk
  const float scale_t = QSEM ? round_to<DT>(a.scale) : a.scale;
  for (int i = tid; i < REP * D; i += 256) {
    const int r = i / D, d = i % D;
    const int h = hk * rep_total + h_off + r;
    const float qv = E::load(static_cast<const typename E::T*>(a.q) + b * a.q_sb + h * a.q_sh +
                             static_cast<int64_t>(l) * a.q_sl + d);
    qs[r][d] = QSEM ? round_to<DT>(qv * scale_t) : qv * scale_t;
  }

  // Phase-C thread layout: value dim `vd`, token subset `sub`.
  const int n_sub = max(1, 256 / Dv);
  const int vd = tid % Dv;
  const int sub = tid / Dv;
  const bool c_active = sub < n_sub && tid < n_sub * Dv;
  float o[REP];
#pragma unroll
  for (int r = 0; r < REP; r++) o[r] = 0.0f;
  float m_run = -3.402823466e38f, l_run = 0.0f;  // lanes r < REP of wave 0 own head r
  // an attention sink (MLXFast semantics only) is one more logit with a
  // zero value row, counted once per row (sdpa_vector.h:93-96, :257-260)
  if (!QSEM && a.sinks && part == 0 && tid < REP) {
    m_run = sink_start(load_as<DT>(a.sinks, a.sinks_dtype, hk * rep_total + h_off + tid), m_run);
    l_run = 1.0f;
  }
  __syncthreads();

  for (int64_t t0 = t_begin; t0 < t_end; t0 += kTile) {
    // ---- phase A: scores
    {
      const int tt = tid / 8, lane = tid % 8;
      const int64_t t = t0 + tt;
      float acc[REP];
#pragma unroll
      for (int r = 0; r < REP; r++) acc[r] = 0.0f;
      if (t < t_end) {
        const TokLoc loc = locate(a.kv, b, t);
        for (int d = lane; d < D; d += 8) {
          const float kv = kv_at<DT, BITS>(a.kv, loc, hk, d, 0, group);
#pragma unroll
          for (int r = 0; r < REP; r++) acc[r] = fmaf(qs[r][d], kv, acc[r]);
        }
      }
#pragma unroll
      for (int r = 0; r < REP; r++) acc[r] = wave_sum(acc[r], 8);
      if (lane == 0) {
#pragma unroll
        for (int r = 0; r < REP; r++) {
          // quantized SDPA stores the scores in the dtype (quantizedMM
          // returns T, KVCache.swift:1945-1949) before the mask is applied
          float s = QSEM ? round_to<DT>(acc[r]) : acc[r];
          bool vis = t < t_end;
          if (vis && a.mask_mode != 0) {
            const int h = hk * rep_total + h_off + r;
            if (a.mask_mode == 1) {
              vis = t <= T - a.L + l;
            } else {
              const int64_t mo = b * a.m_sb + h * a.m_sh + l * a.m_sl + t * a.m_st;
              if (a.mask_mode == 2) {
                vis = static_cast<const uint8_t*>(a.mask)[mo] != 0;
              } else if (QSEM) {
                // scores (T) + mask: a T mask keeps the sum in T, an f32
                // mask promotes it to f32 (KVCache.swift:1963-1969)
                const float add = load_f32(a.mask, a.mask_dtype, mo);
                s = a.mask_dtype == DT ? round_to<DT>(s + add) : s + add;
              } else {
                // the mask in the query dtype; keys below its lowest finite
                // value are skipped (sdpa_vector.h:105-121)
                const float add = load_as<DT>(a.mask, a.mask_dtype, mo);
                vis = add >= -E::kMax;
                s += add;
              }
            }
            if (QSEM && !vis && t < t_end) {
              s = lowest;
              vis = true;
            }
          }
          sc[r][tt] = vis ? s : -INFINITY;
        }
      }
    }
    __syncthreads();
    // ---- phase B: online softmax update (wave 0, lane = token in tile)
    if (tid < 64) {
      const int tt = tid & 31;
#pragma unroll
      for (int r = 0; r < REP; r++) {
        const float s = sc[r][tt];
        float tmax = wave_max(tid < 32 ? s : -INFINITY, 64);
        const float m_old = __shfl(m_run, r, 64);
        const float m_new = fmaxf(m_old, tmax);
        const float p = (tid < 32 && s != -INFINITY) ? __expf(s - m_new) : 0.0f;
        const float psum = wave_sum(p, 64);
        const float al = __expf(m_old - m_new);
        if (tid < 32) sc[r][tt] = p;
        if (tid == r) {
          m_run = m_new;
          l_run = l_run * al + psum;
          alpha_s[r] = al;
        }
      }
    }
    __syncthreads();
    // ---- phase C: o = o * alpha + sum_t p_t v_t
    if (c_active) {
#pragma unroll
      for (int r = 0; r < REP; r++) o[r] *= alpha_s[r];
      for (int tt = sub; tt < kTile; tt += n_sub) {
        const int64_t t = t0 + tt;
        if (t >= t_end) break;
        const TokLoc loc = locate(a.kv, b, t);
        const float vv = kv_at<DT, BITS>(a.kv, loc, hk, vd, 1, group);
#pragma unroll
        for (int r = 0; r < REP; r++) o[r] = fmaf(sc[r][tt], vv, o[r]);
      }
    }
    __syncthreads();
  }

  // combine the token subsets of phase C
  if (c_active) {
#pragma unroll
    for (int r = 0; r < REP; r++) red[(r * n_sub + sub) * Dv + vd] = o[r];
  }
  if (tid < REP) {
    qs[tid][0] = m_run;  // reuse: per-head max / sum
    qs[tid][1] = l_run;
  }
  __syncthreads();
  for (int i = tid; i < REP * Dv; i += 256) {
    const int r = i / Dv, d = i % Dv;
    float acc = 0.0f;
    for (int s2 = 0; s2 < n_sub; s2++) acc += red[(r * n_sub + s2) * Dv + d];
    const float m = qs[r][0], lsum = qs[r][1];
    const int h = hk * rep_total + h_off + r;
    if (a.n_parts == 1) {
      const float v = lsum > 0.0f ? acc / lsum : 0.0f;
      static_cast<typename E::T*>(a.out)[b * a.o_sb + h * a.o_sh + static_cast<int64_t>(l) * a.o_sl +
                                         d] = E::from_f32(v);
    } else {
      const int64_t base = ((row * a.Hq + h) * a.n_parts + part);
      a.ws_o[base * Dv + d] = acc;
      if (d == 0) {
        a.ws_ml[base * 2] = m;
        a.ws_ml[base * 2 + 1] = lsum;
      }
    }
  }
}

// One wave per (row, head): lane l merges dims l, l + 64, .. (Dv <= 256).
// The (max, sum) pairs and partial rows of up to NP parts are loaded before
// any is used, so a merge costs one memory round trip per NP parts (NP = 2,
// 4 or 8, the smallest that holds the launch's parts, so few parts load no
// clamped duplicates).
template <int DT, int NP = 8>
__global__ void __launch_bounds__(256) attn_combine_kernel(AttnArgs a, int64_t n_rh) {
  using E = Elem<DT>;
  const int64_t rh = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);  // row * Hq + h
  if (rh >= n_rh) return;
  const int lane = threadIdx.x & 63;
  const int64_t row = rh / a.Hq;
  const int h = static_cast<int>(rh % a.Hq);
  const int64_t b = row / a.L;
  const int l = static_cast<int>(row % a.L);
  const float* ml = a.ws_ml + rh * a.n_parts * 2;
  const float* wo = a.ws_o + rh * a.n_parts * a.Dv;
  float M = -3.402823466e38f, den = 0.0f;
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int c = 0; c < a.n_parts; c += NP) {
    float m[NP], ls[NP], v[NP][4];
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const int p = min(c + j, a.n_parts - 1);  // (clamped slots are selected away)
      m[j] = ml[2 * p];
      ls[j] = ml[2 * p + 1];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int d = lane + 64 * i;
        v[j][i] = d < a.Dv ? wo[static_cast<int64_t>(p) * a.Dv + d] : 0.0f;
      }
    }
    float Mc = M;
#pragma unroll
    for (int j = 0; j < NP; j++)
      if (c + j < a.n_parts) Mc = fmaxf(Mc, m[j]);
    const float r = __expf(M - Mc);
    den *= r;
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] *= r;
    M = Mc;
#pragma unroll
    for (int j = 0; j < NP; j++) {
      if (c + j < a.n_parts) {
        const float w = __expf(m[j] - M);
        den += w * ls[j];
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = fmaf(w, v[j][i], acc[i]);
      }
    }
  }
  typename E::T* out = static_cast<typename E::T*>(a.out) + b * a.o_sb + h * a.o_sh +
                       static_cast<int64_t>(l) * a.o_sl;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int d = lane + 64 * i;
    if (d < a.Dv) out[d] = E::from_f32(den > 0.0f ? acc[i] / den : 0.0f);
  }
}

// The same merge for launches with few (row, head)s: one wave per (row,
// head, 64 dims), lane l merging dim 64 c + l, the (max, sum) pairs and
// partials of up to 32 parts loaded before any is used (the pairs are the
// same for the whole wave, so they load through the scalar path): four
// times the waves and one memory round trip per 32 parts.
template <int DT>
__global__ void __launch_bounds__(64) attn_combine_narrow_kernel(AttnArgs a, int64_t n_rh) {
  using E = Elem<DT>;
  const int nch = (a.Dv + 63) / 64;
  const int64_t rh = blockIdx.x / nch;  // row * Hq + h
  if (rh >= n_rh) return;
  const int d = 64 * static_cast<int>(blockIdx.x % nch) + threadIdx.x;
  const bool dv = d < a.Dv;
  const int64_t row = rh / a.Hq;
  const int h = static_cast<int>(rh % a.Hq);
  const int64_t b = row / a.L;
  const int l = static_cast<int>(row % a.L);
  const float* ml = a.ws_ml + rh * a.n_parts * 2;
  const float* wo = a.ws_o + rh * a.n_parts * a.Dv + (dv ? d : 0);
  float M = -3.402823466e38f, den = 0.0f, acc = 0.0f;
  for (int c = 0; c < a.n_parts; c += 32) {
    float m[32], ls[32], v[32];
#pragma unroll
    for (int j = 0; j < 32; j++) {
      const int p = min(c + j, a.n_parts - 1);  // (clamped slots are selected away)
      m[j] = ml[2 * p];
      ls[j] = ml[2 * p + 1];
      v[j] = wo[static_cast<int64_t>(p) * a.Dv];
    }
    float Mc = M;
#pragma unroll
    for (int j = 0; j < 32; j++)
      if (c + j < a.n_parts) Mc = fmaxf(Mc, m[j]);
    const float r = __expf(M - Mc);
    den *= r;
    acc *= r;
    M = Mc;
#pragma unroll
    for (int j = 0; j < 32; j++) {
      if (c + j < a.n_parts) {
        const float w = __expf(m[j] - M);
        den += w * ls[j];
        acc = fmaf(w, v[j], acc);
      }
    }
  }
  if (dv) {
    typename E::T* out = static_cast<typename E::T*>(a.out) + b * a.o_sb + h * a.o_sh +
                         static_cast<int64_t>(l) * a.o_sl;
    out[d] = E::from_f32(den > 0.0f ? acc / den : 0.0f);
  }
}

// ------------------------------------------------------------ launchers

static inline unsigned blocks_for(int64_t threads) {
  return static_cast<unsigned>((threads + 255) / 256);
}

template <int DT>
static void quantize_dispatch(int bits, int group, int mode, const RowSrc& src, const RowDst& dst,
                              int64_t rows, int D, hipStream_t st) {
  const unsigned nb = blocks_for(rows * (D / 8));
#define VKV_Q(B, G, M) \
  hipLaunchKernelGGL((quantize_rows_kernel<DT, B, G, M>), dim3(nb), dim3(256), 0, st, src, dst, rows, D)
#define VKV_QM(B, G) \
  do { if (mode == 0) VKV_Q(B, G, 0); else VKV_Q(B, G, 1); } while (0)
#define VKV_QG(B)                               \
  do {                                          \
    if (group == 32) VKV_QM(B, 32);             \
    else if (group == 64) VKV_QM(B, 64);        \
    else if (group == 128) VKV_QM(B, 128);      \
    else throw Error("group_size must be 32, 64 or 128"); \
  } while (0)
  if (bits == 4) VKV_QG(4);
  else if (bits == 8) VKV_QG(8);
  else throw Error("bits must be 4 or 8");
#undef VKV_QG
#undef VKV_QM
#undef VKV_Q
}

void launch_quantize_rows(int dtype, int bits, int group, int mode, const RowSrc& src,
                          const RowDst& dst, int64_t rows, int D, hipStream_t st) {
  if (rows <= 0) return;
  VKV_CHECK(D % group == 0 && D % 8 == 0, "last dim must be a multiple of group_size");
  switch (dtype) {
    case kF32: quantize_dispatch<kF32>(bits, group, mode, src, dst, rows, D, st); break;
    case kF16: quantize_dispatch<kF16>(bits, group, mode, src, dst, rows, D, st); break;
    case kBF16: quantize_dispatch<kBF16>(bits, group, mode, src, dst, rows, D, st); break;
    default: throw Error("unsupported dtype");
  }
  VKV_HIP(hipGetLastError());
}

template <int DT>
static void append_dispatch(int bits, int group, const RowSrc& sk, const RowSrc& sv, const RowDst& dk,
                            const RowDst& dv, int64_t ntok, int H, int D, bool with_v, hipStream_t st) {
  const int hb = 256 / D;
  const dim3 grid(static_cast<unsigned>((ntok + 7) / 8), (H + hb - 1) / hb, with_v ? 2 : 1);
  const AppendDiv dq{fast_div(sk.e1), fast_div(dk.block_size)};
  const TimedLaunch tl = timing_prepare(kTimeAppend);
#define VKV_A(B, G)                                                                            \
  hipExtLaunchKernelGGL((append_affine_kernel<DT, B, G>), grid, dim3(256), 0, st, tl.start, tl.stop, \
                        0, sk, sv, dk, dv, static_cast<uint32_t>(ntok), H, D, dq)
#define VKV_AG(B)                         \
  do {                                    \
    if (group == 32) VKV_A(B, 32);        \
    else if (group == 64) VKV_A(B, 64);   \
    else VKV_A(B, 128);                   \
  } while (0)
  if (bits == 4) VKV_AG(4);
  else VKV_AG(8);
#undef VKV_AG
#undef VKV_A
  VKV_HIP(hipGetLastError());
  timing_commit(tl);
}

bool append_affine_supported(int bits, int group, int D) {
  return (bits == 4 || bits == 8) && (group == 32 || group == 64 || group == 128) && D % group == 0 &&
         (D == 32 || D == 64 || D == 128 || D == 256);
}

void launch_append_affine(int dtype, int bits, int group, const RowSrc& sk, const RowSrc& sv,
                          const RowDst& dk, const RowDst& dv, int64_t ntok, int H, int D, bool with_v,
                          hipStream_t st) {
  if (ntok <= 0) return;
  VKV_CHECK(append_affine_supported(bits, group, D), "append_affine: unsupported geometry");
  // (a table's batch rows are the source's; both matrices share the tokens)
  VKV_CHECK(ntok < (int64_t{1} << 31) && sk.e1 > 0 && sv.e1 == sk.e1 &&
                (dk.slots || (dk.seq_S == sk.e1 && dk.start + sk.e1 < (int64_t{1} << 31))),
            "append_affine: token range");
  switch (dtype) {
    case kF32: append_dispatch<kF32>(bits, group, sk, sv, dk, dv, ntok, H, D, with_v, st); break;
    case kF16: append_dispatch<kF16>(bits, group, sk, sv, dk, dv, ntok, H, D, with_v, st); break;
    case kBF16: append_dispatch<kBF16>(bits, group, sk, sv, dk, dv, ntok, H, D, with_v, st); break;
    default: throw Error("unsupported dtype");
  }
  VKV_HIP(hipGetLastError());
}

void launch_append_rows(int dtype, const RowSrc& sk, const RowSrc& sv, const RowDst& dk,
                        const RowDst& dv, int64_t ntok, int64_t H, int Dk, int Dv, hipStream_t st) {
  if (ntok <= 0 || H <= 0) return;
  const int es = elem_bytes(dtype);
  auto whole = [](int64_t x) { return x % 16 == 0; };
  auto vec = [&](const RowSrc& s, const RowDst& d, int D) {
    return whole(static_cast<int64_t>(reinterpret_cast<uintptr_t>(s.ptr))) && whole(s.s1 * es) &&
           whole(s.s2 * es) && whole(static_cast<int64_t>(reinterpret_cast<uintptr_t>(d.base))) &&
           whole(d.block_bytes) && whole(d.head_bytes) && whole(d.c_off) &&
           whole(static_cast<int64_t>(D) * es);
  };
  const bool v = vec(sk, dk, Dk) && vec(sv, dv, Dv);
  const int64_t per = H * ((static_cast<int64_t>(std::max(Dk, Dv)) * es + 15) / 16);
  const int64_t most = std::max<int64_t>(1, ((int64_t{1} << 31) - 256) / per);  // tokens a launch
  for (int64_t t0 = 0; t0 < ntok; t0 += most) {
    const int64_t n = std::min(most, ntok - t0);
    const dim3 grid(blocks_for(n * per), 2);
    const uint32_t rows = static_cast<uint32_t>(n * H);
    auto run = [&](auto E_, auto V_) {
      hipLaunchKernelGGL((append_rows_kernel<decltype(E_)::value, decltype(V_)::value>), grid,
                         dim3(256), 0, st, sk, sv, dk, dv, t0, rows, Dk, Dv);
    };
    using std::integral_constant;
    if (es == 2 && v) run(integral_constant<int, 2>{}, std::true_type{});
    else if (es == 2) run(integral_constant<int, 2>{}, std::false_type{});
    else if (v) run(integral_constant<int, 4>{}, std::true_type{});
    else run(integral_constant<int, 4>{}, std::false_type{});
    VKV_HIP(hipGetLastError());
  }
}

void launch_dequantize(int dtype, int bits, int group, const uint32_t* wq, const void* scales,
                       const void* biases, void* out, int64_t rows, int D, hipStream_t st) {
  if (rows <= 0) return;
  VKV_CHECK(D % group == 0 && group % 8 == 0, "last dim must be a multiple of group_size");
  const unsigned nb = blocks_for(rows * (D / 8));
#define VKV_DQ(DT, B) \
  hipLaunchKernelGGL((dequantize_kernel<DT, B>), dim3(nb), dim3(256), 0, st, wq, scales, biases, out, rows, D, group)
#define VKV_DQB(DT) do { if (bits == 4) VKV_DQ(DT, 4); else if (bits == 8) VKV_DQ(DT, 8); else throw Error("bits must be 4 or 8"); } while (0)
  switch (dtype) {
    case kF32: VKV_DQB(kF32); break;
    case kF16: VKV_DQB(kF16); break;
    case kBF16: VKV_DQB(kBF16); break;
    default: throw Error("unsupported dtype");
  }
#undef VKV_DQB
#undef VKV_DQ
  VKV_HIP(hipGetLastError());
}

// Whether gather_dequant8_kernel's vector accesses fit the view.
static bool gather8_ok(const GatherArgs& g) {
  if (g.D % 8 || g.group % 8 || reinterpret_cast<uintptr_t>(g.out) % 16 ||
      reinterpret_cast<uintptr_t>(g.out_v) % 16)
    return false;
  const auto a4 = [](int64_t x) { return x % 4 == 0; };
  const KVSrc& kv = g.kv;
  if (kv.qfmt)
    return a4(static_cast<int64_t>(reinterpret_cast<uintptr_t>(kv.base))) && a4(kv.block_bytes) &&
           a4(kv.head_bytes) && a4(kv.kc_off) && a4(kv.vc_off) && kv.head_bytes < (int64_t{1} << 31);
  for (int which = 0; which < 2; which++) {
    if (which != g.which && !g.out_v) continue;
    const Comp& c = which ? kv.vc : kv.kc;
    if (!(a4(static_cast<int64_t>(reinterpret_cast<uintptr_t>(c.ptr))) && a4(c.sb) && a4(c.sh) &&
          a4(c.st)))
      return false;
  }
  return true;
}

template <int DT, int BITS>
static void gather_dispatch_kind(const GatherArgs& g, int out_kind, hipStream_t st) {
  const unsigned nb = blocks_for(static_cast<int64_t>(g.n_seqs) * g.H * g.T * ((g.D + 7) / 8));
  if (out_kind == 0) {
    if constexpr (BITS > 0) {
      const int64_t planes = static_cast<int64_t>(g.n_seqs) * g.H;
      const int64_t per_plane = static_cast<int64_t>(g.T) * (g.D / 8);
      if (gather8_ok(g) && planes > 0 && planes <= 65535 && per_plane > 0 && per_plane < (1 << 30)) {
        const dim3 grid(static_cast<unsigned>((per_plane + 255) / 256), static_cast<unsigned>(planes),
                        g.out_v ? 2u : 1u);
        hipLaunchKernelGGL((gather_dequant8_kernel<DT, BITS>), grid, dim3(256), 0, st, g,
                           fast_div(g.D / 8), fast_div(g.kv.block_size > 0 ? g.kv.block_size : 1),
                           fast_div(g.group / 8));
        return;
      }
    }
    if (g.out_v) {  // element-wise kernel: one launch per matrix
      GatherArgs one = g;
      one.out_v = nullptr;
      for (int which = 0; which < 2; which++) {
        one.which = which;
        one.out = which ? g.out_v : g.out;
        hipLaunchKernelGGL((gather_kernel<DT, BITS, 0>), dim3(nb), dim3(256), 0, st, one);
      }
      return;
    }
    hipLaunchKernelGGL((gather_kernel<DT, BITS, 0>), dim3(nb), dim3(256), 0, st, g);
  } else {
    if constexpr (BITS > 0) {
      // paged chunks take whole words; other layouts (tuples, the values of a
      // keys-only view, outputs off 16 bytes) go code by code
      const int64_t planes = static_cast<int64_t>(g.n_seqs) * g.H;
      const int64_t groups = (static_cast<int64_t>(g.T) + (g.t_begin & 7) + 7) / 8;
      const int64_t threads =
          g.which ? groups * (g.D / 8) : static_cast<int64_t>(g.T) * (g.D * BITS / 128);
      if (g.kv.qfmt && g.kv.table && !(g.which && g.kv.keys_only) && g.D == g.kv.D && g.D % 32 == 0 &&
          planes <= 65535 && threads < (1 << 30) && reinterpret_cast<uintptr_t>(g.out) % 16 == 0) {
        hipLaunchKernelGGL((gather_codes_kernel<DT, BITS>),
                           dim3(blocks_for(threads), static_cast<unsigned>(planes)), dim3(256), 0, st, g);
        return;
      }
      hipLaunchKernelGGL((gather_kernel<DT, BITS, 1>), dim3(nb), dim3(256), 0, st, g);
    } else {
      throw Error("code gather needs an affine view");
    }
  }
}

template <int DT>
static void gather_dispatch(const GatherArgs& g, int out_kind, hipStream_t st) {
  if (g.bits == 0) gather_dispatch_kind<DT, 0>(g, out_kind, st);
  else if (g.bits == 4) gather_dispatch_kind<DT, 4>(g, out_kind, st);
  else if (g.bits == 8) gather_dispatch_kind<DT, 8>(g, out_kind, st);
  else throw Error("bits must be 0, 4 or 8");
}

void launch_gather(const GatherArgs& g, int out_kind, hipStream_t st) {
  if (static_cast<int64_t>(g.n_seqs) * g.H * g.T == 0) return;
  switch (g.dtype) {
    case kF32: gather_dispatch<kF32>(g, out_kind, st); break;
    case kF16: gather_dispatch<kF16>(g, out_kind, st); break;
    case kBF16: gather_dispatch<kBF16>(g, out_kind, st); break;
    default: throw Error("unsupported dtype");
  }
  VKV_HIP(hipGetLastError());
}

void launch_scatter_codes(const ScatterCodesArgs& a, hipStream_t st) {
  const int64_t rows = static_cast<int64_t>(a.n_seqs) * a.H * a.T;
  if (rows <= 0) return;
  const unsigned nb = blocks_for(rows * (a.D / 8));
  const int es = elem_bytes(a.dtype);
  if (a.bits == 4 && es == 2) hipLaunchKernelGGL((scatter_codes_kernel<2, 4>), dim3(nb), dim3(256), 0, st, a);
  else if (a.bits == 4) hipLaunchKernelGGL((scatter_codes_kernel<4, 4>), dim3(nb), dim3(256), 0, st, a);
  else if (a.bits == 8 && es == 2) hipLaunchKernelGGL((scatter_codes_kernel<2, 8>), dim3(nb), dim3(256), 0, st, a);
  else if (a.bits == 8) hipLaunchKernelGGL((scatter_codes_kernel<4, 8>), dim3(nb), dim3(256), 0, st, a);
  else throw Error("bits must be 4 or 8");
  VKV_HIP(hipGetLastError());
}

namespace {
// The copy with its unit dims dropped and dims that are contiguous on both
// sides joined.
Copy4D collapse(const Copy4D& c) {
  Copy4D r = c;
  int m = 0;  // dims kept, innermost first
  int64_t n[4], s[4], d[4];
  for (int i = 3; i >= 0; i--) {
    if (c.n[i] == 1) continue;
    if (m > 0 && c.s[i] == s[m - 1] * n[m - 1] && c.d[i] == d[m - 1] * n[m - 1]) {
      n[m - 1] *= c.n[i];
    } else {
      n[m] = c.n[i];
      s[m] = c.s[i];
      d[m] = c.d[i];
      m++;
    }
  }
  for (int k = 0; k < 4; k++) {
    r.n[3 - k] = k < m ? n[k] : 1;
    r.s[3 - k] = k < m ? s[k] : k == 0;
    r.d[3 - k] = k < m ? d[k] : k == 0;
  }
  return r;
}

// The widest unit (bytes) both sides of a collapsed copy are whole in.
int copy_unit(int es, const Copy4D& c) {
  if (c.s[3] != 1 || c.d[3] != 1) return es;
  int u = 16;
  auto whole = [&](int64_t x) { return x % u == 0; };
  for (; u > es; u /= 2) {
    bool ok = whole(c.n[3] * es) && whole(static_cast<int64_t>(reinterpret_cast<uintptr_t>(c.src))) &&
              whole(static_cast<int64_t>(reinterpret_cast<uintptr_t>(c.dst)));
    for (int i = 0; ok && i < 3; i++) ok = whole(c.s[i] * es) && whole(c.d[i] * es);
    if (ok) break;
  }
  return u;
}

CopyPlan copy_plan(const Copy4D& c, int es, int unit) {
  CopyPlan p{};
  p.src = c.src;
  p.dst = c.dst;
  const int64_t k = unit / es;
  int64_t total = 1;
  for (int i = 0; i < 4; i++) {
    const bool inner = i == 3;
    const int64_t n = inner ? c.n[i] / k : c.n[i];
    p.n[i] = fast_div(n);
    p.s[i] = inner ? c.s[i] : c.s[i] / k;
    p.d[i] = inner ? c.d[i] : c.d[i] / k;
    total *= n;
  }
  p.total = static_cast<uint32_t>(total);
  return p;
}

template <int N>
void launch_copy_units(int unit, const CopyPlan& p0, const CopyPlan& p1, const dim3& grid,
                       hipStream_t st) {
  switch (unit) {
    case 1: hipLaunchKernelGGL((copy_units_kernel<uint8_t, N>), grid, dim3(256), 0, st, p0, p1); break;
    case 2: hipLaunchKernelGGL((copy_units_kernel<uint16_t, N>), grid, dim3(256), 0, st, p0, p1); break;
    case 4: hipLaunchKernelGGL((copy_units_kernel<uint32_t, N>), grid, dim3(256), 0, st, p0, p1); break;
    case 8: hipLaunchKernelGGL((copy_units_kernel<uint64_t, N>), grid, dim3(256), 0, st, p0, p1); break;
    default: hipLaunchKernelGGL((copy_units_kernel<uint4, N>), grid, dim3(256), 0, st, p0, p1);
  }
  VKV_HIP(hipGetLastError());
}

// n copies (1 or 2); copies of 2^31 units or more go in halves of their
// longest dim.
void launch_copies(int es, const Copy4D* c, int n, hipStream_t st) {
  if (es != 1 && es != 2 && es != 4) throw Error("copy4d: element size must be 1, 2 or 4");
  Copy4D r[2];
  CopyPlan p[2];
  int unit = 16, m = 0;
  for (int i = 0; i < n; i++) {
    int64_t total = 1;
    for (int k = 0; k < 4; k++) total *= std::max<int64_t>(0, c[i].n[k]);
    if (total == 0) continue;
    if (total >= int64_t{1} << 31) {
      int big = 0;
      for (int k = 1; k < 4; k++)
        if (c[i].n[k] > c[i].n[big]) big = k;
      Copy4D h = c[i];
      const int64_t half = h.n[big] / 2;
      h.n[big] = half;
      launch_copies(es, &h, 1, st);
      h.n[big] = c[i].n[big] - half;
      h.src = static_cast<const uint8_t*>(h.src) + half * h.s[big] * es;
      h.dst = static_cast<uint8_t*>(h.dst) + half * h.d[big] * es;
      launch_copies(es, &h, 1, st);
      continue;
    }
    r[m] = collapse(c[i]);
    unit = std::min(unit, copy_unit(es, r[m]));
    m++;
  }
  if (m == 0) return;
  uint32_t most = 0;
  for (int i = 0; i < m; i++) {
    p[i] = copy_plan(r[i], es, unit);
    most = std::max(most, p[i].total);
  }
  if (m == 1) p[1] = p[0];
  // four units a thread once that leaves every CU eight workgroups
  constexpr int kN = 4;
  if (most >= 256u * kN * 2048u)
    launch_copy_units<kN>(unit, p[0], p[1], dim3((most + 256u * kN - 1) / (256u * kN), m), st);
  else
    launch_copy_units<1>(unit, p[0], p[1], dim3((most + 255u) / 256u, m), st);
}
}  // namespace

void launch_copy4d(int esize, const void* src, const int64_t* n, const int64_t* s, void* dst,
                   const int64_t* d, hipStream_t st) {
  Copy4D c;
  c.src = src;
  c.dst = dst;
  for (int i = 0; i < 4; i++) {
    c.n[i] = n[i];
    c.s[i] = s[i];
    c.d[i] = d[i];
  }
  launch_copies(esize, &c, 1, st);
}

void launch_copy4d_pair(int esize, const Copy4D& c0, const Copy4D& c1, hipStream_t st) {
  const Copy4D c[2] = {c0, c1};
  launch_copies(esize, c, 2, st);
}

void launch_copy_blocks(const uint8_t* base, int64_t layer_bytes, int n_layers, int64_t block_bytes,
                        const int32_t* src, const int32_t* dst, int n, hipStream_t st) {
  VKV_CHECK(block_bytes % 16 == 0, "block bytes must be a multiple of 16");
  const unsigned gx = static_cast<unsigned>(std::min<int64_t>((block_bytes / 16 + 255) / 256, 64));
  for (int done = 0; done < n; done += BlockPairs::kMax) {
    BlockPairs bp;
    const int cnt = std::min(n - done, BlockPairs::kMax);
    for (int i = 0; i < cnt; i++) {
      bp.src[i] = src[done + i];
      bp.dst[i] = dst[done + i];
    }
    hipLaunchKernelGGL(copy_blocks_kernel, dim3(gx, cnt, n_layers), dim3(256), 0, st,
                       const_cast<uint8_t*>(base), layer_bytes, block_bytes, bp);
    VKV_HIP(hipGetLastError());
  }
}

void launch_fill_i32(int32_t* p, int64_t n, int32_t v, hipStream_t st) {
  if (n <= 0) return;
  const unsigned nb = static_cast<unsigned>(std::min<int64_t>((n + 255) / 256, 4096));
  hipLaunchKernelGGL(fill_i32_kernel, dim3(nb), dim3(256), 0, st, p, n, v);
  VKV_HIP(hipGetLastError());
}

void launch_fill_normal(int dtype, void* data, int64_t n, uint64_t seed, float std, hipStream_t st) {
  if (n <= 0) return;
  const unsigned nb = static_cast<unsigned>(std::min<int64_t>((n + 255) / 256, 1 << 16));
  switch (dtype) {
    case kF32: hipLaunchKernelGGL((fill_normal_kernel<kF32>), dim3(nb), dim3(256), 0, st, data, n, seed, std); break;
    case kF16: hipLaunchKernelGGL((fill_normal_kernel<kF16>), dim3(nb), dim3(256), 0, st, data, n, seed, std); break;
    case kBF16: hipLaunchKernelGGL((fill_normal_kernel<kBF16>), dim3(nb), dim3(256), 0, st, data, n, seed, std); break;
    default: throw Error("unsupported dtype");
  }
  VKV_HIP(hipGetLastError());
}

template <int DT, int BITS, bool QSEM>
static void attn_dispatch_rep(const AttnArgs& a, int64_t rows, hipStream_t st) {
  const int rep = a.Hq / a.Hkv;
  dim3 grid(a.n_parts, a.Hkv, static_cast<unsigned>(rows));
  int done = 0;
  while (done < rep) {
    const int left = rep - done;
    const int chunk = left >= 8 ? 8 : left >= 4 ? 4 : left >= 2 ? 2 : 1;
#define VKV_A(R) \
  hipLaunchKernelGGL((attn_partial_kernel<DT, BITS, R, QSEM>), grid, dim3(256), 0, st, a, done, rep)
    if (chunk == 8) VKV_A(8);
    else if (chunk == 4) VKV_A(4);
    else if (chunk == 2) VKV_A(2);
    else VKV_A(1);
#undef VKV_A
    done += chunk;
  }
  if (a.n_parts > 1) {
    const int64_t n_rh = rows * a.Hq;
    hipLaunchKernelGGL((attn_combine_kernel<DT>), dim3(static_cast<unsigned>((n_rh + 3) / 4)),
                       dim3(256), 0, st, a, n_rh);
  }
}

template <int DT>
static void attn_dispatch(int bits, bool qsem, const AttnArgs& a, int64_t rows, hipStream_t st) {
  if (bits == 0) {
    if (qsem) throw Error("quantized semantics need an affine cache");
    attn_dispatch_rep<DT, 0, false>(a, rows, st);
  } else if (bits == 4) {
    attn_dispatch_rep<DT, 4, true>(a, rows, st);
  } else if (bits == 8) {
    attn_dispatch_rep<DT, 8, true>(a, rows, st);
  } else {
    throw Error("bits must be 0, 4 or 8");
  }
}

void launch_attn_combine(int dtype, const AttnArgs& a, int64_t rows, hipStream_t st) {
  if (a.Dv > 256) throw Error("attention merge supports value dims up to 256");
  const int64_t n_rh = rows * a.Hq;
  const int64_t nch = (a.Dv + 63) / 64;
  if (n_rh * nch <= 2048) {
    // few (row, head)s: the narrow merge's waves fit the chip at once
    const dim3 g(static_cast<unsigned>(n_rh * nch));
    switch (dtype) {
      case kF32: hipLaunchKernelGGL((attn_combine_narrow_kernel<kF32>), g, dim3(64), 0, st, a, n_rh); break;
      case kF16: hipLaunchKernelGGL((attn_combine_narrow_kernel<kF16>), g, dim3(64), 0, st, a, n_rh); break;
      case kBF16: hipLaunchKernelGGL((attn_combine_narrow_kernel<kBF16>), g, dim3(64), 0, st, a, n_rh); break;
      default: throw Error("unsupported dtype");
    }
    VKV_HIP(hipGetLastError());
    return;
  }
  const dim3 grid(static_cast<unsigned>((n_rh + 3) / 4));
  const int np = a.n_parts <= 2 ? 2 : a.n_parts <= 4 ? 4 : 8;
#define VKV_C(T, N) hipLaunchKernelGGL((attn_combine_kernel<T, N>), grid, dim3(256), 0, st, a, n_rh)
#define VKV_CD(T)                   \
  do {                              \
    if (np == 2) VKV_C(T, 2);       \
    else if (np == 4) VKV_C(T, 4);  \
    else VKV_C(T, 8);               \
  } while (0)
  switch (dtype) {
    case kF32: VKV_CD(kF32); break;
    case kF16: VKV_CD(kF16); break;
    case kBF16: VKV_CD(kBF16); break;
    default: throw Error("unsupported dtype");
  }
#undef VKV_CD
#undef VKV_C
  VKV_HIP(hipGetLastError());
}

void launch_attention(int dtype, int bits, int group, bool quant_semantics,
                      const AttnArgs& a, int64_t rows, hipStream_t st) {
  if (rows <= 0) return;
  VKV_CHECK(a.D <= kMaxD && a.Dv <= kMaxD, "head dims above 256 are not supported here");
  VKV_CHECK(a.Hq % a.Hkv == 0, "query heads must be a multiple of kv heads");
  VKV_CHECK(bits == 0 || group == 32 || group == 64 || group == 128,
            "affine attention supports group_size 32, 64 or 128");
  VKV_CHECK(bits == 0 || a.group == group, "the attention arguments carry another group size");
  switch (dtype) {
    case kF32: attn_dispatch<kF32>(bits, quant_semantics, a, rows, st); break;
    case kF16: attn_dispatch<kF16>(bits, quant_semantics, a, rows, st); break;
    case kBF16: attn_dispatch<kBF16>(bits, quant_semantics, a, rows, st); break;
    default: throw Error("unsupported dtype");
  }
  VKV_HIP(hipGetLastError());
}

}  // namespace vkv
