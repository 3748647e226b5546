// vkv_tq.hip -- the TurboQuant KV codec on the device
// (Libraries/MLXLMCommon/TurboQuant/TQEncoder.swift, TQHadamard.swift,
// TQCodebook.swift, TQQJL.swift, TQBitPack.swift).
//
// Encode (keys or values): per vector, the norm in the input dtype T, the
// unit vector in T, the randomized blockwise Hadamard rotation (f32), the
// Lloyd-Max code of every coordinate and, for keys, the residual's norm and
// the signs of its projection through the QJL matrix; codes and signs are
// packed into the reference's flat u32 words (value e of the tensor in word
// e / (32 / bits) at bit (e % (32 / bits)) * bits).  Decode: codebook
// lookup, the QJL correction sqrt(pi/2)/d * |r| * (signs . S) for keys, the
// inverse rotation, times the stored norm, to f16, written straight into the
// cache's unified buffer (f16 or f32) at the vector's token position.
//
// A workgroup of 256 threads takes tiles of 32 vectors.  Head dims 64, 128
// and 256 (one Hadamard block) take the row kernels, which keep each vector
// in the registers of eight lanes (tq_encode_rows / tq_decode_rows); other
// dims take the tile kernels, which stage the tile in LDS.  The two matrix
// products run as f32 fused multiply-add chains in index order (on the f32
// matrix cores in the row kernels), the row sums in double; the same orders
// are what the CPU restatement fixes, so the codes, signs, norms and decoded
// values are bit-exact with it.  Contraction is off in
// this file: every other product and sum rounds as the reference writes it.
#include <hip/hip_ext.h>

#include <algorithm>
#include <type_traits>

#include "vkv_device.h"
#include "vkv_internal.h"

#pragma clang fp contract(off)

namespace vkv {
namespace {

constexpr int kRows = kTqTileRows;
constexpr int kThreads = 256;
static_assert(kRows * 8 == kThreads, "row sums use eight lanes per row");

// f16 of an f32 value that is first rounded to f32: the barrier keeps the
// compiler from folding the product or sum that made v into a mixed
// precision fma that rounds once, straight to f16 (v_fma_mix*).
__device__ __forceinline__ uint16_t f16_of(float v) {
  asm volatile("" : "+v"(v));
  return f32_to_f16(v);
}

__device__ __forceinline__ float round_dt(float v, int dt) {
  if (dt == kF16) return f16_to_f32(f16_of(v));
  if (dt == kBF16) return bf16_to_f32(f32_to_bf16(v));
  return v;
}

// round_dt of a pair for a dtype known at compile time: bf16 by the packed
// hardware conversion (round to nearest even, as f32_to_bf16).
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
template <int DT>
__device__ __forceinline__ void round_pair(float& a, float& b) {
  if constexpr (DT == kBF16) {
    const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
    a = __uint_as_float(w << 16);
    b = __uint_as_float(w & 0xFFFF0000u);
  } else if constexpr (DT == kF16) {
    a = f16_to_f32(f16_of(a));
    b = f16_to_f32(f16_of(b));
  }
}
template <int DT>
__device__ __forceinline__ float round_one(float v) {
  float b = 0.0f;
  round_pair<DT>(v, b);
  return v;
}

// Sum over the 8 lanes of an aligned lane group (every lane gets it).
__device__ __forceinline__ double group8_sum_d(double v) {
  v += __shfl_xor(v, 1);
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 4);
  return v;
}

// The blockwise butterfly of TQHadamard.hadamardTransform over a tile of
// `rows` vectors held in LDS (row stride D): every block (n = 2^L values)
// runs its stages (a + b, a - b) on pairs (g 2h + j, g 2h + h + j), then
// scales by its f32 1 / sqrt(n).  Block sizes are powers of two, so every
// index below is a shift or a mask.
__device__ void hadamard_tile(float* y, int rows, int D, const TqBlocks& bl) {
  const int tid = threadIdx.x;
  for (int b = 0; b < bl.n; ++b) {
    const int n = bl.size[b], off = bl.off[b];
    const int L = __builtin_ctz(n);
    if (L == 0) continue;  // a block of one value: the transform is the identity
    for (int s = 0; s < L; ++s) {
      __syncthreads();
      const int h = 1 << s;
      for (int p = tid; p < (rows << (L - 1)); p += kThreads) {
        const int r = p >> (L - 1), q = p & ((1 << (L - 1)) - 1);
        float* v = y + r * D + off + ((q >> s) << (s + 1)) + (q & (h - 1));
        const float a = v[0], c = v[h];
        v[0] = a + c;
        v[h] = a - c;
      }
    }
    __syncthreads();
    const float sc = bl.scale[b];
    for (int p = tid; p < (rows << L); p += kThreads) {
      float* v = y + (p >> L) * D + off + (p & (n - 1));
      *v = *v * sc;
    }
  }
  __syncthreads();
}

// Packs the tile's values (u8, tile element k = flat element e0 + k) into
// the flat words of `bits` each.  Words wholly inside the tile are stored;
// the (at most two) words it shares with a neighbouring tile are OR-ed into
// the zeroed output.
__device__ void pack_tile(const uint8_t* vals, int64_t e0, int64_t e1, int64_t total, int bits,
                          uint32_t* out) {
  const int vpw = 32 / bits;
  const int64_t w0 = e0 / vpw, w1 = (e1 - 1) / vpw;
  for (int64_t w = w0 + threadIdx.x; w <= w1; w += kThreads) {
    uint32_t word = 0;
    for (int k = 0; k < vpw; ++k) {
      const int64_t e = w * vpw + k;
      if (e >= e0 && e < e1) word |= static_cast<uint32_t>(vals[e - e0]) << (k * bits);
    }
    const int64_t end = (w + 1) * vpw < total ? (w + 1) * vpw : total;
    if (w * vpw >= e0 && end <= e1)
      out[w] = word;
    else if (word)
      atomicOr(out + w, word);
  }
}

// sum_i a[r][i] * M[i * D + j], an f32 fma chain in i order, for the tile's
// rows below `rows`, handed to f(r, j, sum); a(r, i) reads the left operand.
// f must not write the operands.
template <class A, class F>
__device__ void tile_matmul(A&& a, int rows, int D, const float* M, F&& f) {
  for (int p = threadIdx.x; p < rows * D; p += kThreads) {
    const int r = p / D, j = p - r * D;
    float acc = 0.0f;
    for (int i = 0; i < D; ++i) acc = fmaf(a(r, i), M[static_cast<int64_t>(i) * D + j], acc);
    f(r, j, acc);
  }
  __syncthreads();
}

// The codec's tables in LDS: rotation signs, levels and boundaries.
struct TqLds {
  float signs[256];
  float cb[256];
  float bnd[256];
};

__device__ void load_tables(TqLds& t, const float* signs, const float* cb, const float* bnd,
                            int D, int nc) {
  for (int i = threadIdx.x; i < D; i += kThreads) t.signs[i] = signs[i];
  for (int i = threadIdx.x; i < nc; i += kThreads) t.cb[i] = cb[i];
  if (bnd)
    for (int i = threadIdx.x; i < nc - 1; i += kThreads) t.bnd[i] = bnd[i];
}

// Element offset of row r0 + r of a [B, H, Tc] row space inside a strided
// [B, H, T, D] array whose token axis starts at t0, for the tile's rows.
// The host keeps B * H * Tc below 2^31, so the row split is 32-bit.
__device__ void row_offsets(int64_t* off, int64_t r0, int nr, int H, int Tc, int t0, int64_t sb,
                            int64_t sh, int64_t st) {
  const int r = threadIdx.x;
  if (r < nr) {
    const uint32_t row = static_cast<uint32_t>(r0 + r);
    const uint32_t bh = row / static_cast<uint32_t>(Tc), t = row - bh * static_cast<uint32_t>(Tc);
    const uint32_t b = bh / static_cast<uint32_t>(H), h = bh - b * static_cast<uint32_t>(H);
    off[r] = static_cast<int64_t>(b) * sb + static_cast<int64_t>(h) * sh + (t0 + static_cast<int64_t>(t)) * st;
  }
}

__global__ void __launch_bounds__(kThreads) tq_encode_kernel(TqEncodeArgs a) {
  extern __shared__ float lds[];
  const int D = a.D;
  float* y = lds;                                                   // [kRows][D] f32
  uint8_t* codes = reinterpret_cast<uint8_t*>(y + kRows * D);       // [kRows][D]
  uint8_t* sg = codes + kRows * D;                                  // [kRows][D]
  __shared__ float den_s[kRows];
  __shared__ int64_t roff[kRows];
  __shared__ TqLds tb;
  const int tid = threadIdx.x;
  const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.Tc, total = rows * D;
  const bool keys = a.St != nullptr;
  const int nb = a.nc - 1;
  load_tables(tb, a.signs, a.codebook, a.bounds, D, a.nc);
  for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * kRows; r0 < rows;
       r0 += static_cast<int64_t>(gridDim.x) * kRows) {
    const int nr = static_cast<int>(rows - r0 < kRows ? rows - r0 : kRows);
    row_offsets(roff, r0, nr, a.H, a.Tc, a.t0, a.sb, a.sh, a.st);
    __syncthreads();
    // 1. load the tile (rows past the end are zeros)
    for (int e = tid; e < kRows * D; e += kThreads) {
      const int r = e / D, i = e - r * D;
      y[e] = r < nr ? load_f32(a.x, a.dtype, roff[r] + i) : 0.0f;
    }
    __syncthreads();
    // 2. norm in T: T(sqrt(T(sum T(x_i^2)))), the divisor T(norm + T(1e-8));
    //    eight lanes per row, double sums
    {
      const int r = tid >> 3, part = tid & 7;
      double s = 0.0;
      for (int i = part; i < D; i += 8) {
        const float v = y[r * D + i];
        s += static_cast<double>(round_dt(v * v, a.dtype));
      }
      s = group8_sum_d(s);
      const float nrm = round_dt(sqrtf(round_dt(static_cast<float>(s), a.dtype)), a.dtype);
      if (part == 0) {
        den_s[r] = round_dt(nrm + round_dt(1e-8f, a.dtype), a.dtype);
        if (r < nr) a.vec_norms[r0 + r] = f16_of(nrm);
      }
    }
    __syncthreads();
    // 3. unit vector in T, times the rotation signs (f32), rotated
    for (int e = tid; e < kRows * D; e += kThreads) {
      const int r = e / D, i = e - r * D;
      y[e] = round_dt(y[e] / den_s[r], a.dtype) * tb.signs[i];
    }
    hadamard_tile(y, kRows, D, a.blocks);
    // 4. codes (boundaries exceeded); keys keep the residual y - level
    for (int e = tid; e < kRows * D; e += kThreads) {
      const float v = y[e];
      int idx = 0;
      for (int k = 0; k < nb; ++k) idx += v > tb.bnd[k];
      codes[e] = static_cast<uint8_t>(idx);
      if (keys) y[e] = v - tb.cb[idx];
    }
    __syncthreads();
    if (keys) {
      // 5. residual norm: f32(sum f32(r_i^2)) -> sqrt -> f16
      {
        const int r = tid >> 3, part = tid & 7;
        double s = 0.0;
        for (int i = part; i < D; i += 8) {
          const float v = y[r * D + i];
          s += static_cast<double>(v * v);
        }
        s = group8_sum_d(s);
        if (part == 0 && r < nr) a.res_norms[r0 + r] = f16_of(sqrtf(static_cast<float>(s)));
      }
      // 6. projection through S (S^T as the right operand), signs p >= 0
      tile_matmul([&](int r, int i) { return y[r * D + i]; }, nr, D, a.St,
                  [&](int r, int j, float v) { sg[r * D + j] = v >= 0.0f; });
    }
    // 7. pack codes and signs into the flat words
    const int64_t e0 = r0 * D, e1 = (r0 + nr) * D;
    pack_tile(codes, e0, e1, total, a.bits, a.indices);
    if (keys) pack_tile(sg, e0, e1, total, 1, a.qjl);
    __syncthreads();
  }
}

// The tile's elements [e0, e1) of a flat word array of `bits` values, into
// bytes: one thread per word.
__device__ void unpack_tile(const uint32_t* words, int64_t e0, int64_t e1, int bits,
                            uint8_t* out) {
  const int vpw = 32 / bits;
  const uint32_t mask = (1u << bits) - 1u;
  const int64_t w0 = e0 / vpw, w1 = (e1 - 1) / vpw;
  for (int64_t w = w0 + threadIdx.x; w <= w1; w += kThreads) {
    const uint32_t word = words[w];
    const int64_t base = w * vpw - e0;
    for (int k = 0; k < vpw; ++k) {
      const int64_t t = base + k;
      if (t >= 0 && t < e1 - e0) out[t] = static_cast<uint8_t>((word >> (k * bits)) & mask);
    }
  }
}

__global__ void __launch_bounds__(kThreads) tq_decode_kernel(TqDecodeArgs a) {
  extern __shared__ float lds[];
  const int D = a.D;
  float* z = lds;                                                   // [kRows][D]
  uint8_t* codes = reinterpret_cast<uint8_t*>(z + kRows * D);       // [kRows][D]
  uint8_t* sg = codes + kRows * D;                                  // [kRows][D]
  __shared__ int64_t roff[kRows];
  __shared__ float cr[kRows];
  __shared__ float vn[kRows];
  __shared__ TqLds tb;
  const int tid = threadIdx.x;
  const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.Tc;
  const bool keys = a.S != nullptr;
  load_tables(tb, a.signs, a.codebook, nullptr, D, 1 << a.bits);
  for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * kRows; r0 < rows;
       r0 += static_cast<int64_t>(gridDim.x) * kRows) {
    const int nr = static_cast<int>(rows - r0 < kRows ? rows - r0 : kRows);
    row_offsets(roff, r0, nr, a.H, a.Tc, a.t0, a.osb, a.osh, a.ost);
    if (tid < nr) {
      vn[tid] = f16_to_f32(a.vec_norms[r0 + tid]);
      if (keys) cr[tid] = a.qs * f16_to_f32(a.res_norms[r0 + tid]);
    }
    const int64_t e0 = r0 * D, e1 = (r0 + nr) * D;
    unpack_tile(a.indices, e0, e1, a.bits, codes);
    if (keys) unpack_tile(a.qjl, e0, e1, 1, sg);
    __syncthreads();
    for (int e = tid; e < kRows * D; e += kThreads) z[e] = e < nr * D ? tb.cb[codes[e]] : 0.0f;
    if (keys) {
      for (int e = nr * D + tid; e < kRows * D; e += kThreads) sg[e] = 0;
      __syncthreads();
      // z += (sqrt(pi/2) / d * |r|) * (signs . S)
      tile_matmul([&](int r, int i) { return sg[r * D + i] ? 1.0f : -1.0f; }, nr, D, a.S,
                  [&](int r, int j, float v) { z[r * D + j] = z[r * D + j] + cr[r] * v; });
    }
    hadamard_tile(z, kRows, D, a.blocks);
    for (int e = tid; e < nr * D; e += kThreads) {
      const int r = e / D, i = e - r * D;
      const float w = z[e] * tb.signs[i] * vn[r];
      const uint16_t hv = f16_of(w);
      const int64_t o = roff[r] + i;
      if (a.out_dtype == kF16)
        static_cast<uint16_t*>(a.out)[o] = hv;
      else
        static_cast<float*>(a.out)[o] = f16_to_f32(hv);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Row kernels for head dims 64, 128 and 256 (one Hadamard block of D
// values).  Eight adjacent lanes hold a vector, lane p the E = D / 8
// contiguous values [p E, p E + E) in registers: the butterflies with h < E
// run inside a lane, those with h = E, 2E, 4E between lanes p and p ^ h / E
// (DPP moves), so the rotation needs no LDS and no barrier.  Every value is
// formed by the same operation on the same operands as in the tile kernels
// above (the norms' double sums take their terms in another order; a sum of
// at most 256 f32 terms is exact in double unless they span more than 29
// binades, so its f32 rounding is the same).  LDS keeps only the code bytes
// to pack or unpack and, for keys, the projection's operand rows.
//
// Bound: at 128 dims the f32 matrix product takes ~54 us of 257 792 keys
// (4.2 GMAC; [8, 8, 4028] of a compressed layer), the vector work (norm,
// division, rotation, codes) ~65; the two overlap little, all waves of a CU
// being in step, and giving waves different priorities by slot did not part
// them (129 / 133 us).  Measured there: encode keys 197 -> 127 us (vector FMA
// chains and true divisions before), decode keys 189 -> 125; values, without
// a projection, 81 -> 61 and 53 -> 54.

// The value of lane (lane ^ M) for M in {1, 2, 4}: the partner inside an
// aligned group of eight lanes.
template <int M>
__device__ __forceinline__ float lane_xor(float v) {
  const int i = __float_as_int(v);
  if constexpr (M == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0xB1, 0xF, 0xF, true));
  if constexpr (M == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x4E, 0xF, 0xF, true));
  // lane ^ 4 = (lane ^ 3) ^ 7: a quad reversal, then the half-row mirror
  const int t = __builtin_amdgcn_mov_dpp(i, 0x1B, 0xF, 0xF, true);
  return __int_as_float(__builtin_amdgcn_mov_dpp(t, 0x141, 0xF, 0xF, true));
}

// One butterfly stage between lanes p and p ^ M: the lower lane keeps
// a + c, the upper a - c (a the lower lane's value, c the upper's).  The
// product by +-1 is exact, so the fma rounds the same sum or difference.
template <int M, int E>
__device__ __forceinline__ void cross_stage(float (&x)[E], int part) {
  const float s = (part & M) ? -1.0f : 1.0f;
#pragma unroll
  for (int k = 0; k < E; ++k) x[k] = fmaf(x[k], s, lane_xor<M>(x[k]));
}

// hadamardTransform of one block of D = 8 E values held as above: stages
// h = 1, 2, ..., D / 2 in order, then times the block's f32 1 / sqrt(D).
template <int E>
__device__ __forceinline__ void row_butterflies(float (&x)[E], int part, float scale) {
#pragma unroll
  for (int h = 1; h < E; h <<= 1)
#pragma unroll
    for (int k = 0; k < E; ++k)
      if (!(k & h)) {
        const float a = x[k], c = x[k + h];
        x[k] = a + c;
        x[k + h] = a - c;
      }
  cross_stage<1>(x, part);
  cross_stage<2>(x, part);
  cross_stage<4>(x, part);
#pragma unroll
  for (int k = 0; k < E; ++k) x[k] = x[k] * scale;
}

// Element offset of row `row` of a [B, H, Tc] row space inside a strided
// [B, H, T, D] array whose token axis starts at t0 (row < 2^31).
__device__ __forceinline__ int64_t row_offset(int64_t row, int H, int Tc, int t0, int64_t sb,
                                              int64_t sh, int64_t st) {
  const uint32_t rw = static_cast<uint32_t>(row);
  const uint32_t bh = rw / static_cast<uint32_t>(Tc), t = rw - bh * static_cast<uint32_t>(Tc);
  const uint32_t b = bh / static_cast<uint32_t>(H), h = bh - b * static_cast<uint32_t>(H);
  return static_cast<int64_t>(b) * sb + static_cast<int64_t>(h) * sh +
         (t0 + static_cast<int64_t>(t)) * st;
}

// E contiguous values of dtype dt from element offset `off` (16-byte
// aligned: the launcher checks the base and the strides) as f32.
template <int E>
__device__ __forceinline__ void load_run(const void* p, int dt, int64_t off, float (&x)[E]) {
  if (dt == kF32) {
    const float4* q = reinterpret_cast<const float4*>(static_cast<const float*>(p) + off);
#pragma unroll
    for (int u = 0; u < E / 4; ++u) {
      const float4 v = q[u];
      x[4 * u] = v.x; x[4 * u + 1] = v.y; x[4 * u + 2] = v.z; x[4 * u + 3] = v.w;
    }
  } else {
    const uint4* q = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p) + off);
    const bool bf = dt == kBF16;
#pragma unroll
    for (int u = 0; u < E / 8; ++u) {
      const uint4 v = q[u];
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint16_t lo = static_cast<uint16_t>(w[c]), hi = static_cast<uint16_t>(w[c] >> 16);
        x[8 * u + 2 * c] = bf ? bf16_to_f32(lo) : f16_to_f32(lo);
        x[8 * u + 2 * c + 1] = bf ? bf16_to_f32(hi) : f16_to_f32(hi);
      }
    }
  }
}

// The flat word range of a tile: rows [r0, r0 + nr) of D values hold
// elements [r0 D, (r0 + nr) D), words from w0 on, the first element `lead`
// values into its word (32-bit arithmetic: r0 < 2^31, D <= 256).
struct TileWords {
  int64_t w0;
  int lead, n, nw;
};
__device__ __forceinline__ TileWords tile_words(int64_t r0, int nr, int D, int vpw) {
  const uint32_t q = static_cast<uint32_t>(r0) / static_cast<uint32_t>(vpw);
  const uint32_t rem = static_cast<uint32_t>(r0) - q * static_cast<uint32_t>(vpw);
  TileWords t;
  t.w0 = static_cast<int64_t>(q) * D + static_cast<int64_t>(rem * D / vpw);
  t.lead = static_cast<int>(rem * D % vpw);
  t.n = nr * D;
  t.nw = (t.lead + t.n + vpw - 1) / vpw;
  return t;
}

// pack_tile for the row kernels: words that start and end inside the tile
// (or end the tensor) are stored, the rest OR-ed into the zeroed output.
// With a power-of-two width no word crosses a row, so the bytes are read
// four at a time.
__device__ void pack_rows(const uint8_t* vals, int64_t r0, int nr, int D, bool last, int bits,
                          uint32_t* out) {
  const int vpw = 32 / bits;
  const TileWords tw = tile_words(r0, nr, D, vpw);
  if ((vpw & 3) == 0 && tw.lead == 0 && D % vpw == 0) {
    for (int lw = threadIdx.x; lw < tw.nw; lw += kThreads) {
      const uint32_t* v4 = reinterpret_cast<const uint32_t*>(vals + lw * vpw);
      uint32_t word = 0;
      for (int k = 0; k < vpw / 4; ++k) {
        const uint32_t v = v4[k];
        const uint32_t c = (v & 0xffu) | (((v >> 8) & 0xffu) << bits) |
                           (((v >> 16) & 0xffu) << (2 * bits)) | ((v >> 24) << (3 * bits));
        word |= c << (4 * k * bits);
      }
      out[tw.w0 + lw] = word;
    }
    return;
  }
  for (int lw = threadIdx.x; lw < tw.nw; lw += kThreads) {
    const int base = lw * vpw - tw.lead;
    uint32_t word = 0;
    for (int k = 0; k < vpw; ++k) {
      const int t = base + k;
      if (t >= 0 && t < tw.n) word |= static_cast<uint32_t>(vals[t]) << (k * bits);
    }
    if (base >= 0 && (base + vpw <= tw.n || last))
      out[tw.w0 + lw] = word;
    else if (word)
      atomicOr(out + tw.w0 + lw, word);
  }
}

// unpack_tile for the row kernels (bytes of the tile's elements).
__device__ void unpack_rows(const uint32_t* words, int64_t r0, int nr, int D, int bits,
                            uint8_t* out) {
  const int vpw = 32 / bits;
  const uint32_t mask = (1u << bits) - 1u;
  const TileWords tw = tile_words(r0, nr, D, vpw);
  if ((vpw & 3) == 0 && tw.lead == 0 && D % vpw == 0) {
    for (int lw = threadIdx.x; lw < tw.nw; lw += kThreads) {
      const uint32_t word = words[tw.w0 + lw];
      uint32_t* o4 = reinterpret_cast<uint32_t*>(out + lw * vpw);
      for (int k = 0; k < vpw / 4; ++k) {
        const uint32_t v = word >> (4 * k * bits);
        o4[k] = (v & mask) | (((v >> bits) & mask) << 8) | (((v >> (2 * bits)) & mask) << 16) |
                (((v >> (3 * bits)) & mask) << 24);
      }
    }
    return;
  }
  for (int lw = threadIdx.x; lw < tw.nw; lw += kThreads) {
    const uint32_t word = words[tw.w0 + lw];
    const int base = lw * vpw - tw.lead;
    for (int k = 0; k < vpw; ++k) {
      const int t = base + k;
      if (t >= 0 && t < tw.n) out[t] = static_cast<uint8_t>((word >> (k * bits)) & mask);
    }
  }
}

// acc(r, j) = sum_i a(r, i) M(i, j) of a tile of 32 rows, on f32 matrix
// cores: v_mfma_f32_16x16x4_f32 adds its four products in index order with a
// fused multiply-add each (the codec tests hold the signs and decoded values
// to the CPU's fmaf chains bit for bit), so a chain of D / 4 of them is the f32 chain in i order that
// the codec fixes, at twice the rate of unpacked vector FMAs and beside them.
// Wave w takes columns [w D / 4, (w + 1) D / 4): CT tiles of 16 columns x 2 of
// 16 rows.  A operand of step s: lane (r, g) holds a(r, 4 s + g); B: M(4 s +
// g, j0 + r); acc[rt][ct][i]: row 16 rt + 4 g + i, column j0 + 16 ct + r.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <int D>
struct RowsMatrix {
  static constexpr int CT = D / 64, S = D / 4;
  // M's operands stay in registers up to 128 dims (64 of them); at 256 they
  // are read per step
  static constexpr bool kHeld = D <= 128;
  float b[kHeld ? CT : 1][kHeld ? S : 1];
  const float* base;
  __device__ __forceinline__ void load(const float* M) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    base = M + (lane >> 4) * D + w * (D / 4) + (lane & 15);
    if constexpr (kHeld) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int s = 0; s < S; ++s) b[ct][s] = base[4 * s * D + 16 * ct];
    }
  }
  // a4(rt, s4): the four A operands of steps 4 s4 .. + 3 of row tile rt
  template <class A>
  __device__ __forceinline__ void run(A&& a4, f32x4_t (&acc)[2][CT]) const {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[rt][ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto quad = [&](int s4) __attribute__((always_inline)) {
      f32x4_t x[2] = {a4(0, s4), a4(1, s4)};
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          float m;
          if constexpr (kHeld) m = b[ct][4 * s4 + u];
          else m = base[4 * (4 * s4 + u) * D + 16 * ct];
#pragma unroll
          for (int rt = 0; rt < 2; ++rt)
            acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[rt][u], m, acc[rt][ct], 0, 0, 0);
        }
    };
    if constexpr (kHeld) {
#pragma unroll
      for (int s4 = 0; s4 < S / 4; ++s4) quad(s4);
    } else {
#pragma unroll 2
      for (int s4 = 0; s4 < S / 4; ++s4) quad(s4);
    }
  }
};

// x[k] / den rounded to DT, for the run of a vector: by the correctly rounded
// reciprocal and two correction steps, as the quantizer divides
// (affine_quantize8), where no step can lose bits: a divisor in [2^-60,
// 2^20] whose mantissa is not all ones, values that are zero or at least
// 2^-100 (quotients of 2^-120 and more: none is denormal, and every
// remainder is a multiple of 2^-147); a wave that holds others divides.  The
// sign of a zero is lost, which no later step sees.
template <int DT, int E>
__device__ __forceinline__ void unit_run(float (&x)[E], float den) {
  uint32_t least = ~0u;
#pragma unroll
  for (int k = 0; k < E; ++k) least = min(least, (__float_as_uint(x[k]) & 0x7fffffffu) - 1u);
  const bool fast = den >= 0x1p-60f && den <= 0x1p20f && least >= __float_as_uint(0x1p-100f) - 1u &&
                    (__float_as_uint(den) & 0x7fffffu) != 0x7fffffu;
  if (__builtin_amdgcn_ballot_w64(!fast) == 0) {
    const float inv = 1.0f / den;
#pragma unroll
    for (int k = 0; k < E; ++k) {
      float q = x[k] * inv;
      q = fmaf(fmaf(-q, den, x[k]), inv, q);
      x[k] = fmaf(fmaf(-q, den, x[k]), inv, q);
    }
  } else {
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = x[k] / den;
  }
#pragma unroll
  for (int k = 0; k < E; k += 2) round_pair<DT>(x[k], x[k + 1]);
}

// Waves a SIMD: three hide a tile's barriers under the others' matrix and
// vector work where the held matrix (64 registers at 128 dims) leaves room.
template <int D, bool KEYS>
constexpr int tq_waves() {
  return KEYS && D == 128 ? 3 : 1;
}

template <int D, bool KEYS, int DT>
__global__ void __launch_bounds__(kThreads)
    __attribute__((amdgpu_waves_per_eu(tq_waves<D, KEYS>()))) tq_encode_rows(TqEncodeArgs a) {
  constexpr int E = D / 8, S = D / 4, CT = D / 64;
  constexpr int kPitch = D + 4;  // floats of a residual row: rows start 4 banks apart
  extern __shared__ float lds[];
  float* y = lds;                                             // keys: [kRows][kPitch] residuals
  uint8_t* codes = reinterpret_cast<uint8_t*>(lds + (KEYS ? kRows * kPitch : 0));  // [kRows][D]
  __shared__ float cb_s[256], bnd_s[256];
  const int tid = threadIdx.x, r = tid >> 3, part = tid & 7;
  const int lane = tid & 63, wave = tid >> 6;
  const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.Tc;
  const int nb = a.nc - 1;
  for (int i = tid; i < a.nc; i += kThreads) cb_s[i] = a.codebook[i];
  for (int i = tid; i < nb; i += kThreads) bnd_s[i] = a.bounds[i];
  float rs[E];
#pragma unroll
  for (int k = 0; k < E; ++k) rs[k] = a.signs[part * E + k];
  RowsMatrix<KEYS ? D : 64> mat;
  if constexpr (KEYS) mat.load(a.St);
  const float scale = a.blocks.scale[0];
  const float eps = round_one<DT>(1e-8f);
  __syncthreads();
  for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * kRows; r0 < rows;
       r0 += static_cast<int64_t>(gridDim.x) * kRows) {
    const int nr = static_cast<int>(rows - r0 < kRows ? rows - r0 : kRows);
    const bool live = r < nr;
    // 1. the lane's run of the vector (rows past the end are zeros)
    float x[E];
    if (live) {
      load_run<E>(a.x, DT, row_offset(r0 + r, a.H, a.Tc, a.t0, a.sb, a.sh, a.st) + part * E, x);
    } else {
#pragma unroll
      for (int k = 0; k < E; ++k) x[k] = 0.0f;
    }
    // 2. norm in T, the divisor T(norm + T(1e-8))
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < E; k += 2) {
      float u = x[k] * x[k], v = x[k + 1] * x[k + 1];
      round_pair<DT>(u, v);
      s += static_cast<double>(u);
      s += static_cast<double>(v);
    }
    s = group8_sum_d(s);
    const float nrm = round_one<DT>(sqrtf(round_one<DT>(static_cast<float>(s))));
    const float den = round_one<DT>(nrm + eps);
    if (part == 0 && live) a.vec_norms[r0 + r] = f16_of(nrm);
    // 3. unit vector in T, times the rotation signs, rotated
    unit_run<DT>(x, den);
#pragma unroll
    for (int k = 0; k < E; ++k) x[k] = x[k] * rs[k];
    row_butterflies<E>(x, part, scale);
    // 4. codes; keys keep the residual y - level
    int idx[E];
#pragma unroll
    for (int k = 0; k < E; ++k) idx[k] = 0;
    for (int b = 0; b < nb; ++b) {
      const float bv = bnd_s[b];
#pragma unroll
      for (int k = 0; k < E; ++k) idx[k] += x[k] > bv;
    }
    {
      uint32_t* c4 = reinterpret_cast<uint32_t*>(codes + r * D + part * E);
#pragma unroll
      for (int u = 0; u < E / 4; ++u)
        c4[u] = static_cast<uint32_t>(idx[4 * u]) | (static_cast<uint32_t>(idx[4 * u + 1]) << 8) |
                (static_cast<uint32_t>(idx[4 * u + 2]) << 16) |
                (static_cast<uint32_t>(idx[4 * u + 3]) << 24);
    }
    if constexpr (KEYS) {
      // 5. residual norm: f32(sum f32(r_i^2)) -> sqrt -> f16
      double q = 0.0;
#pragma unroll
      for (int k = 0; k < E; ++k) {
        const float v = x[k] - cb_s[idx[k]];
        x[k] = v;
        q += static_cast<double>(v * v);
      }
      q = group8_sum_d(q);
      if (part == 0 && live) a.res_norms[r0 + r] = f16_of(sqrtf(static_cast<float>(q)));
      // the residuals in the matrix product's operand order: element 4 s + g
      // of a row at g S + s
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float* yg = y + r * kPitch + g * S + part * (E / 4);
        if constexpr (E == 8) {
          *reinterpret_cast<float2*>(yg) = make_float2(x[g], x[4 + g]);
        } else {
#pragma unroll
          for (int u = 0; u < E / 16; ++u)
            reinterpret_cast<float4*>(yg)[u] =
                make_float4(x[16 * u + g], x[16 * u + 4 + g], x[16 * u + 8 + g], x[16 * u + 12 + g]);
        }
      }
    }
    __syncthreads();
    // 6. projection through S (S^T as the right operand), signs p >= 0: a
    // ballot holds 16 columns of 4 rows, lane row < 32 stores its row's words
    if constexpr (KEYS) {
      f32x4_t acc[2][CT];
      const float* ya = y + (lane & 15) * kPitch + (lane >> 4) * S;
      mat.run([&](int rt, int s4) __attribute__((always_inline)) {
        return *reinterpret_cast<const f32x4_t*>(ya + 16 * rt * kPitch + 4 * s4);
      }, acc);
      uint32_t bits[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        bits[ct] = 0;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint64_t bal = __builtin_amdgcn_ballot_w64(acc[rt][ct][i] >= 0.0f);
            if ((lane >> 4) == rt && (lane & 3) == i)
              bits[ct] = static_cast<uint32_t>(bal >> (16 * ((lane >> 2) & 3))) & 0xFFFFu;
          }
      }
      if (lane < nr) {
        uint16_t* q16 = reinterpret_cast<uint16_t*>(a.qjl) + (r0 + lane) * (D / 16) + wave * CT;
        if constexpr (CT == 1) {
          *q16 = static_cast<uint16_t>(bits[0]);
        } else {
#pragma unroll
          for (int c = 0; c < CT; c += 2)
            *reinterpret_cast<uint32_t*>(q16 + c) = bits[c] | bits[c + 1] << 16;
        }
      }
    }
    // 7. pack the codes into the flat words
    pack_rows(codes, r0, nr, D, r0 + nr == rows, a.bits, a.indices);
    __syncthreads();
  }
}

template <int D, bool KEYS>
__global__ void __launch_bounds__(kThreads)
    __attribute__((amdgpu_waves_per_eu(tq_waves<D, KEYS>()))) tq_decode_rows(TqDecodeArgs a) {
  constexpr int E = D / 8, CT = D / 64;
  constexpr int kPitch = D + 4;
  extern __shared__ float lds[];
  float* z = lds;                                             // keys: [kRows][kPitch]
  uint8_t* codes = reinterpret_cast<uint8_t*>(lds + (KEYS ? kRows * kPitch : 0));  // [kRows][D]
  __shared__ float cb_s[256], cr_s[kRows];
  const int tid = threadIdx.x, r = tid >> 3, part = tid & 7;
  const int lane = tid & 63, wave = tid >> 6;
  const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.Tc;
  for (int i = tid; i < (1 << a.bits); i += kThreads) cb_s[i] = a.codebook[i];
  float rs[E];
#pragma unroll
  for (int k = 0; k < E; ++k) rs[k] = a.signs[part * E + k];
  RowsMatrix<KEYS ? D : 64> mat;
  if constexpr (KEYS) mat.load(a.S);
  const float scale = a.blocks.scale[0];
  for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * kRows; r0 < rows;
       r0 += static_cast<int64_t>(gridDim.x) * kRows) {
    const int nr = static_cast<int>(rows - r0 < kRows ? rows - r0 : kRows);
    const bool live = r < nr;
    // keys: the sign words of this lane's rows of the matrix product (rows
    // past the end repeat the last)
    constexpr int W = D / 32;
    uint32_t sw[2][KEYS ? W : 1];
    if constexpr (KEYS) {
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const int row = min(16 * rt + (lane & 15), nr - 1);
#pragma unroll
        for (int w = 0; w < W; ++w) sw[rt][w] = a.qjl[(r0 + row) * W + w];
      }
      if (tid < nr) cr_s[tid] = a.qs * f16_to_f32(a.res_norms[r0 + tid]);
    }
    unpack_rows(a.indices, r0, nr, D, a.bits, codes);
    const float vn = live ? f16_to_f32(a.vec_norms[r0 + r]) : 0.0f;
    __syncthreads();
    float x[E];
    if constexpr (KEYS) {
      // z = level + (sqrt(pi/2) / d * |r|) * (signs . S); fma(+-1, S, q) is
      // the sum or difference the reference's sign product rounds.  Operand
      // 4 s + g of a row is +-1 by bit 4 s + g of its words.
      f32x4_t acc[2][CT];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int w = 0; w < W; ++w) sw[rt][w] = ~sw[rt][w] >> (lane >> 4);
      mat.run([&](int rt, int s4) __attribute__((always_inline)) {
        f32x4_t v;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int s = 4 * s4 + u;
          v[u] = __uint_as_float((sw[rt][s / 8] << (31 - 4 * (s & 7)) & 0x80000000u) | 0x3F800000u);
        }
        return v;
      }, acc);
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int rr = 16 * rt + 4 * (lane >> 4) + i;
          // (rows past the end hold stale codes and are not kept)
          const float cr = cr_s[rr];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            const int j = wave * (D / 4) + 16 * ct + (lane & 15);
            z[rr * kPitch + j] = cb_s[codes[rr * D + j]] + cr * acc[rt][ct][i];
          }
        }
      __syncthreads();
      const float4* z4 = reinterpret_cast<const float4*>(z + r * kPitch + part * E);
#pragma unroll
      for (int u = 0; u < E / 4; ++u) {
        const float4 v = live ? z4[u] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        x[4 * u] = v.x; x[4 * u + 1] = v.y; x[4 * u + 2] = v.z; x[4 * u + 3] = v.w;
      }
    } else {
      const uint32_t* c4 = reinterpret_cast<const uint32_t*>(codes + r * D + part * E);
#pragma unroll
      for (int u = 0; u < E / 4; ++u) {
        const uint32_t w = live ? c4[u] : 0u;
#pragma unroll
        for (int c = 0; c < 4; ++c) x[4 * u + c] = live ? cb_s[(w >> (8 * c)) & 0xffu] : 0.0f;
      }
    }
    row_butterflies<E>(x, part, scale);
    if (live) {
      const int64_t o = row_offset(r0 + r, a.H, a.Tc, a.t0, a.osb, a.osh, a.ost) + part * E;
      uint16_t hv[E];
#pragma unroll
      for (int k = 0; k < E; ++k) hv[k] = f16_of(x[k] * rs[k] * vn);
      if (a.out_dtype == kF16) {
        uint4* q = reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + o);
#pragma unroll
        for (int u = 0; u < E / 8; ++u) {
          uint32_t w[4];
#pragma unroll
          for (int c = 0; c < 4; ++c)
            w[c] = static_cast<uint32_t>(hv[8 * u + 2 * c]) |
                   (static_cast<uint32_t>(hv[8 * u + 2 * c + 1]) << 16);
          q[u] = make_uint4(w[0], w[1], w[2], w[3]);
        }
      } else {
        float4* q = reinterpret_cast<float4*>(static_cast<float*>(a.out) + o);
#pragma unroll
        for (int u = 0; u < E / 4; ++u)
          q[u] = make_float4(f16_to_f32(hv[4 * u]), f16_to_f32(hv[4 * u + 1]),
                             f16_to_f32(hv[4 * u + 2]), f16_to_f32(hv[4 * u + 3]));
      }
    }
    __syncthreads();
  }
}

// dst = src converted (4-D strided, element strides, round to nearest even
// when narrowing): the cast of MLX's concatenation and slice assignment.
__global__ void __launch_bounds__(256) cast4d_kernel(const void* src, int sdt, int64_t n0,
                                                     int64_t n1, int64_t n2, int64_t n3,
                                                     int64_t s0, int64_t s1, int64_t s2,
                                                     int64_t s3, void* dst, int ddt, int64_t d0,
                                                     int64_t d1, int64_t d2, int64_t d3) {
  const int64_t n = n0 * n1 * n2 * n3;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < n;
       e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    int64_t r = e;
    const int64_t i3 = r % n3;
    r /= n3;
    const int64_t i2 = r % n2;
    r /= n2;
    const int64_t i1 = r % n1, i0 = r / n1;
    const float v = load_f32(src, sdt, i0 * s0 + i1 * s1 + i2 * s2 + i3 * s3);
    const int64_t o = i0 * d0 + i1 * d1 + i2 * d2 + i3 * d3;
    if (ddt == kF16)
      static_cast<uint16_t*>(dst)[o] = f16_of(v);
    else if (ddt == kBF16)
      static_cast<uint16_t*>(dst)[o] = f32_to_bf16(v);
    else
      static_cast<float*>(dst)[o] = v;
  }
}

// The exact tokens and the empty window of a unified buffer in one launch:
// per (b, h) row (blockIdx.y) the sink tokens, the tail tokens (cast as
// cast4d_kernel casts, a copy where the dtypes agree) and zeros, U dims a
// thread (8 where rows are whole 16-byte units).  A compressed layer has 324
// such tokens a row (64 rows x 128 to f32: 10.6 MB written): five launches of
// ~5 us before; 9.0 us at one dim a thread, 5.5 at eight.
template <int U>
__global__ void __launch_bounds__(256) tq_exact_kernel(TqExactArgs a) {
  const uint32_t per = static_cast<uint32_t>(a.D) / U, tokens = 256u / per;  // D <= 256
  const uint32_t u = threadIdx.x / per, d = (threadIdx.x - u * per) * U;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * tokens + u;
  if (u >= tokens || t >= static_cast<int64_t>(a.n_sink) + a.n_tail + a.n_zero) return;
  const int64_t row = blockIdx.y;
  const bool tail = t >= a.n_sink, zero = t >= static_cast<int64_t>(a.n_sink) + a.n_tail;
  const int64_t k = t - (tail ? a.n_sink : 0);  // token of its source
  const int64_t at = zero ? a.zero_at + (k - a.n_tail) : tail ? a.tail_at + k : t;
  const int64_t o = row * a.row_elems + at * a.D + d;
  const void* src = tail ? a.tail : a.sink;
  const int sdt = tail ? a.tail_dtype : a.sink_dtype;
  const int64_t s = (row * (tail ? a.n_tail : a.n_sink) + k) * a.D + d;
  if constexpr (U == 8) {
    if (a.dtype != kF32 && (zero || sdt == a.dtype)) {
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (!zero) v = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(src) + s);
      *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + o) = v;
      return;
    }
  }
  float x[U];
  if (zero) {
#pragma unroll
    for (int e = 0; e < U; ++e) x[e] = 0.0f;
  } else if constexpr (U == 8) {
    load_run<8>(src, sdt, s, x);
  } else {
    x[0] = load_f32(src, sdt, s);
  }
  if (a.dtype == kF32) {
    float* q = static_cast<float*>(a.out) + o;
    if constexpr (U == 8) {
      reinterpret_cast<float4*>(q)[0] = make_float4(x[0], x[1], x[2], x[3]);
      reinterpret_cast<float4*>(q)[1] = make_float4(x[4], x[5], x[6], x[7]);
    } else {
      *q = x[0];
    }
  } else {
    uint16_t* q = static_cast<uint16_t*>(a.out) + o;
    if (U == 1 && !zero && sdt == a.dtype) {
      *q = static_cast<const uint16_t*>(src)[s];
    } else {
#pragma unroll
      for (int e = 0; e < U; ++e) q[e] = a.dtype == kF16 ? f16_of(x[e]) : f32_to_bf16(x[e]);
    }
  }
}

// Zeros over `rows` runs of `run` units of T, `pitch` units apart.
template <class T>
__global__ void __launch_bounds__(256) zero_runs_kernel(T* base, int64_t pitch, int64_t run,
                                                        int64_t rows) {
  const int64_t n = run * rows;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; e < n;
       e += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = e / run;
    base[r * pitch + (e - r * run)] = T{};
  }
}

int grid_for(int64_t rows, int64_t most = 2048) {
  const int64_t t = (rows + kRows - 1) / kRows;
  return static_cast<int>(t < most ? (t > 0 ? t : 1) : most);
}
// The workgroups of a row launch: with the matrix held in registers, those
// that run at once (three a CU at 128 dims), so that each loads it once.
int rows_grid(int64_t rows, int D, bool keys) {
  return grid_for(rows, keys && D == 128 ? 768 : 2048);
}

// The row kernels take head dims 64, 128 and 256 (one Hadamard block) over
// an array whose base and strides keep every lane's run 16-byte aligned.
bool rows_kernel_fits(int D, const TqBlocks& bl, const void* base, int es, int64_t s0, int64_t s1,
                      int64_t s2) {
  if (!(D == 64 || D == 128 || D == 256) || bl.n != 1) return false;
  return reinterpret_cast<uintptr_t>(base) % 16 == 0 && (s0 * es) % 16 == 0 &&
         (s1 * es) % 16 == 0 && (s2 * es) % 16 == 0;
}

}  // namespace

// Whether the launch of these arguments writes every word of the packed codes
// (and signs) itself; otherwise words shared by tiles are OR-ed into zeros.
static bool tq_rows_launch(const TqEncodeArgs& a) {
  return rows_kernel_fits(a.D, a.blocks, a.x, a.dtype == kF32 ? 4 : 2, a.sb, a.sh, a.st);
}
bool tq_encode_needs_zero_codes(const TqEncodeArgs& a) {
  const int vpw = 32 / a.bits;  // widths that divide a row: no word crosses a tile
  return !(tq_rows_launch(a) && (vpw & 3) == 0 && a.D % vpw == 0);
}
bool tq_encode_needs_zero_signs(const TqEncodeArgs& a) { return !tq_rows_launch(a); }

void launch_tq_encode(const TqEncodeArgs& a, hipStream_t st) {
  const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.Tc;
  if (rows <= 0) return;
  VKV_CHECK(rows < (int64_t{1} << 31), "TurboQuant encodes fewer than 2^31 vectors per call");
  VKV_CHECK(a.D >= 2 && a.D <= 256, "TurboQuant head dims must be in [2, 256]");
  VKV_CHECK(a.bits >= 1 && a.bits <= 8, "TurboQuant index bits must be in [1, 8]");
  const dim3 g(tq_rows_launch(a) ? rows_grid(rows, a.D, a.St != nullptr) : grid_for(rows)), b(kThreads);
  // the key launch (the QJL projection) is the one the timing aid records
  const TimedLaunch tl = a.St ? timing_prepare(kTimeTqEncode) : TimedLaunch{};
  if (tq_rows_launch(a)) {
    const size_t lds = static_cast<size_t>(kRows) * (a.St ? 4 * (a.D + 4) + a.D : a.D);
    auto run = [&](auto D_, auto K_, auto T_) {
      hipExtLaunchKernelGGL((tq_encode_rows<decltype(D_)::value, decltype(K_)::value, decltype(T_)::value>),
                            g, b, lds, st, tl.start, tl.stop, 0, a);
    };
    using std::integral_constant;
    auto dims = [&](auto K_, auto T_) {
      if (a.D == 64) run(integral_constant<int, 64>{}, K_, T_);
      else if (a.D == 128) run(integral_constant<int, 128>{}, K_, T_);
      else run(integral_constant<int, 256>{}, K_, T_);
    };
    auto kind = [&](auto T_) { a.St ? dims(std::true_type{}, T_) : dims(std::false_type{}, T_); };
    if (a.dtype == kBF16) kind(integral_constant<int, kBF16>{});
    else if (a.dtype == kF16) kind(integral_constant<int, kF16>{});
    else kind(integral_constant<int, kF32>{});
  } else {
    const size_t lds = static_cast<size_t>(kRows) * a.D * (4 + 1 + 1);
    hipExtLaunchKernelGGL(tq_encode_kernel, g, b, lds, st, tl.start, tl.stop, 0, a);
  }
  VKV_HIP(hipGetLastError());
  if (a.St) timing_commit(tl);
}

void launch_tq_decode(const TqDecodeArgs& a, hipStream_t st) {
  const int64_t rows = static_cast<int64_t>(a.B) * a.H * a.Tc;
  if (rows <= 0) return;
  VKV_CHECK(rows < (int64_t{1} << 31), "TurboQuant decodes fewer than 2^31 vectors per call");
  VKV_CHECK(a.D >= 2 && a.D <= 256, "TurboQuant head dims must be in [2, 256]");
  VKV_CHECK(a.bits >= 1 && a.bits <= 8, "TurboQuant index bits must be in [1, 8]");
  const bool fits = rows_kernel_fits(a.D, a.blocks, a.out, a.out_dtype == kF32 ? 4 : 2, a.osb, a.osh, a.ost);
  const dim3 g(fits ? rows_grid(rows, a.D, a.S != nullptr) : grid_for(rows)), b(kThreads);
  const TimedLaunch tl = a.S ? timing_prepare(kTimeTqDecode) : TimedLaunch{};
  if (fits) {
    const size_t lds = static_cast<size_t>(kRows) * (a.S ? 4 * (a.D + 4) + a.D : a.D);
    switch (a.D) {
      case 64: a.S ? hipExtLaunchKernelGGL((tq_decode_rows<64, true>), g, b, lds, st, tl.start, tl.stop, 0, a)
              : hipExtLaunchKernelGGL((tq_decode_rows<64, false>), g, b, lds, st, tl.start, tl.stop, 0, a);
      break;
      case 128: a.S ? hipExtLaunchKernelGGL((tq_decode_rows<128, true>), g, b, lds, st, tl.start, tl.stop, 0, a)
              : hipExtLaunchKernelGGL((tq_decode_rows<128, false>), g, b, lds, st, tl.start, tl.stop, 0, a);
      break;
      default: a.S ? hipExtLaunchKernelGGL((tq_decode_rows<256, true>), g, b, lds, st, tl.start, tl.stop, 0, a)
              : hipExtLaunchKernelGGL((tq_decode_rows<256, false>), g, b, lds, st, tl.start, tl.stop, 0, a);
      break;
    }
  } else {
    const size_t lds = static_cast<size_t>(kRows) * a.D * (4 + 1 + 1);
    hipExtLaunchKernelGGL(tq_decode_kernel, g, b, lds, st, tl.start, tl.stop, 0, a);
  }
  VKV_HIP(hipGetLastError());
  if (a.S) timing_commit(tl);
}

void launch_tq_exact(const TqExactArgs& a, int64_t bh, hipStream_t st) {
  const int64_t n = static_cast<int64_t>(a.n_sink) + a.n_tail + a.n_zero;
  if (n <= 0 || bh <= 0) return;
  VKV_CHECK(a.D >= 1 && a.D <= 256, "TurboQuant head dims must be in [2, 256]");
  // 16-byte units: every row of every array starts on one
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool wide = a.D % 8 == 0 && a.row_elems % 8 == 0 && aligned(a.out) && aligned(a.sink) && aligned(a.tail);
  const int64_t tokens = 256 / (wide ? a.D / 8 : a.D);
  for (int64_t r0 = 0; r0 < bh; r0 += 65535) {
    TqExactArgs b = a;
    const int es = a.dtype == kF32 ? 4 : 2;
    b.out = static_cast<uint8_t*>(a.out) + r0 * a.row_elems * es;
    auto at = [&](const void* p, int dt, int64_t tokens) {
      return p ? static_cast<const uint8_t*>(p) + r0 * tokens * a.D * (dt == kF32 ? 4 : 2) : nullptr;
    };
    b.sink = at(a.sink, a.sink_dtype, a.n_sink);
    b.tail = at(a.tail, a.tail_dtype, a.n_tail);
    const dim3 grid(static_cast<unsigned>((n + tokens - 1) / tokens),
                    static_cast<unsigned>(std::min<int64_t>(65535, bh - r0)));
    if (wide)
      hipLaunchKernelGGL(tq_exact_kernel<8>, grid, dim3(256), 0, st, b);
    else
      hipLaunchKernelGGL(tq_exact_kernel<1>, grid, dim3(256), 0, st, b);
    VKV_HIP(hipGetLastError());
  }
}

void launch_zero_runs(void* base, int64_t pitch_bytes, int64_t run_bytes, int64_t rows,
                      hipStream_t st) {
  if (run_bytes <= 0 || rows <= 0) return;
  VKV_CHECK(pitch_bytes % 2 == 0 && run_bytes % 2 == 0 && reinterpret_cast<uintptr_t>(base) % 2 == 0,
            "zeroed runs are whole 2-byte units");
  const bool wide = pitch_bytes % 16 == 0 && run_bytes % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(base) % 16 == 0;
  const int64_t unit = wide ? 16 : 2, n = run_bytes / unit * rows;
  const int g = static_cast<int>(std::min<int64_t>((n + 255) / 256, 4096));
  if (wide)
    hipLaunchKernelGGL(zero_runs_kernel<uint4>, dim3(g), dim3(256), 0, st, static_cast<uint4*>(base),
                       pitch_bytes / 16, run_bytes / 16, rows);
  else
    hipLaunchKernelGGL(zero_runs_kernel<uint16_t>, dim3(g), dim3(256), 0, st,
                       static_cast<uint16_t*>(base), pitch_bytes / 2, run_bytes / 2, rows);
  VKV_HIP(hipGetLastError());
}

void launch_cast4d(const void* src, int sdt, const int64_t* shape, const int64_t* sstr, void* dst,
                   int ddt, const int64_t* dstr, hipStream_t st) {
  const int64_t n = shape[0] * shape[1] * shape[2] * shape[3];
  if (n <= 0) return;
  const int g = static_cast<int>(std::min<int64_t>((n + 255) / 256, 4096));
  hipLaunchKernelGGL(cast4d_kernel, dim3(g), dim3(256), 0, st, src, sdt, shape[0], shape[1],
                     shape[2], shape[3], sstr[0], sstr[1], sstr[2], sstr[3], dst, ddt, dstr[0],
                     dstr[1], dstr[2], dstr[3]);
  VKV_HIP(hipGetLastError());
}

}  // namespace vkv
