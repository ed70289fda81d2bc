// Helpers shared by the attention kernels (forward and backward) of libfastops_hip.so.
#pragma once
#include "common.hpp"

namespace fo {

#define FO_LDS __attribute__((address_space(3)))
#define FO_GLOBAL __attribute__((address_space(1)))

template <typename T> struct Ops;
template <> struct Ops<__bf16> {
  typedef bf16x8 vec8;
  static __device__ __forceinline__ f32x16 mfma(vec8 a, vec8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Ops<_Float16> {
  typedef f16x8 vec8;
  static __device__ __forceinline__ f32x16 mfma(vec8 a, vec8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};

// swizzle of 16-byte chunks inside a tile row; `row` is the row inside the tile
template <int D>
__device__ __forceinline__ int swz(int row) {
  if constexpr (D == 128) return ((row & 3) << 2) | ((row >> 2) & 3);              // 16 chunks per 256-byte row
  else { const int R = row >> 1; return ((R & 1) << 2) | ((R >> 1) & 3); }          // 8 chunks per 128-byte row
}

__device__ __forceinline__ float half_swap(float x) {
  // value held by the lane 32 positions away
  auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, x), __builtin_bit_cast(int, x), false, false);
  return __builtin_bit_cast(float, (threadIdx.x & 32) ? r[0] : r[1]);
}

// 16 bytes per lane, global -> LDS without passing through registers. LDS receives the 64 lanes' pieces back to back
// starting at `dst` (wave-uniform); the global address is per lane.
// An LDS-DMA instruction reads M0 (the LDS destination) and needs one wait state after the scalar instruction that
// wrote it. The compiler adds that s_nop for its own builtin; inside an asm statement nobody does, so it is spelled out
// here, and the build's assembly check (asm_lint.py) verifies it for every kernel.
// (hipcc also parses device functions in its host pass, where GCN assembly cannot be checked: the bodies exist in the
// device pass only.)
__device__ __forceinline__ void dma16_uniform_base(const void* base, uint32_t byte_off, FO_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst)), "v"(byte_off), "s"(base) : "memory", "m0");
#endif
}
// ... with the LDS address as a wave-uniform register plus a constant: one scalar instruction forms it in M0
template <int IMM>
__device__ __forceinline__ void dma16_uniform_base_lds_imm(const void* base, uint32_t byte_off, uint32_t lds_base) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(byte_off), "s"(base), "n"(IMM) : "memory", "m0", "scc");
#endif
}
// ... by the lanes of `lanes` only: the others' 16 bytes of LDS stay as they are. (For wave-uniform code: every lane is
// active before and after. The write of EXEC is also the wait state that M0 needs.)
__device__ __forceinline__ void dma16_uniform_base_of_lanes(const void* base, uint32_t byte_off, uint32_t dst, uint64_t lanes) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" ::"s"(dst), "v"(byte_off), "s"(base), "s"(lanes) : "memory", "m0");
#endif
}
__device__ __forceinline__ void dma16_lane_ptr(const void* ptr, FO_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst)), "v"(ptr) : "memory", "m0");
#endif
}

// A operand of a 32x32x16 MFMA from a row-major tile in LDS: lane = row l32 of block `blk`, 8 elements at
// column 16*ks + 8*hh
template <typename T, int D>
__device__ __forceinline__ typename Ops<T>::vec8 row_frag(FO_LDS const char* tile, int blk, int ks, int l32, int hh) {
  const int row = 32 * blk + l32;
  return *(FO_LDS const typename Ops<T>::vec8*)(tile + row * (D * 2) + (((2 * ks + hh) ^ swz<D>(row)) * 16));
}
// A operand = transpose of a tile block: M = 32 columns (d = 32*db ..), K = 16 rows of the tile in the order the 32x32
// accumulator layout hands them over as a B operand (rows 16*t + 4*hh + {0..3} and + 8)
template <typename T, int D>
__device__ __forceinline__ typename Ops<T>::vec8 col_frag(FO_LDS const char* tile, int t, int db, int lane) {
  const int hh = lane >> 5, L16 = lane & 15, g16 = (lane >> 4) & 1;
  const int row0 = 16 * t + 4 * hh + (L16 >> 2), row1 = row0 + 8;
  const int chunk = 4 * db + 2 * g16 + ((L16 & 3) >> 1);
  const int sub = (L16 & 1) * 8;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FO_LDS s16x4*)(tile + row0 * (D * 2) + ((chunk ^ swz<D>(row0)) * 16) + sub));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FO_LDS s16x4*)(tile + row1 * (D * 2) + ((chunk ^ swz<D>(row1)) * 16) + sub));
  return __builtin_bit_cast(typename Ops<T>::vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Sixteen zero bytes in device memory. A head_dim below the 64 or 128 columns a kernel is compiled for is handled by
// addresses alone: whatever would read columns past the true head_dim - a lane's piece of a tile copy, a fragment
// loaded from a row - reads these zeros instead, so the padded columns of every operand are zero (they add nothing to a
// product) and nothing is read past the end of a row; stores of such columns are skipped.
static __device__ __attribute__((aligned(16))) const uint32_t kZero16[4] = {0u, 0u, 0u, 0u};
template <typename T>
__device__ __forceinline__ const T* live_or_zero(const T* ptr, int col, int d) {
  return col < d ? ptr : (const T*)kZero16;
}

// Column count a kernel computes with, for a head_dim d on kernels laid out for D columns: the products leave out what
// lies past the next multiple of 32.
constexpr int live_columns(int D, int d) { return D == 128 ? (d <= 96 ? 96 : 128) : (d <= 32 ? 32 : 64); }

// Dropout of attention probabilities, as the reference defines it (flash_attention_triton.py:38-50,125,216-219): element
// (b*H + h, q, key) has the 32-bit index  offset + (b*H + h)*Sq*Sk + q*Sk + key  (all arithmetic modulo 2^32); the index,
// xored with the seed, goes through an integer hash, and the element is KEPT iff the hash exceeds
// uint32(fp32(p) * 2^32); kept probabilities are multiplied by 1 / (1 - p). Row sums (and so LSE) use the
// undropped probabilities.
struct DropoutParams {
  uint32_t seed;
  uint32_t threshold;     // uint32(fp32(p) * fp32(4294967295)), computed on the host
  uint32_t offset;        // low 32 bits of the generator offset
  float keep_scale;       // 1 / (1 - p) in fp32; 1 when dropout is off
  float keep_prob;        // 1 - p
  float keep_log2;        // log2 of keep_scale
};
__host__ __device__ __forceinline__ bool dropout_keep(uint32_t index, uint32_t seed, uint32_t threshold) {
  uint32_t a = index ^ seed;
  a ^= a >> 4;
  a = (a ^ 0xDEADBEEFu) + (a << 5);
  a ^= a >> 11;
  return a > threshold;
}
// The mask over a run of consecutive indices, mostly without hashing each of them. The hash mixes little: with the low L
// bits of the index free, x = index ^ seed is an aligned block of 2^L values; so is y = x ^ (x >> 4), whose bits from L
// on depend on x's bits from L on only; z = (y ^ 0xDEADBEEF) + (y << 5) then lies in [z0, z0 + 33 (2^L - 1)], i.e. in at
// most two values A of z >> (L + 6); and the hash z ^ (z >> 11) has A ^ (A >> 11) in its bits from L + 6 on. Where both
// of those are above, or both below, the threshold's bits, all 2^L elements are kept, or all dropped. A run that starts
// inside a block spans two blocks. What remains undecided is hashed element by element: 0.0-0.5 % of the runs of
// 32 rows x 1024 keys at p = 0.1-0.17 (12 heads x 2048-8192 keys, 96 heads x 1024 keys), because the kept indices form
// long bands: about one run in ten is dropped as a whole.
enum : int { kDropAll = 0, kKeepAll = 1, kDropMixed = 2 };
template <int L>
__host__ __device__ __forceinline__ int dropout_block(uint32_t index, uint32_t seed, uint32_t threshold) {
  constexpr uint32_t low = (1u << L) - 1u;
  const uint32_t x = (index ^ seed) & ~low;
  const uint32_t y = (x ^ (x >> 4)) & ~low;
  const uint32_t z0 = ((y ^ 0xDEADBEEFu) & ~low) + (y << 5), z1 = z0 + 33u * low;    // (modulo 2^32, as the hash)
  const uint32_t a0 = z0 >> (L + 6), a1 = z1 >> (L + 6), t = threshold >> (L + 6);
  const uint32_t w0 = a0 ^ (a0 >> 11), w1 = a1 ^ (a1 >> 11);
  return (w0 > t && w1 > t) ? kKeepAll : (w0 < t && w1 < t) ? kDropAll : kDropMixed;
}
// indices first .. first + n - 1, n at most 2^L
template <int L>
__host__ __device__ __forceinline__ int dropout_run(uint32_t first, uint32_t n, uint32_t seed, uint32_t threshold) {
  const int a = dropout_block<L>(first, seed, threshold), b = dropout_block<L>(first + n - 1u, seed, threshold);
  return a == b ? a : kDropMixed;
}
inline DropoutParams make_dropout(float p, uint32_t seed, uint64_t rng_offset) {
  DropoutParams d;
  d.seed = seed;
  d.threshold = (uint32_t)(p * 4294967296.0f);       // fp32 product; fp32(4294967295) is 2^32
  d.offset = (uint32_t)rng_offset;
  d.keep_prob = 1.0f - p;
  d.keep_scale = 1.0f / d.keep_prob;
  d.keep_log2 = log2f(d.keep_scale);
  return d;
}

// Dropout where a lane owns a query row (forward and dQ kernels; flash_attention_triton.py:125,216-219,524-532): in the
// forward, P of a dropped element becomes zero after the row sums have been taken, and 1 / (1 - p) is applied with the
// normalisation of O. Hashing every element costs about twelve integer instructions per score, more than twice the rest
// of the softmax (forward, 12 heads x 8192 keys at head_dim 128: 559 us against 352 us without dropout). So at every
// kDropSpanTiles-th 64-key tile a wave looks at its rows' next 1024 elements as a whole (dropout_run): nearly always all of
// them are kept, or all dropped, or every row is one or the other. Where a row is neither, every tile of the span is
// looked at by itself, and the few rows for which that does not decide it either are hashed by the wave together, one
// element per lane. (Hashing such spans whole, or such tiles whole, is little work in total, but all of it falls on a few
// workgroups that the launch then waits for: 193 and 159 us at 12 heads x 4096 keys, where no dropout takes 124 us.)
// Forward at p = 0.1, head_dim 128, hashing every element -> this: 12 heads x 4096 keys 181 -> 133 us (no dropout 124), x 8192
// 562 -> 435 (364), x 2048 causal 62 -> 38 (32); head_dim 64, 8 x 12 heads x 1024 causal 44 -> 24 (25). What was left is the
// workgroups whose rows the mask's bands begin or end in, for which a launch of one workgroup per unit waits: the pipelined forward
// kernel reads the mask as words that are always there (Words) instead of asking every step whether it applies one, and the verdicts
// of a span's tiles are worked out together (look_at_span), over the tests per tile: 12 heads x 4096 132 -> 129 -> 124 us (no dropout
// 105), x 8192 437 -> 427 -> 410 (357), 6 x 3000 64 -> 59 -> 57 (44).
constexpr int kDropSpanTiles = 1024 / 64;
template <int QB>
struct DropRows {
  static constexpr int kRows = 3, kMasked = 4;
  int state = kKeepAll;                 // wave-uniform: kKeepAll, kDropAll, kRows (every row is one or the other), kMasked
  bool by_tile = false;
  uint32_t bits[QB][2];                 // all ones / all zeros: the lane's row of block b is kept / dropped; kMasked: the lane's row of block b: bit (r & 3) + 8 (r >> 2) of word kb = the element in register r of
                                        // the 32-key block kb is kept
  uint32_t tiles[QB];                   // by_tile: bit t = the lane's row of block b is kept over tile t of the span, bit 16 + t = dropped
  static __device__ __forceinline__ uint32_t index(const DropoutParams& d, int bh, int Sq, int Sk, int row, int key) {
    return d.offset + ((uint32_t)bh * (uint32_t)Sq + (uint32_t)row) * (uint32_t)Sk + (uint32_t)key;
  }
  // the state of key tile `tile` (of those from key0 on), asked for every tile in turn; row0: the wave's first row (block b is 32 b rows further)
  template <typename P>
  __device__ __forceinline__ void look(const P& d_in, int bh, int Sq, int Sk, int row0, int tile, int key0 = 0) {
    if (__builtin_expect(tile % kDropSpanTiles == 0, 0)) {      // (laid out away from the tile loops)
      const DropoutParams d = {d_in.seed, d_in.threshold, d_in.offset, 1.0f, 1.0f, 0.0f};
      look_at_span(d, bh, Sq, Sk, row0, key0 + tile * 64);
    }
    if (__builtin_expect(by_tile, 0)) {
      const DropoutParams d = {d_in.seed, d_in.threshold, d_in.offset, 1.0f, 1.0f, 0.0f};
      look_at_tile(d, bh, Sq, Sk, row0, tile % kDropSpanTiles, key0 + tile * 64);
    }
  }
  // The next kDropSpanTiles tiles from key0 on as a whole; where some row is neither kept nor dropped over all of them, every row's
  // verdict for each of the tiles. A tile's 64 elements lie in two of the 64-element blocks of dropout_block, neighbours share one: 17
  // blocks for the 16 tiles, nine by each half of the wave (which hold the same rows).
  __device__ __forceinline__ void look_at_span(const DropoutParams& d, int bh, int Sq, int Sk, int row0, int key0) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
    bool any_mixed = false, any_keep = false, any_drop = false;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const int v = dropout_run<10>(index(d, bh, Sq, Sk, row0 + 32 * b + l32, key0), 64 * kDropSpanTiles, d.seed, d.threshold);
      bits[b][0] = bits[b][1] = v == kKeepAll ? 0xFFFFFFFFu : 0u;
      any_keep |= __builtin_amdgcn_ballot_w64(v == kKeepAll) != 0;
      any_drop |= __builtin_amdgcn_ballot_w64(v == kDropAll) != 0;
      any_mixed |= __builtin_amdgcn_ballot_w64(v == kDropMixed) != 0;
    }
    state = any_keep && any_drop ? kRows : any_keep ? kKeepAll : kDropAll;
    by_tile = any_mixed;
    if (!any_mixed) return;
    constexpr int kHalf = kDropSpanTiles / 2;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      uint32_t at = index(d, bh, Sq, Sk, row0 + 32 * b + l32, key0 + 64 * kHalf * hh), keep = 0u, drop = 0u;
#pragma unroll 1
      for (int i = 0; i <= kHalf; ++i, at += 64u) {
        const int v = dropout_block<6>(at, d.seed, d.threshold);
        keep |= (v == kKeepAll ? 1u : 0u) << i;
        drop |= (v == kDropAll ? 1u : 0u) << i;
      }
      keep &= keep >> 1;
      drop &= drop >> 1;
      const uint32_t mine = (keep & ((1u << kHalf) - 1u)) | (drop & ((1u << kHalf) - 1u)) << kDropSpanTiles;
      const uint32_t other = __builtin_bit_cast(uint32_t, half_swap(__builtin_bit_cast(float, mine)));
      tiles[b] = hh ? other | mine << kHalf : mine | other << kHalf;
    }
  }
  // one of those tiles; its rows that are neither are hashed
  __device__ __forceinline__ void look_at_tile(const DropoutParams& d, int bh, int Sq, int Sk, int row0, int t, int key0) {
    const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
    uint64_t mixed_rows = 0, keep_rows = 0, drop_rows = 0;
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      const bool keep = (tiles[b] >> t) & 1u, drop_it = (tiles[b] >> (t + kDropSpanTiles)) & 1u;
      bits[b][0] = bits[b][1] = keep ? 0xFFFFFFFFu : 0u;
      keep_rows |= __builtin_amdgcn_ballot_w64(keep);
      drop_rows |= __builtin_amdgcn_ballot_w64(drop_it);
      const uint64_t neither = __builtin_amdgcn_ballot_w64(!keep && !drop_it);
      mixed_rows |= neither;
      uint32_t mixed = (uint32_t)neither;                       // (both halves of the wave hold the same rows)
      while (mixed != 0) {
        const int i = __builtin_ctz(mixed);
        mixed &= mixed - 1;
        const uint64_t k = __builtin_amdgcn_ballot_w64(dropout_keep(index(d, bh, Sq, Sk, row0 + 32 * b + i, key0 + lane), d.seed, d.threshold));
        if (l32 == i) { bits[b][0] = (uint32_t)k >> (4 * hh); bits[b][1] = (uint32_t)(k >> 32) >> (4 * hh); }
      }
    }
    state = mixed_rows != 0 ? kMasked : keep_rows != 0 && drop_rows != 0 ? kRows : keep_rows != 0 ? kKeepAll : kDropAll;
  }
  // What the pipelined forward kernel keeps of the state: an AND mask per pair of P values, word [kb][b][r / 2] for registers r and r + 1 of
  // 32-key block kb. Set where a span begins and at the tiles of a span that is looked at tile by tile; nothing else of a tile asks
  // what the state is.
  typedef uint32_t Words[2][QB][8];
  template <typename P>
  __device__ __forceinline__ void look(const P& d_in, int bh, int Sq, int Sk, int row0, int tile, Words& words, int key0) {
    if (__builtin_expect(tile % kDropSpanTiles != 0 && !by_tile, 1)) return;
    look(d_in, bh, Sq, Sk, row0, tile, key0);
    if (state == kMasked) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int w = 0; w < 8; ++w) {
            const int at = 2 * (w & 1) + 8 * (w >> 1);
            const uint32_t lo = (uint32_t)((int)(bits[b][kb] << (31 - at)) >> 31), hi = (uint32_t)((int)(bits[b][kb] << (30 - at)) >> 31);
            words[kb][b][w] = (lo & 0xFFFFu) | (hi & 0xFFFF0000u);
          }
    } else {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int w = 0; w < 8; ++w) words[kb][b][w] = bits[b][0];
    }
    // (opaque: the words stay in registers as they are)
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int w = 0; w < 8; ++w) asm volatile("" : "+v"(words[kb][b][w]));
  }
  // P of the 32-key block kb as two B operands (registers 0..7 and 8..15) per block of rows. (One branch, straight code where
  // whole rows are dropped: every taken branch holds up a wave that is alone on its SIMD, and with one per case and block a
  // workgroup with such rows took 30 % longer.)
  template <typename V>
  __device__ __forceinline__ void apply(int kb, V (&p)[QB][2]) const {
    typedef __attribute__((ext_vector_type(4))) uint32_t u4;
    if (__builtin_expect(state == kMasked, 0)) {
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          u4 w = __builtin_bit_cast(u4, p[b][t]);
#pragma unroll
          for (int u = 0; u < 8; u += 2) {
            const int at = (u & 3) + 8 * (u >> 2) + 16 * t;
            const uint32_t lo = (uint32_t)((int)(bits[b][kb] << (31 - at)) >> 31), hi = (uint32_t)((int)(bits[b][kb] << (30 - at)) >> 31);
            w[u >> 1] &= (lo & 0xFFFFu) | (hi & 0xFFFF0000u);
          }
          p[b][t] = __builtin_bit_cast(V, w);
        }
    } else {
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          u4 w = __builtin_bit_cast(u4, p[b][t]);
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] &= bits[b][0];
          p[b][t] = __builtin_bit_cast(V, w);
        }
    }
  }
  // a 64-key tile of fp32 values in two accumulators
  __device__ __forceinline__ void apply(f32x16 (&acc)[2]) const {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int at = (r & 3) + 8 * (r >> 2);
        const uint32_t m = (uint32_t)((int)(bits[0][kb] << (31 - at)) >> 31);
        const float x = acc[kb][r];                     // (a bit cast of the vector's element itself takes element 0)
        acc[kb][r] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & m);
      }
  }
};

// Additive bias on the scaled scores (flash_attention_triton.py:176-198, attention_ref.py:50-51): element
// (b, h, q, key) at bias + b*strides[0] + h*strides[1] + q*strides[2] + key, a stride of 0 broadcasting that dimension
// (the reference's "vector" bias is strides[2] == 0); fp32 or the operand type.
struct BiasParams {
  const void* ptr;
  int64_t strides[3];
  int is_f32;
  int dma_ok;   // forward: base and the three strides are multiples of 16 bytes, tiles may be copied with 16-byte pieces
  int lines;    // forward: those are multiples of 128 bytes, a cache line
  int vec_ok;   // base and the three strides are multiples of 4 elements: 4 consecutive keys may be read with one load
};
template <typename T>
__device__ __forceinline__ float load_bias(const BiasParams& bp, int64_t at) {
  return bp.is_f32 ? ((const float*)bp.ptr)[at] : (float)((const T*)bp.ptr)[at];
}
// four consecutive elements of type E (float or the operand type) from an address that is a multiple of 4 elements
template <typename E>
__device__ __forceinline__ void load_bias4(const E* at, float* out) {
  typedef __attribute__((ext_vector_type(4))) E e4;
  const e4 t = *(const e4*)at;
#pragma unroll
  for (int u = 0; u < 4; ++u) out[u] = (float)t[u];
}

// the same with 4 bytes per lane (LDS receives 256 bytes)
__device__ __forceinline__ void dma4_lane_ptr(const void* ptr, FO_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst)), "v"(ptr) : "memory", "m0");
#endif
}
// ... from a wave-uniform base plus a per-lane byte offset
__device__ __forceinline__ void dma4_uniform_base(const void* base, uint32_t byte_off, FO_LDS void* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)dst)), "v"(byte_off), "s"(base) : "memory", "m0");
#endif
}

// A bias with a query stride where a lane owns a query row (forward and dQ kernels): the wave's 32 rows x 64 keys of a key tile,
// copied straight into LDS (or KEYS of the keys), ELT bytes per element, ROW bytes per row; 16-byte piece s of a row holds the row's piece
// s ^ (row mod pieces), so that 32 rows' reads of the same piece are spread over the banks. One buffer per wave: once a
// tile's values are read (they start or join its score accumulators) the next tile's copy begins. Needs the
// 16-byte alignment of dma_ok. Pieces past the end re-read the last one that holds a key - of which the part behind the last
// key is read too, up to the next 16-byte boundary, and may hold anything - and rows past the end the last row; the kernels
// mask both after the bias has been applied.
template <typename T, int ELT, int KEYS = 64>
struct BiasRows {
  static constexpr int PIECE_KEYS = 16 / ELT, ROW = KEYS * ELT, PIECES = ROW / 16, ROWS_PER_DMA = 64 / PIECES, BYTES = 32 * ROW;
  // `row0`: element (b, h, 0, 0); q0w: the wave's first row
  static __device__ __forceinline__ void copy(const BiasParams& bp, int64_t row0, int q0w, int Sq, int Sk, int key0, FO_LDS char* dst, int lane_in) {
    int lane = lane_in;
    asm volatile("" : "+v"(lane));           // (computed anew per tile: no registers held across the loop)
#pragma unroll
    for (int i = 0; i < 32 / ROWS_PER_DMA; ++i) {
      const int row = i * ROWS_PER_DMA + lane / PIECES, piece = (lane % PIECES) ^ (row & (PIECES - 1));
      const int64_t at = row0 + (int64_t)min(q0w + row, Sq - 1) * bp.strides[2] + min(key0 + piece * PIECE_KEYS, (Sk - 1) / PIECE_KEYS * PIECE_KEYS);
      dma16_lane_ptr((const char*)bp.ptr + at * ELT, dst + i * 1024);
    }
  }
  // f(r, value) for registers 0..15 (four times four consecutive keys) of 32-key block kb of the lane's row
  template <typename F>
  static __device__ __forceinline__ void each(FO_LDS const char* src, int kb, int l32_in, int hh, F f) {
    int l32 = l32_in;
    asm volatile("" : "+v"(l32));            // (as in copy)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (ELT == 4) {
        const f32x4 v = *(FO_LDS const f32x4*)(src + l32 * ROW + (((8 * kb + 2 * j + hh) ^ (l32 & (PIECES - 1))) * 16));
#pragma unroll
        for (int u = 0; u < 4; ++u) f(4 * j + u, v[u]);
      } else {
        typedef __attribute__((ext_vector_type(4))) T vec4;
        const vec4 v = *(FO_LDS const vec4*)(src + l32 * ROW + (((4 * kb + j) ^ (l32 & (PIECES - 1))) * 16) + hh * 8);
#pragma unroll
        for (int u = 0; u < 4; ++u) f(4 * j + u, (float)v[u]);
      }
    }
  }
};

// Attention of a few query rows over many keys (attn_decode.hip)
struct DecodeParams {
  const void *q, *k, *v;
  void* o;
  float* lse;
  float* ws;                            // n_split > 1: decode_workspace_bytes() of it
  int B, H, Sq, Sk;
  int n_kv;                             // heads with keys of their own: H, or 1 (multi-query)
  int n_split;                          // workgroups that share the keys of a row block
  int64_t qs[3], ks[3], vs[3], os[3];   // element strides: batch, head, sequence
  float scale_log2e;
};
// rows that read the same keys, and 32-row blocks of them
__host__ __device__ inline int decode_rows(int H, int n_kv, int Sq) { return n_kv == 1 ? H * Sq : Sq; }
int decode_split(int B, int H, int n_kv, int Sq, int Sk, int D, int n_cu);
int64_t decode_workspace_bytes(int B, int H, int Sq, int D, int n_split);
template <typename T, int D> int launch_decode(const DecodeParams& p, hipStream_t stream);

}  // namespace fo
