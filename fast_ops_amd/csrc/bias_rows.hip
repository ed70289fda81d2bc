// A bias whose rows do not start on 16-byte boundaries (an odd number of keys), copied into rows that do. The attention kernels
// copy tiles of a bias with a query stride straight into LDS in 16-byte pieces, which such rows do not allow: element by
// element instead, every lane of its own row, the backward took 1161 us at 12 heads x 3071 causal (bf16 bias), where the copy
// costs 100 us (HBM-bound: every element read and written once) and what follows 180.
#include "common.hpp"

namespace fo {

// 16 bytes of a row of `out` per lane; the elements behind the last key of a row become zero
template <typename E>
__global__ void __launch_bounds__(256) bias_rows_kernel(const E* __restrict__ in, int64_t sb, int64_t sh, int64_t sq, E* __restrict__ out,
                                                        int64_t out_row, int64_t n_pieces, int H, int Sq, int Sk) {
  constexpr int N = 16 / sizeof(E);
  typedef E vec __attribute__((ext_vector_type(N)));
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (at >= n_pieces) return;
  const int64_t per_row = out_row / N, row = at / per_row;
  const int key = (int)(at - row * per_row) * N;
  const int64_t bh = row / Sq, q = row - bh * Sq, b = bh / H, h = bh - b * H;
  const E* src = in + b * sb + h * sh + q * sq + key;
  vec v;
  if (key + N <= Sk) {
    __builtin_memcpy(&v, src, 16);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = key + i < Sk ? src[i] : (E)0;
  }
  *(vec*)(out + row * out_row + key) = v;
}

}  // namespace fo

extern "C" int fo_attn_bias_rows(const void* bias, const int64_t* strides, int elt_bytes, int B, int H, int Sq, int Sk, void* out, int64_t out_row,
                                 void* stream) {
  if (!bias || !strides || !out) return FO_ERR_NULL_POINTER;
  if (elt_bytes != 2 && elt_bytes != 4) return FO_ERR_BAD_DTYPE;
  if (B <= 0 || H <= 0 || Sq <= 0 || Sk <= 0 || out_row < Sk || (int64_t)B * H > 0x7FFFFFFFll || out_row > (1ll << 31)) return FO_ERR_BAD_SHAPE;
  if (strides[0] < 0 || strides[1] < 0 || strides[2] < 0 || out_row * elt_bytes % 16 != 0) return FO_ERR_BAD_STRIDE;
  if (((uintptr_t)bias & (uintptr_t)(elt_bytes - 1)) || ((uintptr_t)out & 15u)) return FO_ERR_MISALIGNED;
  const int64_t rows = (int64_t)B * H * Sq, per_row = out_row * elt_bytes / 16;
  if (rows > (1ll << 40) / per_row) return FO_ERR_BAD_SHAPE;
  const int64_t n = rows * per_row, blocks = (n + 255) / 256;
  if (blocks > 0x7FFFFFFFll) return FO_ERR_BAD_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (elt_bytes == 2)
    fo::bias_rows_kernel<uint16_t><<<(unsigned)blocks, 256, 0, s>>>((const uint16_t*)bias, strides[0], strides[1], strides[2], (uint16_t*)out, out_row, n, H, Sq, Sk);
  else
    fo::bias_rows_kernel<uint32_t><<<(unsigned)blocks, 256, 0, s>>>((const uint32_t*)bias, strides[0], strides[1], strides[2], (uint32_t*)out, out_row, n, H, Sq, Sk);
  return fo::launch_status();
}
