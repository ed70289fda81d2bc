// What the translation units of the attention backward share: attn_bwd.hip (dK/dV and the dQ kernel that computes the scores
// again) and attn_bwd_dq_of_ds.hip (dQ from stored dS).
#pragma once
#include "attn_bwd_plan.hpp"
#include "attn_common.hpp"

namespace fo {

constexpr int kPartBytes = 2 * kBwdRows * 128 * 4;     // dK and dV of a block in fp32: each wave's accumulators, 1 KiB per four registers

struct AttnBwdParams {
  const void *q, *k, *v, *o, *d_o;
  const float* lse;
  float* delta;       // [B, H, Sq]: -rowsum(dO O) (1 - dropout_p), written by the dQ kernel (dS kept: by attn_bwd_rows_kernel)
  char* ds;           // not null: where the dK/dV kernel leaves dS for the dQ kernel (see ds_chunk)
  float* nlse;        // [B, H, Sq], written with delta: -LSE / softmax_scale (with dropout: of an LSE lower by log(1 / (1 - p))); dS kept, but for a bias
                      // with a query stride: -LSE log2 e of the same LSE
  void *dq, *dk, *dv;
  int B, H, Sq, Sk;
  int d;                // true head_dim: a multiple of 8, at most the D the kernels are compiled for
  int64_t qs[3], ks[3], vs[3], os[3], dos[3], dqs[3], dks[3], dvs[3];   // element strides: batch, head, sequence
  float scale, scale_log2e, neg_inv_scale_log2e;   // softmax scale, scale * log2 e, -1 / (scale * log2 e)
  int head_group;       // heads per group in the order of the workgroups (see bwd_item)
  DropoutParams drop;   // used by the kernels instantiated with dropout only
  BiasParams bias;      // used by the kernels instantiated with bias only
  // dS kept: how the query tiles of key blocks are shared (see kWholeBlock); n_items 0 = a workgroup per block, as bwd_item has it
  char* part;
  int n_items, n_merges;
  uint32_t items[kMaxItems], merges[kMaxMerges];
};

// Which (head, block) a workgroup of the dQ or dK/dV kernel owns. Blocks are numbered in the order they should start:
// when causal, the heaviest first (the last query blocks, the first key blocks), so that the light ones fill the gaps
// at the end. Taking every head's block 0, then every head's block 1, ... walks through the operands of all heads
// once per block index; with many heads they no longer stay in the caches between two visits (512 heads of 2 MiB:
// the kernels become HBM-bound), so the heads are taken in groups of head_group, group after group.
__device__ inline void bwd_item(const AttnBwdParams& prm, int n_blk, int& bh, int& blk) {
  const int n_bh = prm.B * prm.H, per_group = prm.head_group * n_blk;
  const int grp = blockIdx.x / per_group, r = blockIdx.x - grp * per_group;
  const int heads = min(prm.head_group, n_bh - grp * prm.head_group);
  bh = grp * prm.head_group + r % heads;
  blk = r / heads;
}

__device__ inline char* dkdv_part(const AttnBwdParams& prm, uint32_t part, int bh, int wave) {
  return prm.part + ((int64_t)part * prm.B * prm.H + bh) * kPartBytes + wave * (kPartBytes / kBwdWaves);
}

constexpr float kLog2e = 1.4426950408889634f;

// ---------------------------------------------------------------------------------------------------------------------
// dQ from stored dS, where that has room (ds_bytes_of): the dK/dV kernel runs first and leaves dS, rounded to the operand
// type for its own dK = dS^T Q, in memory, and dQ is one product of it with K. That saves computing S, dP and the exponential a second
// time - two of the backward's seven products - for 2 bytes written and read per (query, key) pair, which the memory-side cache
// holds for most of the sizes this is chosen at. The rows' LSE and delta then come from a kernel of their own.
//
// dS lies in chunks of 64 queries x 32 keys (4 KiB): block qb of 32 queries x group t of 16 queries, 1 KiB each; inside one, a key's 16
// queries are 32 bytes, in the order in which the dK/dV kernel's lanes hold them: position 8 hh + u is query (u & 3) + 8 (u >> 2) + 4 hh
// of the 16. The chunks of a query tile follow one another, as the dQ kernel reads them. Key k of group t stands at place k ^ 4 t: two groups' keys that one transposing LDS read takes lie in different banks.
constexpr int kDsChunk = 4096;
__host__ __device__ inline int64_t ds_key_blocks(int Sk) { return ((int64_t)Sk + kBwdRows - 1) / kBwdRows * (kBwdRows / 32); }
__host__ __device__ inline int64_t ds_query_tiles(int Sq) { return ((int64_t)Sq + kBwdTile - 1) / kBwdTile; }
// byte offset of the chunk of 32-key block kb and 64-query tile qt
__device__ inline int64_t ds_chunk(const AttnBwdParams& prm, int bh, int kb, int qt) {
  return (((int64_t)bh * ds_query_tiles(prm.Sq) + qt) * ds_key_blocks(prm.Sk) + kb) * kDsChunk;
}
// Two teams of waves in a workgroup of that kernel: the chain of tiles is half as long and a workgroup has its unit to itself, as two of one team would have it together. It
// gains where units would hold two and others one, or causal ones of unequal length, for a good while: this kernel, one team -> two, us,
//   causal: 12 x 3072 with a bias 47.1 -> 41.6, 12 x 4096 61.3 -> 50.8, 16 x 4096 74.0 -> 58.5, 4 x 8192 94.0 -> 83.8, 32 x 1800 36.1 -> 31.9,
//     12 x 6144 105 -> 98, 12 x 8192 (768 blocks) 171 -> 166; not: 32 x 4096 (1024) 122 -> 131, 64 x 1024 24.8 -> 26.1, 16 x 2048 (256) 25.1 -> 25.8
//   not causal: 12 x 3072 (288 blocks) 76.4 -> 68.7; not: 12 x 4096 (384) 90.4 -> 91.6, 24 x 2304 (432) 57.5 -> 60.1, 64 x 2048 110 -> 126
// and at other head dims the same: 24 x 2000 causal at 112 34.0 -> 26.8, 12 x 3000 causal 41.1 -> 37.8; not: 64 x 777 x 1250 at 80 (448) 30.5 -> 35.0,
// 24 x 1500 at 112 (288) 40.2 -> 40.7, 16 x 2000 at 96 (256) 25.2 -> 26.0.
inline bool dq_two_teams(int64_t n_bh, int Sq, int Sk, bool causal, int n_merges) {
  constexpr int kTwoTeamsFromKeys = 1536;
  const int asked = tune(g_attn_bwd_dq_teams);
  if (asked > 0) return asked == 2;
  const int64_t units = device_cus(), blocks = n_bh * ((Sq + kBwdRows - 1) / kBwdRows);
  return Sk >= kTwoTeamsFromKeys && (causal ? blocks + n_bh * n_merges > units && blocks <= 3 * units : blocks > units && blocks <= units + units / 4);
}
template <typename T> int launch_bwd_rows(const AttnBwdParams& p, bool drop, bool tile_bias, hipStream_t s);
template <typename T> int launch_dq_of_ds(const AttnBwdParams& p, bool causal, bool tile_bias, hipStream_t s);

// A wave's 32 finished gradient rows (accumulator layout: lane = row l32, registers 4*rg + u = columns
// 32*db + 8*rg + 4*hh + u) written to memory. Straight from the registers that is 8 bytes per lane to 32 different
// rows per instruction (4.3 us per workgroup for dK and dV, during which the workgroup's LDS and registers keep the
// next one waiting); instead the rows are rounded into LDS (`stage`, 32 rows padded by 16 bytes each, this wave's
// own) and leave as whole 16-byte pieces, 64 lanes covering consecutive rows. Rows from n_rows on and columns from the true head_dim `d` on are not written.
template <typename T, int D>
__device__ __forceinline__ void store_rows_via_lds(const f32x16 (&acc)[D / 32], float mul, FO_LDS char* stage, T* base, int64_t stride,
                                                   int row0, int n_rows, int d, int lane) {
  constexpr int ROW_BYTES = D * 2, OROW = ROW_BYTES + 16, CH = ROW_BYTES / 16;
  typedef __attribute__((ext_vector_type(4))) T vec4;
  typedef __attribute__((ext_vector_type(4))) int i32x4;
  const int l32 = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      vec4 o4;
#pragma unroll
      for (int u = 0; u < 4; ++u) o4[u] = (T)(acc[db][rg * 4 + u] * mul);
      *(FO_LDS vec4*)(stage + l32 * OROW + (32 * db + 8 * rg + 4 * hh) * 2) = o4;
    }
#pragma unroll
  for (int it = 0; it < 32 * CH / 64; ++it) {
    const int idx = it * 64 + lane, row = idx / CH, ch = idx % CH;
    const i32x4 piece = *(FO_LDS const i32x4*)(stage + row * OROW + ch * 16);
    if (row0 + row < n_rows && ch * 8 < d) *(i32x4*)(base + (int64_t)(row0 + row) * stride + ch * 8) = piece;
  }
}
constexpr int stage_bytes(int D) { return 32 * (D * 2 + 16); }   // per wave and matrix

}  // namespace fo
