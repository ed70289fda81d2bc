// How the pipelined 128-row forward kernel shares the keys of a query block between workgroups. Plain C++, as attn_bwd_plan.hpp.
#pragma once
#include "attn_bwd_plan.hpp"

namespace fo {

// The same question as for the dK/dV kernel (make_dkdv_plan), of query blocks: a workgroup has a compute unit to itself, so few heads leave
// most of the chip idle and a causal launch waits for its longest block. The workgroups of a shared block leave O, not yet normalised, and
// each row's reference and sum in fp32, and a second launch adds them in order. Entries as there (key tiles in the place of query
// tiles); a piece has two tiles at least: causal, every row of the block then sees a key of the last one.
// The price of a piece: timed over 4 to 16 heads x 1024 to 8192 keys, whole blocks and every block in two and three pieces, a launch at
// head_dim 128 takes 0.66 us per tile of the longest chain of workgroups, with 6 tiles for each workgroup of it, and 0.26 per tile of the
// mean; 3.3 us for the merge and 1.5 per hundred parts (to 3 %). Not causal only up to 5/4 of a round of whole blocks: from there on all
// units work all the time, at the clock their power leaves (12 x 4096, 384 blocks, at head_dim 64 70 -> 82 us).
// Whole blocks -> shared, us, without bias; with a padding mask and dropout 0.1; with a bf16 bias per query:
//   head_dim 128: 4 x 2048 33.6 -> 28.0, 44.0 -> 29.5, 40.2 -> 27.7; causal 32.1 -> 23.7, 39.2 -> 25.8, 40.9 -> 25.8; 4 x 4096 57.5 -> 49.6, 76.0 ->
//     54.3, 86.6 -> 62.4; causal 55.6 -> 37.3, 65.0 -> 39.8, 73.0 -> 47.2; 6 x 4096 causal 56.5 -> 44.0, 67.2 -> 47.3, 86.0 -> 61.1; 8 x 3000
//     causal 44.7 -> 38.9, 52.9 -> 41.2, 85.1 -> 58.9; 12 x 3072 (288 blocks; whole ones on the plain kernel) 85.5 -> 72.7, 100 -> 81.3, 115 ->
//     103; 4 x 8192 causal 106 -> 88, 126 -> 100
//   head_dim 64: 4 x 2048 25.8 -> 19.3, 36.8 -> 20.9, 33.7 -> 21.4; 6 x 4096 causal 45.0 -> 33.8, 52.7 -> 36.5, 62.9 -> 44.2; 12 x 3072 53.0 ->
//     42.6, 81.3 -> 59.6, 86.4 -> 74.4
constexpr int kFwdPlanRows = 128, kFwdPlanKeys = 64;
constexpr int fwd_plan_tiles(int blk, int Sk, bool causal) {
  const int all = (Sk + kFwdPlanKeys - 1) / kFwdPlanKeys, seen = kFwdPlanRows / kFwdPlanKeys * (blk + 1);
  return causal && seen < all ? seen : all;
}
inline DkdvPlan make_fwd_plan(int n_bh, int Sq, int Sk, bool causal, int asked, int cus) {
  const int n_blk = (Sq + kFwdPlanRows - 1) / kFwdPlanRows;
  if (asked == 0 || n_blk > kMaxItems || n_bh > cus || (asked < 0 && (int64_t)n_bh * n_blk > (causal ? 4 * cus : cus + cus / 4))) return DkdvPlan();
  return share_blocks(n_bh, n_blk, [&](int blk) { return fwd_plan_tiles(blk, Sk, causal); }, causal, asked, cus, {12, 2, 10, 24, 2, true}, 94);
}

}  // namespace fo
