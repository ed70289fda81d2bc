// How the pipelined 128-row forward kernel shares the keys of a query block between workgroups. Plain C++, as attn_bwd_plan.hpp.
#pragma once
#include "attn_bwd_plan.hpp"

namespace fo {

// The same question as for the dK/dV kernel (make_dkdv_plan), of query blocks: a workgroup has a compute unit to itself, so few heads leave
// most of the chip idle and a causal launch waits for its longest block. The workgroups of a shared block leave O, not yet normalised, and
// each row's reference and sum in fp32, and a second launch adds them in order. Entries as there (key tiles in the place of query
// tiles); a piece has two tiles at least: causal, every row of the block then sees a key of the last one.
// The price of a piece: timed over 4 to 16 heads x 1024 to 8192 keys, whole blocks and every block in two and three pieces, a launch at
// head_dim 128 without bias and dropout takes 0.66 us per tile of the longest chain of workgroups, with 6 tiles for each workgroup of it,
// and 0.23 to 0.26 per tile of the mean; 3.5 us for the merge and 1.5 per hundred parts (residuals 3.4 % rms, 8 % at most). The same
// prices serve the other calls, which they fit less well: fitted to each, residuals are 5 % with a padding mask and dropout and 6 to 9 % at
// head_dim 64, where without a bias two workgroups share a unit and the plan counts one. What is chosen took at most 1.5 % longer than
// whole blocks in any of 184 calls. Not causal only up to 5/4 of a round of whole blocks: from there on all units work all the time, at the clock
// their power leaves (12 x 4096, 384 blocks: in two pieces at head_dim 64 70 -> 70 us, at 128 120 -> 124, with a padding mask and dropout 144 ->
// 139, but plain 134).
// Whole blocks -> shared, us, without bias; with a padding mask and dropout 0.1; with a bf16 bias per query:
//   head_dim 128: 4 x 2048 31.7 -> 27.2, 45.0 -> 28.6, 41.0 -> 27.8; causal 31.6 -> 23.4, 40.1 -> 25.8, 41.6 -> 25.5; 4 x 4096 56.5 -> 49.4, 79.9 ->
//     55.3, 74.1 -> 56.4; causal 54.7 -> 37.6, 67.4 -> 41.3, 73.6 -> 46.3; 6 x 4096 causal 56.3 -> 45.2, 71.0 -> 49.4, 74.6 -> 56.6; 8 x 3000
//     causal 43.2 -> 39.4, 54.0 -> 42.2, 57.5 -> 47.6; 12 x 3072 (288 blocks; whole ones on the plain kernel) 85.6 -> 72.8, 103 -> 82.1, 112 ->
//     95.4; 4 x 8192 causal 105 -> 88, 131 -> 103
//   head_dim 64: 4 x 2048 24.9 -> 18.7, 38.4 -> 20.6, 34.7 -> 21.4; 6 x 4096 causal 44.3 -> 33.5, 57.4 -> 39.0, 63.0 -> 44.3; 12 x 3072 51.3 ->
//     42.8, 74.2 (plain) -> 62.2, 82.9 (plain) -> 70.5
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
