// How the dK/dV kernel that keeps dS shares key blocks between workgroups. Plain C++: the host plans, the kernels read the entries.
#pragma once
#include <cstdint>

namespace fo {

constexpr int kBwdWaves = 4;
constexpr int kBwdRows = 32 * kBwdWaves;   // rows (queries or keys) owned by a workgroup
constexpr int kBwdTile = 64;               // rows of a streamed tile

// An item of the dK/dV kernel that keeps dS: key block | piece << 8 | pieces << 12 | part << 16; the block's query tiles are shared by
// `pieces` workgroups, each of which leaves its sums in part `part` (of every head: see dkdv_part). A merge: key block | pieces << 12 |
// first part << 16.
constexpr int kMaxItems = 96, kMaxMerges = 48;
constexpr uint32_t kWholeBlock = 0xFFFF1000u;

// Which key blocks' query tiles several workgroups share (DkdvPlan). A workgroup of the dK/dV kernel has a compute unit to itself,
// so a launch takes as long as the unit that ends last: 12 heads x 3072 are 288 workgroups for 256 units, two rounds of which the
// second is an eighth full; causal they are 288 of 48, 46, ... 2 tiles; 4 heads x 2048 are 64. Every candidate (the blocks of the
// last round, or all, in 2 to 4 pieces; causal: those above a share of a unit's mean) is laid out as the hardware would, longest first,
// with two tiles' time to start a piece, one to leave its sums and 128 KiB of them to add; the best is taken if it ends before 0.82
// (causal 0.90) of the time of whole blocks: units that are idle let the others run at a higher clock, so that less than what is
// laid out is gained. Whole backward, whole blocks -> shared, us, in brackets the share laid out:
//   4 heads x 4096 causal, key bias, dropout 158 -> 109 (0.52); 6 x 3000 the same 131 -> 96 (0.60); 6 x 2500, dropout 120 -> 95 (0.68)
//   12 x 3072 237 -> 201, with a bf16 bias with a query stride 298 -> 253 (0.69); 8 x 3072 causal with one 121 -> 111 (0.73); 8 x 4096
//   causal 147 -> 138 (0.77); 12 x 6144 709 -> 661 (0.80); 12 x 3072 causal 134 -> 125, with a bias 152 -> 150 (0.89)
//   not taken: 12 x 4096 335 -> 348, with key bias and dropout 360 -> 352 (0.84: one line for all forms of a call, which these two lie on either
//   side of); 6 x 4096 165 -> 158 in 4 pieces (1.1)
constexpr int kMaxPieces = 4;
struct DkdvPlan {
  int n_items = 0, n_merges = 0, n_parts = 0;
  uint32_t items[kMaxItems], merges[kMaxMerges];
};
// when the last of n_bh workgroups for each of n entries (cost[], longest first) ends, each on that of `cus` units that is free first
inline int makespan(const int* cost, int n, int n_bh, int cus) {
  struct { int at, units; } grp[2 * kMaxItems + 2];      // units free from a time on, ascending
  int n_grp = 1, last = 0;
  grp[0] = {0, cus};
  for (int e = 0; e < n; ++e)
    for (int left = n_bh; left > 0;) {
      const int take = left < grp[0].units ? left : grp[0].units, end = grp[0].at + cost[e];
      left -= take;
      last = end > last ? end : last;
      if ((grp[0].units -= take) == 0) {
        for (int i = 1; i < n_grp; ++i) grp[i - 1] = grp[i];
        --n_grp;
      }
      int at = n_grp;
      while (at > 0 && grp[at - 1].at > end) --at;
      if (at > 0 && grp[at - 1].at == end) { grp[at - 1].units += take; continue; }
      for (int i = n_grp; i > at; --i) grp[i] = grp[i - 1];
      grp[at] = {end, take};
      ++n_grp;
    }
  return last;
}
// What a piece costs beside its tiles, in half tiles: to start it, to leave its sums; and to add them: for the launch, and parts that are
// added in the time of a half tile. The tiles a piece needs. Causal: whether every block in equally many pieces is laid out as well.
struct ShareCost { int start, leave, merge, parts_per, least; bool alike; };
// tiles(blk): of each of n_blk blocks; asked: 0 none are shared, > 1 every block in so many pieces, -1 what ends before `percent` of whole blocks
template <typename Tiles>
inline DkdvPlan share_blocks(int n_bh, int n_blk, Tiles tiles_of, bool causal, int asked, int cus, ShareCost price, int percent) {
  DkdvPlan best;
  int64_t sum = 0;
  int n_tiles[kMaxItems];
  for (int blk = 0; blk < n_blk; ++blk) sum += n_tiles[blk] = tiles_of(blk);
  auto tiles = [&](int blk) { return n_tiles[blk]; };
  const int mean = (int)((sum * n_bh + cus - 1) / cus);
  int cost[kMaxItems], best_time = 0;
  // pieces_of(blk) for every block -> entries, longest first; false if there are too many
  auto lay_out = [&](auto pieces_of, DkdvPlan& plan) -> bool {
    for (int blk = 0; blk < n_blk; ++blk) {
      const int s = pieces_of(blk);
      if (plan.n_items + s > kMaxItems || (s > 1 && plan.n_merges == kMaxMerges)) return false;
      if (s > 1) plan.merges[plan.n_merges++] = (uint32_t)blk | (uint32_t)s << 12 | (uint32_t)plan.n_parts << 16;
      for (int i = 0; i < s; ++i) {
        const uint32_t item = (uint32_t)blk | (uint32_t)i << 8 | (uint32_t)s << 12 | (s > 1 ? (uint32_t)plan.n_parts++ << 16 : kWholeBlock >> 16 << 16);
        const int c = 2 * (tiles(blk) * (i + 1) / s - tiles(blk) * i / s) + price.start + (s > 1 ? price.leave : 0);
        int at = plan.n_items++;
        for (; at > 0 && cost[at - 1] < c; --at) { cost[at] = cost[at - 1]; plan.items[at] = plan.items[at - 1]; }
        cost[at] = c;
        plan.items[at] = item;
      }
    }
    return true;
  };
  // the time of `cost` can be no less than its longest entry's, nor than all of it over all units
  auto at_least = [&](int64_t all, int longest) { const int64_t even = (all * n_bh + cus - 1) / cus; return even > longest ? even : longest; };
  auto consider = [&](auto pieces_of, bool forced) {
    // (most candidates are ruled out by that alone: 12 heads x 4096 causal, where nothing is shared, 14.8 -> 1.6 us of host time)
    if (!forced) {
      int64_t all = 0;
      int longest = 0, parts = 0;
      for (int blk = 0; blk < n_blk; ++blk) {
        const int s = pieces_of(blk), c = 2 * ((tiles(blk) + s - 1) / s) + price.start + (s > 1 ? price.leave : 0);
        all += 2 * tiles(blk) + s * (price.start + (s > 1 ? price.leave : 0));
        parts += s > 1 ? s : 0;
        longest = c > longest ? c : longest;
      }
      if (parts == 0 || at_least(all, longest) + (int64_t)parts * n_bh / price.parts_per + price.merge >= best_time) return;
    }
    DkdvPlan plan;
    if (!lay_out(pieces_of, plan) || plan.n_merges == 0) return;
    const int time = makespan(cost, plan.n_items, n_bh, cus) + plan.n_parts * n_bh / price.parts_per + price.merge;
    if (forced || time < best_time) { best_time = time; best = plan; }
  };
  if (asked > 1) {
    consider([&](int blk) { const int t = tiles(blk) / price.least; return t < 1 ? 1 : t < asked ? t : asked; }, true);
    return best;
  }
  DkdvPlan whole;
  if (!lay_out([](int) { return 1; }, whole)) return best;
  best_time = makespan(cost, whole.n_items, n_bh, cus) * percent / 100;
  constexpr int kMinTiles = 4;
  auto fits = [&](int blk, int s) { const int most = tiles(blk) / kMinTiles; return s < most ? s : most > 1 ? most : 1; };
  if (causal) {
    for (int f = 4; f >= 2; --f) {
      const int most = mean * f / 4 > kMinTiles ? mean * f / 4 : kMinTiles;
      consider([&](int blk) { const int s = (tiles(blk) + most - 1) / most; return fits(blk, s > kMaxPieces ? kMaxPieces : s); }, false);
    }
    for (int s = 2; price.alike && s <= kMaxPieces; ++s) consider([&](int blk) { return fits(blk, s); }, false);
  } else {
    const int rest = ((n_bh * n_blk) % cus + n_bh - 1) / n_bh;
    for (int s = 2; s <= kMaxPieces; ++s) {
      consider([&](int blk) { return blk >= n_blk - rest ? fits(blk, s) : 1; }, false);
      consider([&](int blk) { return fits(blk, s); }, false);
    }
  }
  return best;
}
inline DkdvPlan make_dkdv_plan(int n_bh, int Sq, int Sk, bool causal, int asked, int cus) {
  const int n_blk = (Sk + kBwdRows - 1) / kBwdRows, n_qt = (Sq + kBwdTile - 1) / kBwdTile;
  if (asked == 0 || n_blk > kMaxItems || n_bh > cus || (asked < 0 && (int64_t)n_bh * n_blk > 4 * cus)) return DkdvPlan();
  // (the heads in one group, see launch_bwd)
  if (2 * ((int64_t)Sq + Sk) * 128 * 2 * n_bh > (256ll << 20)) return DkdvPlan();
  auto tiles = [&](int blk) { const int first = kBwdRows / kBwdTile * blk; return causal ? (first < n_qt ? n_qt - first : 0) : n_qt; };
  return share_blocks(n_bh, n_blk, tiles, causal, asked, cus, {4, 2, 4, 32, 1, false}, causal ? 90 : 82);
}

}  // namespace fo
