// mer_grouped_plan.hpp -- how a grouped call is cut and what scratch it needs
// (run_grouped, mer_grouped.hip).  Host arithmetic on sizes only, without
// HIP, so that it can be compiled and checked anywhere.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace mer {

constexpr uint32_t kMaxGroupedExperts = 4096;  // table entries the grouping kernel counts in LDS
constexpr uint32_t kMaxGroupedPairs = 4096;    // routed (token, slot) pairs per call
constexpr uint32_t kGroupRecDwords = 32;       // one block's input record, in every mode

// Input formats of the projection kernels (mer_grouped.hip).
enum GroupMode : uint32_t { kGroupDigits = 0, kGroupQ8Act = 1, kGroupF16Pair = 2 };

struct GroupTile {
  const uint8_t *blob;  // the expert's blob
  uint32_t start;       // first pair of the tile in plist
  uint32_t count;       // pairs in the tile: 1..16 (kGroupDigits) or 1..64
};

struct GroupedPlan {
  GroupMode mode;
  uint32_t max_tiles;  // token tiles the grouping kernel emits at most
  uint32_t n_parts;    // K parts of the down projection
  uint32_t part_blocks;  // 32-weight blocks of each
  // Scratch regions, in floats from its start (the first 64 hold the tile
  // count), 256-byte aligned.  h is held as f32 and then, in place, as
  // records: a block of 32 elements takes 128 bytes either way.
  size_t plist, pair_ok, tiles, xg, hg, xs, hs, partial;
  size_t need;  // floats with the down projection in one part
  size_t want;  // floats for the parts of this call and of any smaller one
};

// K parts of the down projection that the sums' region holds, if the scratch
// has `floats`.
inline void fit_parts(GroupedPlan &pl, uint32_t n_pairs, size_t d_model, size_t d_ff, size_t floats) {
  const size_t one = (size_t)n_pairs * d_model;
  const uint32_t hblocks = (uint32_t)(d_ff / 32);
  while (pl.n_parts > 1 && pl.partial + pl.n_parts * one > floats) pl.n_parts /= 2;
  // whole stages of four blocks
  pl.part_blocks = pl.n_parts == 1 ? hblocks : (hblocks + 4 * pl.n_parts - 1) / (4 * pl.n_parts) * 4;
  pl.n_parts = (hblocks + pl.part_blocks - 1) / pl.part_blocks;
}

// `q4`: Q4_0 weights, else Q8_0; `q8act`: Q4_0 under MER_MOE_QMM.  Sizes are
// those that mer_hip_moe_grouped accepts: d_model and d_ff multiples of 64,
// n_tok * top_k <= kMaxGroupedPairs, 1 <= table_len <= kMaxGroupedExperts.
inline GroupedPlan plan_grouped(bool q4, bool q8act, size_t d_model, size_t d_ff, uint32_t n_tok, uint32_t top_k,
                                uint32_t table_len) {
  GroupedPlan pl{};
  const uint32_t n_pairs = n_tok * top_k;
  const uint32_t max_experts = n_pairs < table_len ? n_pairs : table_len;
  const size_t xblocks = d_model / 32, hblocks = d_ff / 32;
  // Down rows in up to 4 K parts (whole 4-block stages, about 64 blocks or
  // more) until 2048 workgroups share the launch: 512 run at once, and a short
  // last round of whole rows idles the chip.  Mixtral Q4_0 down, us with one
  // part / with parts: 64 tokens 195 / 94, 128 tokens 281 / 119, 2048 tokens
  // 1200 / 1105 (combine 20 / 33).
  const size_t gate_tiles = (2 * d_ff + 255) / 256, down_tiles = (d_model + 255) / 256;
  pl.n_parts = 1;
  const size_t wgs = (n_pairs / 64 + (max_experts + 1) / 2) * down_tiles;
  while (pl.n_parts < 4 && wgs * pl.n_parts < 2048 && hblocks >= 128 * pl.n_parts) pl.n_parts *= 2;

  // Tiles of 64 pairs on f16 MFMA (gbig), or the int8 kernel's tiles of 16.
  // An f16 workgroup is one chain over K (0.3 us a block) whatever its pairs,
  // so it takes pairs enough to fill the tiles and workgroups enough to fill
  // the chip: `at_once`, those of a projection on average over the blocks of
  // K that they walk (64-pair tiles, and half a one per expert).  Few pairs
  // need more of them.  Few workgroups still win where the parts shorten long
  // down rows, which the int8 kernel walks whole.  Q4_0 wins from fewer pairs,
  // given workgroups for several rounds (QMatMul's sums carry a scale per
  // pair, and Q8_0 moves twice the bytes).
  //
  // Call us, int8 / f16, experts picked at random, at about 8, 12, 16 and 20
  // pairs an expert: 256 x (7168 x 2048) Q4_0 2043 / 1943, 2294 / 2006, 2806 /
  // 2066 (8, 12, 16), QMatMul 1985 / 2122, 2197 / 2166, 2694 / 2227, Q8_0 2870
  // / 3069, 3105 / 3146, 3745 / 3229; 8 x (4096 x 14336) Q4_0 280 / 286, 295 /
  // 289, 407 / 298, 460 / 303, QMatMul 277 / 324, 294 / 329, 409 / 334, 444 /
  // 340.  At 40 and more pairs on few workgroups: 1 x (4096 x 1536) Q8_0, 48
  // pairs, 46 / 137; 4 x (4096 x 384) Q8_0, 59 each, 43 / 119; on short chains
  // 2 x (512 x 13760) Q8_0, 17 each, 134 / 73.  Over 1803 calls of random
  // sizes and routes the choice costs 0.6% on average against the faster
  // kernel each time (always int8: 11%; f16 wherever there are 16 pairs an
  // expert: 14%); 30 of the 684 calls that it gives to f16 are 2 to 16% slower
  // there, most where a few experts take most pairs.
  const size_t tiles2 = n_pairs / 32 + max_experts;  // twice the tiles
  const size_t chain = xblocks + hblocks / pl.n_parts;
  const size_t at_once = tiles2 * (gate_tiles * xblocks + down_tiles * hblocks) / (2 * chain);
  bool big = n_pairs >= 16 * max_experts &&
             ((at_once >= 160 && n_pairs * at_once >= 4000 * (size_t)max_experts) || (pl.n_parts == 4 && d_ff >= 4 * d_model));
  if (q4 && !q8act)
    big = big || (n_pairs >= 12 * max_experts && at_once >= 512) || (n_pairs >= 8 * max_experts && at_once >= 1600);
  pl.mode = !big ? kGroupDigits : q8act ? kGroupQ8Act : kGroupF16Pair;
  if (!big) pl.n_parts = 1;
  const uint32_t tile_pairs = big ? 64u : 16u;
  // At most n_pairs / tile_pairs full tiles plus one partial tile per
  // distinct expert.
  pl.max_tiles = n_pairs / tile_pairs + max_experts;

  // Scratch.  A call that is no larger than an earlier one in any size must
  // not make the workspace grow (a captured graph holds its addresses), while
  // the kernel and the number of parts change back and forth with the sizes:
  // so every region is one function of the sizes for all kernels, growing in
  // each of them, and the sums' region is that of the most parts a smaller
  // call could take: n_parts > 1 needs wgs * n_parts < 4096, each workgroup
  // 64 pairs by 256 rows, so n_parts * n_pairs * d_model < 2^26.
  auto up64 = [](size_t v) { return (v + 63) / 64 * 64; };
  size_t at = 64;
  auto region = [&](size_t floats) {
    const size_t r = at;
    at += up64(floats);
    return r;
  };
  pl.plist = region(n_pairs);
  pl.pair_ok = region(n_pairs);
  pl.tiles = region((size_t)(n_pairs / 16 + max_experts) * sizeof(GroupTile) / 4);
  pl.xg = region((size_t)n_tok * xblocks * kGroupRecDwords);
  pl.hg = region((size_t)n_pairs * hblocks * kGroupRecDwords);
  pl.xs = region(n_tok);
  pl.hs = region(n_pairs);
  pl.partial = at;
  const size_t one = (size_t)n_pairs * d_model, most = (hblocks >= 256 ? 4 : hblocks >= 128 ? 2 : 1) * one;
  const size_t cap = size_t(1) << 26;
  pl.need = at + up64(one);
  pl.want = at + up64(most < cap ? most : cap > one ? cap : one);
  fit_parts(pl, n_pairs, d_model, d_ff, pl.want);
  return pl;
}

}  // namespace mer
