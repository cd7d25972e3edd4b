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

// `q8act`: Q4_0 under MER_MOE_QMM.  Sizes are those that mer_hip_moe_grouped
// accepts: d_model and d_ff multiples of 64, n_tok * top_k <=
// kMaxGroupedPairs, 1 <= table_len <= kMaxGroupedExperts.
inline GroupedPlan plan_grouped(bool q8act, size_t d_model, size_t d_ff, uint32_t n_tok, uint32_t top_k,
                                uint32_t table_len) {
  GroupedPlan pl{};
  const uint32_t n_pairs = n_tok * top_k;
  const uint32_t max_experts = n_pairs < table_len ? n_pairs : table_len;
  const size_t xblocks = d_model / 32, hblocks = d_ff / 32;
  // Tiles of 64 pairs on f16 MFMA (gbig) from 16 pairs per expert on average,
  // or 8 where the experts alone give the 512 resident workgroups four
  // rounds; else the int8 kernel's tiles of 16.  Call us, int8 / f16, at 8
  // pairs: Qwen3 Q8_0 138 / 158, Mixtral Q4_0 282 / 287, DeepSeek-V3 Q4_0
  // (4096 workgroups) 1424 / 1119; at 16 pairs: 208 / 207, 434 / 302, 2290 /
  // 1600; Mixtral under MER_MOE_QMM at 8 and 16: 279 / 331, 433 / 342.
  const size_t expert_wgs = (size_t)max_experts * ((2 * d_ff + 255) / 256);
  const bool big = n_pairs >= 16 * max_experts || (n_pairs >= 8 * max_experts && expert_wgs >= 2048);
  pl.mode = !big ? kGroupDigits : q8act ? kGroupQ8Act : kGroupF16Pair;
  const uint32_t tile_pairs = big ? 64u : 16u;
  // At most n_pairs / tile_pairs full tiles plus one partial tile per
  // distinct expert.
  pl.max_tiles = n_pairs / tile_pairs + max_experts;
  // Down rows in up to 4 K parts (whole 4-block stages, about 64 blocks or
  // more) until 2048 workgroups share the launch: 512 run at once, and a short
  // last round of whole rows idles the chip.  Mixtral Q4_0 down, us with one
  // part / with parts: 64 tokens 195 / 94, 128 tokens 281 / 119, 2048 tokens
  // 1200 / 1105 (combine 20 / 33).
  pl.n_parts = 1;
  if (big) {
    const size_t wgs = (n_pairs / tile_pairs + (max_experts + 1) / 2) * ((d_model + 255) / 256);
    while (pl.n_parts < 4 && wgs * pl.n_parts < 2048 && hblocks >= 128 * pl.n_parts) pl.n_parts *= 2;
  }

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
