// Which query tile each workgroup of the bidirectional prefill launch takes.  Plain C++ (the rule is also
// compiled and enumerated on the CPU).
//
// Workgroup b runs on XCD b % 8.  The XCDs take turns over the (sequence, kv head) pairs, so that each has tiles of
// every sequence: a contiguous eighth of the items per XCD gave them unequal lengths (6 sequences of 1023 to
// 1914 tokens, 16/8 heads: 185 us that way, 158 this way).  An XCD takes whole pairs, whose K/V then stays in its L2,
// where that shares the work: with kv heads that are a multiple of 8, or with at least as many pairs per XCD as a pair
// has query tiles (64 of 512 tokens, 4/4 heads: 53 us, in parts 56; contiguous eighths 55).  Otherwise it would leave
// XCDs idle (fewer than 8 pairs) or uneven (64 of 100 to 2000 tokens, 8/1 heads: 540, in parts 467; contiguous 568),
// and a pair is cut into 2, 4 or 8 interleaved parts of its query tiles, one per XCD.  The parts move on by one XCD
// from each round of 8 to the next, so over 8 pairs every XCD takes exactly num_qtiles tiles, and only the last,
// incomplete 8 leave workgroups without one.  (An empty workgroup costs the dispatcher as much as a short one: with a
// slot for every part whether or not it holds a tile, 2048 sequences of 30 tokens with 5 kv heads took 1992 us
// against 252, and with parts that stay on their XCD 7 of 600 tokens with 6 took 49 against 31.)
#pragma once

#include <algorithm>
#include <cstdint>

#ifdef __HIP__
#define OXR_HOST_DEVICE __host__ __device__
#else
#define OXR_HOST_DEVICE
#endif

namespace oxr {

struct QueryTile {
  int pair, tile;  // no tile when pair >= the number of pairs
};

inline int log2_parts(int num_kv_heads, int num_pairs, int num_qtiles) {
  if (num_pairs / 8 >= num_qtiles) return 0;
  return num_kv_heads % 8 == 0 ? 0 : num_kv_heads % 4 == 0 ? 1 : num_kv_heads % 2 == 0 ? 2 : 3;
}

// Tiles of a part (tiles part, part + parts, ... of num_qtiles).
OXR_HOST_DEVICE inline int part_tiles(int part, int num_qtiles, int log2_parts) {
  return (num_qtiles - part + (1 << log2_parts) - 1) >> log2_parts;
}

OXR_HOST_DEVICE inline QueryTile query_tile(int block, int num_qtiles, int log2_parts) {
  const int xcd = block & 7, slot = block >> 3, mask = (1 << log2_parts) - 1;
  const int eight = slot / num_qtiles;  // 8 pairs are num_qtiles workgroups of each XCD
  int left = slot - eight * num_qtiles, round = 0, part = xcd & mask;
  for (int n; left >= (n = part_tiles(part, num_qtiles, log2_parts)); ++round) {
    left -= n;
    part = (part - 1) & mask;
  }
  return {8 * eight + (round << (3 - log2_parts)) + (xcd >> log2_parts),
          num_qtiles - 1 - (part + (left << log2_parts))};
}

// Workgroups of the launch: up to the last that has a tile.
inline int64_t query_tile_blocks(int num_pairs, int num_qtiles, int log2_parts) {
  const int mask = (1 << log2_parts) - 1, rest = num_pairs % 8;
  const int64_t whole = (int64_t)(num_pairs / 8) * num_qtiles;  // slots of every XCD
  int64_t blocks = 8 * whole;
  for (int xcd = 0; xcd < 8; ++xcd) {
    int64_t slots = 0;
    for (int round = 0; (round << (3 - log2_parts)) + (xcd >> log2_parts) < rest; ++round)
      slots += part_tiles((xcd - round) & mask, num_qtiles, log2_parts);
    if (slots > 0) blocks = std::max(blocks, 8 * (whole + slots - 1) + xcd + 1);
  }
  return blocks;
}

}  // namespace oxr
