"""The bidirectional prefill launch's rule from workgroups to query tiles (csrc/query_tiles.h), compiled for the CPU
and enumerated: every (pair, tile) has exactly one workgroup, the XCDs (workgroup b runs on XCD b % 8) get equal
shares, and no workgroup is without a tile but in the last, incomplete 8 pairs."""

from __future__ import annotations

import subprocess

import pytest

from conftest import PACKAGE, ROOT

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "query_tiles.h"
int main(int argc, char** argv) {
  const int kv = atoi(argv[1]);
  for (int i = 2; i + 1 < argc; i += 2) {
    const int pairs = kv * atoi(argv[i]), tiles = atoi(argv[i + 1]);
    const int parts = oxr::log2_parts(kv, pairs, tiles);
    const int64_t blocks = oxr::query_tile_blocks(pairs, tiles, parts);
    printf("%d %d %lld", pairs, tiles, (long long)blocks);
    for (int b = 0; b < blocks; ++b) {
      const oxr::QueryTile t = oxr::query_tile(b, tiles, parts);
      if (t.pair < pairs) printf(" %d %d %d", b, t.pair, t.tile);
    }
    printf("\n");
  }
  const int most = 8388607 / kv * kv;
  printf("%lld\n", (long long)oxr::query_tile_blocks(most, 1, oxr::log2_parts(kv, most, 1)));
}
"""

SIZES = [(seqs, tiles) for seqs in (1, 2, 3, 7, 8, 9, 31) for tiles in (1, 2, 3, 5, 7, 8, 9, 16, 33)]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    work = tmp_path_factory.mktemp("query_tiles")
    (work / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", f"-I{ROOT / PACKAGE / 'csrc'}", str(work / "main.cpp"), "-o",
                    str(work / "main")], check=True)
    return work / "main"


@pytest.mark.parametrize("kv", [1, 2, 3, 4, 5, 6, 8, 12, 16])
def test_every_tile_once_in_equal_shares(program, kv: int) -> None:
    args = [str(x) for size in SIZES for x in size]
    lines = subprocess.run([str(program), str(kv), *args], check=True, capture_output=True, text=True).stdout.splitlines()
    for line in lines[:-1]:
        pairs, tiles, blocks, *rest = map(int, line.split())
        items = list(zip(rest[0::3], rest[1::3], rest[2::3]))
        assert sorted((p, t) for _, p, t in items) == [(p, t) for p in range(pairs) for t in range(tiles)]
        per_xcd = [sum(b % 8 == x for b, _, _ in items) for x in range(8)]
        # Each 8 pairs are shared equally; the last 1 to 7 differ by no more than one pair's tiles.
        assert max(per_xcd) - min(per_xcd) <= (tiles if pairs % 8 else 0), (pairs, tiles, per_xcd)
        assert blocks == pairs * tiles or (pairs % 8 and pairs * tiles < blocks < pairs * tiles + 8 * tiles)
    assert int(lines[-1]) <= 8388607  # of 512 threads: the most a launch holds
