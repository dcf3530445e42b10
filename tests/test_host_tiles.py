"""Rows of the LDS-tiled grouped GEMMs' tiles, from the header that the kernels take them from (CPU only)."""

from __future__ import annotations

import os
import subprocess

import pytest

from tests.helpers import tile_rows

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "inference-server_amd", "csrc")


@pytest.mark.parametrize("exact,rows", [(0, 192), (1, 144)])
def test_groups_read_their_own_rows(tmp_path, exact, rows):
    """The fragments that the two wave groups read are the rows of an activation slot, each once and none past
    its end (144 rows: five fragments of group 0, four of group 1)."""
    src = tmp_path / "rows.cc"
    src.write_text("""#include <cstdio>
#include "prefill_rows.h"
int main() {
  const int rows = moe_prefill_rows(%d);
  for (int g = 0; g < 2; ++g)
    for (int mi = 0; mi < pf_group_frags(rows, g); ++mi)
      for (int r = 0; r < 16; ++r) std::printf("%%d\\n", pf_group_row0(rows, g) + 16 * mi + r);
}
""" % exact)
    exe = tmp_path / "rows"
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    read = [int(v) for v in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()]
    assert read == list(range(rows))


@pytest.mark.parametrize("fp8,H,I,rows,height", [
    (1, 2048, 768, [144] * 16, 128),  # 32 tiles of 128 rows x 8 column blocks: a CU for each item
    (0, 2048, 768, [144] * 16, 128),
    (1, 2048, 768, [144] * 17, 192),  # one round of 192-row tiles, two of 128-row ones
    (0, 2048, 768, [144] * 17, 192),
    (1, 2048, 768, [190] * 8 + [210] * 24, 128),  # 64 and 56 tiles, two rounds of either
    (0, 2048, 768, [190] * 8 + [210] * 24, 128),
    (1, 2048, 768, [430] * 16, 128),  # 64 and 48 tiles, two rounds of either
    (0, 2048, 768, [430] * 16, 128),
    (1, 2048, 768, [300] * 16, 192),  # 48 and 32 tiles: two rounds and one
    (1, 2048, 768, [150] * 128, 192),
    (1, 2048, 768, [64] * 128, 128),  # one tile each, whatever the height
    (1, 2048, 768, [3000] + [0] * 15, 128),
    (1, 512, 512, [129] * 32, 128),   # 64 tiles x 4 column blocks
    (1, 512, 512, [129] * 33, 192),
    (1, 4096, 1536, [144] * 4, 144),  # exact accumulation
    (0, 4096, 1536, [144] * 8, 128),
    (1, 2048, 768, [8] * 16, 16),     # 8 pairs per expert: streaming tiles
    (1, 384, 512, [144] * 4, 64),     # H % 256 != 0: as before
])
def test_tile_height_by_items(pkg, fp8, H, I, rows, height):
    """On 256 CUs: 128-row tiles where they take no more rounds of work items, else the tallest."""
    assert tile_rows(pkg, rows, sum(rows), H, I, 1, fp8)[0] == height


@pytest.mark.parametrize("H,most", [(2048, 192), (4096, 144)])
def test_an_experts_tiles_are_equally_high(pkg, H, most):
    """As few tiles as the height allows, in whole 16-row fragments, none a fragment per tile or more below
    another; on streaming tiles every tile but the last is full."""
    counts = list(range(1, 1200, 7)) + [143, 144, 145, 191, 192, 193, 288, 289, 384, 385, 576, 577, 0]
    for part in (counts[i:i + 64] for i in range(0, len(counts), 64)):
        got, rows = tile_rows(pkg, part, sum(part), H, 1536, 1, 1)
        assert got in (128, most)
        for n, h in zip(part, rows.tolist()):
            tiles = -(-n // got)
            assert 0 < h <= got and h % 16 == 0 and -(-n // h) == tiles
            if tiles > 1:
                assert h - (n - (tiles - 1) * h) < 16 * tiles
    got, rows = tile_rows(pkg, [40] + [1] * 7, 47, H, 1536, 1, 1)
    assert got == 16 and (rows == 16).all()
