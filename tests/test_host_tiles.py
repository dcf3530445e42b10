"""Rows of the LDS-tiled grouped GEMMs' tiles, from the header that the kernels take them from (CPU only)."""

from __future__ import annotations

import os
import subprocess

import pytest

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


def tiles_of(rows, height):
    return sum(-(-r // height) for r in rows)


@pytest.mark.parametrize("fp8,H,I,rows,height", [
    (1, 2048, 768, [144] * 16, 128),  # 32 tiles of 128 rows x 8 column blocks: a CU for each item
    (0, 2048, 768, [144] * 16, 128),
    (1, 2048, 768, [144] * 17, 192),
    (0, 2048, 768, [144] * 17, 192),
    (1, 2048, 768, [64] * 128, 192),
    (1, 2048, 768, [3000] + [0] * 15, 128),
    (1, 512, 512, [129] * 32, 128),   # 64 tiles x 4 column blocks
    (1, 512, 512, [129] * 33, 192),
    (1, 4096, 1536, [144] * 4, 144),  # exact accumulation
    (0, 4096, 1536, [144] * 8, 128),
    (1, 2048, 768, [8] * 16, 16),     # 8 pairs per expert: streaming tiles
    (1, 384, 512, [144] * 4, 64),     # H % 256 != 0: as before
])
def test_tile_height_by_items(pkg, fp8, H, I, rows, height):
    """128-row tiles where all their work items run at once on 256 CUs, else the tallest."""
    lib = pkg._lib.load()
    assert lib.moe_mi355x_experts_tile_rows(sum(rows), H, I, len(rows), 1, fp8, tiles_of(rows, 128)) == height
