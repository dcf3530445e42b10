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
