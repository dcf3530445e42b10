// Rows of the LDS-tiled grouped GEMMs' tiles: their height, and the wave group that holds each 16-row
// fragment.  Plain constexpr C++, for host and device.
#pragma once

// Rows per tile at most.
constexpr int moe_prefill_rows(bool exact) { return exact ? 144 : 192; }

// Lower tiles where those fit the chip at once: with at most this many tiles of kPrefillLowRows rows, every
// work item (tile, column block) of both GEMMs has a CU of its own, and a launch takes as long as its
// tallest tile.  With more, the taller tiles' single pass over an expert's weights counts.  Qwen3-30B-A3B
// experts, gate_up + down on 192- / 128-row tiles: 16 experts with 144 rows each (256 items of 128-row
// tiles) FP8 31.5 + 20.7 / 27.3 + 16.4 us, bf16 44.1 + 27.6 / 39.8 + 22.3; 24 experts (384 items) FP8 36.2 +
// 20.6 / 48.1 + 25.9, bf16 51.9 + 28.6 / 71.2 + 36.1.  Exact accumulation: 144 rows throughout (16 experts of
// Qwen3-235B-A22B leave no room, 8 are level).
constexpr int kPrefillLowRows = 128;
constexpr int moe_prefill_low_tiles(bool exact, int H, int I, int cus) {
  return exact ? 0 : cus / (H / 256 > I / 128 ? H / 256 : I / 128);
}

// 16-row fragments of a full tile of `rows` rows that wave group g (0 or 1) holds: those numbered 2 m + g.
constexpr int pf_group_frags(int rows, int g) { return (rows / 16 - g + 1) / 2; }

// First row of group g's part of an activation slot of `rows` rows: group 0's rows, then group 1's.
constexpr int pf_group_row0(int rows, int g) { return g == 0 ? 0 : 16 * pf_group_frags(rows, 0); }

static_assert(pf_group_row0(moe_prefill_rows(true), 1) + 16 * pf_group_frags(moe_prefill_rows(true), 1) ==
                  moe_prefill_rows(true),
              "the groups' parts fill a slot and end with it");
