// Rows of the LDS-tiled grouped GEMMs' tiles: their height, and the wave group that holds each 16-row
// fragment.  Plain constexpr C++, for host and device.
#pragma once

// Rows per tile.
constexpr int moe_prefill_rows(bool exact) { return exact ? 144 : 192; }

// 16-row fragments of a full tile of `rows` rows that wave group g (0 or 1) holds: those numbered 2 m + g.
constexpr int pf_group_frags(int rows, int g) { return (rows / 16 - g + 1) / 2; }

// First row of group g's part of an activation slot of `rows` rows: group 0's rows, then group 1's.
constexpr int pf_group_row0(int rows, int g) { return g == 0 ? 0 : 16 * pf_group_frags(rows, 0); }

static_assert(pf_group_row0(moe_prefill_rows(true), 1) + 16 * pf_group_frags(moe_prefill_rows(true), 1) ==
                  moe_prefill_rows(true),
              "the groups' parts fill a slot and end with it");
