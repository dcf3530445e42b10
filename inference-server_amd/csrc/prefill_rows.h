// Rows of the LDS-tiled grouped GEMMs' tiles: their height, and the wave group that holds each 16-row
// fragment.  Plain constexpr C++, for host and device.
#pragma once

// Rows per tile at most.
constexpr int moe_prefill_rows(bool exact) { return exact ? 144 : 192; }

// Lower tiles where they take no more rounds: a launch hands its work items (tile, column block) out one per
// CU and round, so with as many rounds it ends sooner the lower they are, and with fewer the taller tiles'
// single pass over an expert's weights counts.  n_low tiles of kPrefillLowRows rows against n_high of
// moe_prefill_rows, in both GEMMs (nb1 and nb2 column blocks).  Qwen3-30B-A3B experts layer, MI355X:
// 128- / 192-row tiles, FP8 and bf16: 16 experts with 145 rows (one round of either) 61.2 / 74.5 us and 76.2 /
// 88.2, with 430 rows (two of either) 117.6 / 129.3 and 137.4 / 152.8; 24 experts with 145 rows (two against
// one) 93.8 / 84.5 and 121.9 / 101.3.  Where the rounds of only one GEMM grow either can win: 8 experts with 1200
// rows 142.8 / 150.3 us, 20 experts with about 240 rows each 108.5 / 94.1.  Exact accumulation: 144 rows
// throughout (16 experts of Qwen3-235B-A22B leave no room, 8 are level).
constexpr int kPrefillLowRows = 128;
constexpr bool pf_cut_low(int n_low, int n_high, int nb1, int nb2, int cus) {
  return (n_low * nb1 + cus - 1) / cus <= (n_high * nb1 + cus - 1) / cus &&
         (n_low * nb2 + cus - 1) / cus <= (n_high * nb2 + cus - 1) / cus;
}

// Rows per tile of an expert with n rows, at most `rows` (a multiple of 16) each: the same number of tiles,
// equally high in whole fragments, since a launch takes as long as the tallest of its last round.
// The same layer against full tiles and a remainder: 24 experts with 200 rows 127.6 -> 107.2 us, 32 experts
// 138.3 -> 119.3, 4096 Zipf-routed tokens on 128 experts 325.8 -> 320.4; 16 experts of Qwen3-235B-A22B (exact)
// with 145 rows 243 -> 187 us, with 300 rows 355 -> 316.  Level where there are many rounds (64 experts
// with 500 rows 414 / 413 us).
constexpr int pf_even_rows(int n, int rows) {
  if (n <= rows) return rows;
  const int tiles = (n + rows - 1) / rows;
  return ((n + tiles - 1) / tiles + 15) / 16 * 16;
}

// 16-row fragments of a full tile of `rows` rows that wave group g (0 or 1) holds: those numbered 2 m + g.
constexpr int pf_group_frags(int rows, int g) { return (rows / 16 - g + 1) / 2; }

// First row of group g's part of an activation slot of `rows` rows: group 0's rows, then group 1's.
constexpr int pf_group_row0(int rows, int g) { return g == 0 ? 0 : 16 * pf_group_frags(rows, 0); }

static_assert(pf_group_row0(moe_prefill_rows(true), 1) + 16 * pf_group_frags(moe_prefill_rows(true), 1) ==
                  moe_prefill_rows(true),
              "the groups' parts fill a slot and end with it");
