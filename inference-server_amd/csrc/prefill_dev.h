// What the LDS-tiled grouped GEMMs of the larger batches share (gemm_prefill.hip: FP8 MFMA and bf16
// experts; gemm_prefill_exact.hip: FP8 experts accumulated exactly): arguments, work items, epilogues
// and the launch grid.
//
// Tile: a few 16-row groups of one expert's sorted rows x 256 weight rows x 128-byte K blocks.
//   gate_up: the 256 weight rows are 128 gate rows [n0, n0+128) and the matching 128 up rows
//            [I+n0, I+n0+128), so one tile yields 128 complete h columns = one quantisation group.
//            The epilogue computes h = silu(g)*u in the reference's bf16 rounding order and, for
//            FP8, the per-row group amax and the e4m3 intermediate with its scale.
//   down:    256 output columns; bf16(z) at the pair's original row t*k+j (the combine weights it).
// Workgroup: two groups of four waves; group g owns the 16-row groups 2 m + g of the tile, wave wn of
// a group 64 of the 256 weight rows.  Work scales with the rows a tile really holds: fragments, MFMAs
// and epilogue of 16-row groups past its end are left out.
#pragma once

#include "common.h"
#include "lds_dma.h"

namespace {
using namespace moe_lds;

enum { PF_GATE_UP = 0, PF_DOWN = 1 };

constexpr int PBN = 256;               // weight rows per tile
constexpr int PBK = 128;               // bytes of a K block
constexpr int P_BSLOT = PBN * PBK;     // 32 KB
constexpr int kMaxKB = 32;             // FP8: K <= 4096
constexpr int P_THREADS = 512;

struct PrefillArgs {
  const uint8_t* a;        // gate_up: xq [T, K] (token rows); down: hq [S, K] (sorted rows); bf16: x, h
  const float* sa;         // activation scales [rows, K/128]
  const uint8_t* w;        // [E, Nw, K]
  const float* sw;         // [E, Nw/128, K/128]
  const int32_t* perm;     // sorted row -> flat pair
  const int32_t* tiles;    // {expert, first sorted row, rows, 0}
  const int32_t* n_tiles;
  uint16_t* pairs;         // down: output [S, N] by flat pair
  uint8_t* hq;             // gate_up: e4m3 intermediate [S, N]
  float* sh;               // gate_up: its scales [S, N/128]
  uint16_t* h;             // bf16 weights, gate_up: the bf16 intermediate [S, N]
  int K;                   // reduction length (elements)
  int N;                   // gate_up: I; down: H
  int topk;
  int n_nblk;              // column blocks per tile: gate_up I/128, down H/256
};

struct PfItem {
  int e, row0, rows, nb;
};

__device__ __forceinline__ PfItem pf_item(const PrefillArgs& p, int item) {
  const int tile = item / p.n_nblk;
  const int4 ti = const_ld4(p.tiles, tile);
  return {ti.x, ti.y, ti.z, item - tile * p.n_nblk};
}

// 16-row fragments of wave group g in a tile of `rows` rows, at least one (a tile of up to 16 rows
// gives group 1 a fragment of repeated rows, whose results are never stored)
__device__ __forceinline__ int pf_frags(int rows, int g) { return rows > 16 ? (((rows + 15) >> 4) - g + 1) >> 1 : 1; }

template <int N>
struct Int {
  static constexpr int value = N;
};

struct F4 {
  float v[4];
  __device__ __forceinline__ float& operator[](int i) { return v[i]; }
};
// An empty volatile asm that takes and returns v_: the value is computed before this point and the
// volatile asm statements keep their order, which holds each MFMA and each scale FMA in its slot.
#define PF_PIN(v_) asm volatile("" : "+v"(v_))

// Weight row (of the tile's 256) that lies in LDS row r: within each 32, rows 8 a + 4 b + c (b < 2, c < 4)
// lie at 16 b + 4 a + c.  A result lane holds rows 4 a + c of a 16-row fragment, c = 0..3, and with them
// of two neighbouring fragments eight adjacent columns: half the stores, of 64 adjacent bytes a row
// instead of 32 (Qwen3-30B-A3B, down at 4096 Zipf-routed tokens 131 -> 114 us, bf16 4096 tokens 189 -> 170,
// bf16 1700 tokens 122 -> 117 us; gate_up's h stores are a tenth of its time and stayed level).
__device__ __forceinline__ int pf_weight_row(int r) {
  return (r & ~31) | ((r & 12) << 1) | ((r >> 2) & 4) | (r & 3);
}

// The epilogues.  Lane (lr, lg) of wave wn holds, for tile rows r = (2 mi + g) 16 + lr, the columns
// 32 (ni / 2) + 8 lg + 4 (ni % 2) + q of this wave's 64 (down) in acc[mi][ni][q]; gate_up: of its 32 h
// columns, the gate in fragments 0, 1 and up in 2, 3.

// gate_up, bf16 experts: h in bf16.
template <int NM, class Acc>
__device__ __forceinline__ void pf_store_h_bf16(Acc& acc, const PrefillArgs& p, const PfItem& it, int g, int wn, int lr,
                                                int lg) {
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) {
    const int r = (2 * mi + g) * 16 + lr;
    if (r < it.rows) {
      uint16_t* dst = p.h + (long)(it.row0 + r) * p.N + it.nb * 128 + wn * 32 + 8 * lg;
      uint32_t v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ni = q >> 1, c = 2 * (q & 1);
        v[q] = (uint32_t)f32_to_bf16(silu_mul_bf16(acc[mi][ni][c], acc[mi][ni + 2][c])) |
               ((uint32_t)f32_to_bf16(silu_mul_bf16(acc[mi][ni][c + 1], acc[mi][ni + 2][c + 1])) << 16);
      }
      *(uint4*)dst = make_uint4(v[0], v[1], v[2], v[3]);
    }
  }
}

// gate_up, FP8 experts, before the group's barrier: h into acc[mi][0..1] and its row maxima over the
// wave's 32 columns into amax (the group's [4 waves][rows], row stride `stride`).
template <int NM, class Acc>
__device__ __forceinline__ void pf_silu_amax(Acc& acc, float* amax, int stride, int wn, int lr, int lg) {
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) {
    float m = 0.f;
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float h = silu_mul_bf16(acc[mi][ni][q], acc[mi][ni + 2][q]);
        acc[mi][ni][q] = h;
        m = fmaxf(m, fabsf(h));
      }
    // the four lanes lr, lr+16, lr+32, lr+48 share the row
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    if (lg == 0) amax[wn * stride + mi * 16 + lr] = m;
  }
}

// After it: the e4m3 codes of h and their scales.
template <int NM, class Acc>
__device__ __forceinline__ void pf_quant_h(Acc& acc, const float* amax, int stride, const PrefillArgs& p,
                                           const PfItem& it, int g, int wn, int lr, int lg) {
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) {
    const int r = (2 * mi + g) * 16 + lr, rl = mi * 16 + lr;
    const float am = fmaxf(fmaxf(amax[rl], amax[stride + rl]), fmaxf(amax[2 * stride + rl], amax[3 * stride + rl]));
    const float sc = am > 0.f ? am / MOE_FP8_MAX : 1.0f;
    if (r < it.rows) {
      const long srow = it.row0 + r;
      // h / s rounded as the oracle's division (div_rn): h and amax are bf16, so 448 h / amax
      // often lands exactly on an e4m3 rounding midpoint, where h * (1 / s) (two roundings)
      // falls on either side (0.05% of the codes differed that way)
      uint32_t v[2];
#pragma unroll
      for (int ni = 0; ni < 2; ++ni)
        v[ni] = pack4_e4m3(clamp_fp8(div_rn(acc[mi][ni][0], sc)), clamp_fp8(div_rn(acc[mi][ni][1], sc)),
                           clamp_fp8(div_rn(acc[mi][ni][2], sc)), clamp_fp8(div_rn(acc[mi][ni][3], sc)));
      *(uint2*)(p.hq + srow * p.N + it.nb * 128 + wn * 32 + 8 * lg) = make_uint2(v[0], v[1]);
      if (wn == 0 && lg == 0) p.sh[srow * (p.N / MOE_GROUP) + it.nb] = sc;
    }
  }
}

// down: bf16(z) at the pairs' rows (pairs of the tile's rows in LDS).
template <int NM, class Acc>
__device__ __forceinline__ void pf_store_pairs(Acc& acc, const int* s_pairs, const PrefillArgs& p, const PfItem& it,
                                               int g, int wn, int lr, int lg) {
#pragma unroll
  for (int mi = 0; mi < NM; ++mi) {
    const int r = (2 * mi + g) * 16 + lr;
    if (r < it.rows) {
      const long pr = s_pairs[r];
      uint16_t* dst = p.pairs + pr * p.N + it.nb * 256 + wn * 64 + 8 * lg;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint32_t v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int ni = 2 * s + (q >> 1), c = 2 * (q & 1);
          v[q] = (uint32_t)f32_to_bf16(acc[mi][ni][c]) | ((uint32_t)f32_to_bf16(acc[mi][ni][c + 1]) << 16);
        }
        *(uint4*)(dst + 32 * s) = make_uint4(v[0], v[1], v[2], v[3]);
      }
    }
  }
}

// One persistent workgroup per CU, in whole rounds of the eight XCDs, at most one per work item.
unsigned pf_grid(const PrefillArgs& a, int max_tiles) {
  const long max_items = (long)max_tiles * a.n_nblk;
  long grid = moe_cu_count();
  if (grid > max_items) grid = max_items;
  grid = (grid + 7) / 8 * 8;
  return (unsigned)(grid < 8 ? 8 : grid);
}

}  // namespace
