// Grouped GEMMs of the larger batches (more than 8 pairs per expert) on LDS tiles: FP8 experts
// accumulated on the FP8 MFMA (H <= 2048) and bf16 experts.  Tile, arguments and epilogues: prefill_dev.h.
//
// 192 rows per tile: a tile's weights are read once for all of an expert's rows up to 192 (at 128 rows
// a tile, an expert of 129 .. 192 rows takes its weights through LDS twice).
//
// Bound by the stream of weights up to about 128 rows per expert (Qwen3-30B-A3B, 300 tokens: gate_up
// 403 MB in 75.6 us, 5.3 TB/s), beyond by the issue of the operand DMA, which stretches a compute phase of
// 785 cycles (768 of MFMAs) to 1265.  Against one 8-wave group with two register sets of fragments on
// 128-row tiles, gate_up + down: 300 tokens 80.4 + 46.9 -> 75.6 + 44.4 us, uniform 2048 tokens 132 + 80 ->
// 101 + 63 us (its 129 .. 160-row experts were two tiles each), Zipf-routed 4096 tokens 183 + 128 -> 170 +
// 108 us; bf16 experts, 1700 tokens 203 + 117 -> 196 + 114 us, 300 tokens level (184 + 82: rows of 4 KB meet
// on the same memory channels).
//
// The two wave groups (waves 0-3 and 4-7: one wave of each on every SIMD) run the same program half a
// K block apart: while one issues the MFMAs of a K block (a compute phase), the other reads its next
// fragments from LDS (a load phase), with a barrier between phases, so the LDS reads of one wave lie
// under the MFMAs of the other wave of its SIMD without a second register set for fragments; that
// leaves the registers for up to 6 x 4 MFMA tiles of accumulators per wave.
//   phase 2s:     group 0 computes K block s      group 1 loads the fragments of s
//   phase 2s + 1: group 0 loads those of s + 1    group 1 computes s
//
// Operands reach LDS by global->LDS DMA, the weights through a ring of three 32 KB K blocks, the
// activations through two 12 KB slots per group (a group reads only its own rows, so a slot is free
// half a K block earlier than a shared one would be).
//   group 0 in phase 2s - 1 (load):     half of the weights of block s + 2 (ring slot of s - 1, last
//                                       read in phase 2s - 2)
//           in phase 2s (compute):      its rows of block s + 2 (slot of s, read in phase 2s - 1)
//   group 1 in phase 2s + 1 (compute):  its rows of block s + 2 (slot of s, read in phase 2s), then
//                                       the other half of the weights of s + 3 (ring slot of s)
// Weights thus have four phases to land (they come from HBM), activations three.  The waits before
// the barriers leave everything younger in flight.
//
// Persistent grid: one workgroup per CU.  Work items (tile, column block) are handed out so that
// the workgroups on one XCD (hardware places workgroup w on XCD w % 8) take consecutive items:
// they share the expert's weights and the tile's activations in that XCD's L2.  The DMA stream
// runs across items.
#include "prefill_dev.h"

namespace {

constexpr int PBM = moe_prefill_rows(false);  // rows per tile
constexpr int PGM = PBM / 2;           // rows of a wave group
constexpr int PNM = PGM / 16;          // 16-row fragments of a wave
constexpr int P_ASLOT = PGM * PBK;     // 12 KB
constexpr int P_NA = P_ASLOT / 4096;   // A DMA instructions of a wave per K block, at most
constexpr int P_NB = P_BSLOT / 8192;   // B DMA instructions of a wave per K block

// One lane's 16-byte operand h of the bf16 MFMAs within its 32-byte fragment (chunks 2 g and
// 2 g + 1 of the row for lane group g).
__device__ __forceinline__ v8bf frag_half(const v8i& f, int h) {
  return __builtin_bit_cast(v8bf, make_uint4(f[4 * h], f[4 * h + 1], f[4 * h + 2], f[4 * h + 3]));
}

template <bool BF>
struct AccOf {
  typedef v4f type;
};
template <>
struct AccOf<false> {
  typedef F4 type;
};

// BF: bf16 operands.  A K block is 64 elements, 128 bytes per row like the e4m3 one, so layout,
// DMA and fragment reads are the same; each fragment feeds two v_mfma_f32_16x16x32_bf16 that
// accumulate in fp32 in the MFMA (no scales, no FMAs).
template <int MODE, bool BF>
__global__ __launch_bounds__(P_THREADS, 1) void grouped_gemm_prefill_kernel(PrefillArgs p) {
  __shared__ __attribute__((aligned(16))) uint8_t s_b[3][P_BSLOT];
  __shared__ __attribute__((aligned(16))) uint8_t s_a[2][2][P_ASLOT];  // [slot][group]
  __shared__ __attribute__((aligned(16))) float s_sa[2][2][PGM];       // activation scales, as s_a
  __shared__ __attribute__((aligned(16))) int s_perm[3][PBM];          // pairs of the tile's rows, by item mod 3
  __shared__ __attribute__((aligned(16))) float s_swt[3][2][kMaxKB];   // weight scales per K block, as s_perm
  __shared__ float s_amax[2][4][PGM];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave >> 2, wn = wave & 3;
  const int lr = lane & 15, lg = lane >> 4;
  const int c0 = 2 * lg;
  const int K = BF ? 2 * p.K : p.K;  // bytes per operand row
  const int KB = K / PBK;
  const int Nw = MODE == PF_GATE_UP ? 2 * p.N : p.N;
  const int nblk128 = Nw / PBK;
  const int n_items = const_ld(p.n_tiles, 0) * p.n_nblk;
  const int G = gridDim.x;  // a multiple of 8
  const int my_slot = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  if (my_slot >= n_items) return;  // workgroup-uniform
  const int n_my = (n_items - my_slot + G - 1) / G;  // items of this workgroup: my_slot + j G
  const uint32_t lds_b = __builtin_amdgcn_readfirstlane(lds_u32(&s_b[0][0])) + 1024 * wave;
  const uint32_t lds_a = __builtin_amdgcn_readfirstlane(lds_u32(&s_a[0][0][0])) + g * P_ASLOT + 1024 * wn;
  const uint32_t lds_sa = __builtin_amdgcn_readfirstlane(lds_u32(&s_sa[0][0][0])) + (g * PGM + (PGM / 4) * wn) * 4;
  const uint32_t lds_perm = __builtin_amdgcn_readfirstlane(lds_u32(&s_perm[0][0]));
  const uint32_t lds_swt = __builtin_amdgcn_readfirstlane(lds_u32(&s_swt[0][0][0]));

  // DMA lane assignment: one instruction fills 8 rows x 128 B (block jb = rows 8 jb ..).  Lane L
  // writes position L & 7 of row 8 jb + (L >> 3), which holds logical chunk (L & 7) ^ swz_key(row)
  // = (L & 7) ^ ((L >> 3) ^ (jb & 1)).  A wave fills weight blocks wave + 8 i and the blocks
  // wn + 4 i of its group's rows, so jb & 1 = wn & 1 for all of them.
  const int dma_r = lane >> 3;
  const int dma_lc = (lane & 7) ^ ((dma_r ^ (wn & 1)) & 7);
  const int frag_off0 = lr * 128 + ((c0 ^ swz_key(lr)) << 4);  // within a 16-row fragment group
  const int frag_off1 = lr * 128 + (((c0 + 1) ^ swz_key(lr)) << 4);
  uint32_t b_voff[P_NB];
#pragma unroll
  for (int i = 0; i < P_NB; ++i) {
    const int br = 8 * (wave + 8 * i);
    const int wrow = pf_weight_row(br + dma_r);
    // gate_up: tile rows 128.. are the up rows, I - 128 rows further on
    b_voff[i] = (uint32_t)((MODE == PF_GATE_UP && br >= 128 ? p.N - 128 + wrow : wrow) * K + dma_lc * 16);
  }

  // ---- issue side: where the next K block of the activations and of the weights is read and put ----
  uint32_t a_voff[P_NA];  // per-lane A byte offsets of the item whose activations are being issued
  uint32_t sa_voff = 0;   // per-lane activation-scale byte offset (lanes < PGM / 4)
  const uint8_t *pa = p.a, *pb = nullptr;
  const float* psa = p.sa;
  // item (of this workgroup) and its K blocks not yet issued
  int jA = 0, leftA = KB, jB = 0, leftB = KB;

  // tables of item j into slot j % 3: pairs of its rows (rows past its end repeat the last) and the
  // weight scales of its K blocks (gate_up: gate block nb and up block I/128 + nb; down: blocks
  // 2 nb and 2 nb + 1, the two 128-row halves).  At most one instruction per wave.
  auto table = [&](int j, int slot) __attribute__((always_inline)) {
    const PfItem it = pf_item(p, my_slot + j * G);
    if (wave < PBM / 64) {
      dma_b32<0>((uint32_t)(it.row0 + min(64 * wave + lane, it.rows - 1)) * 4u, p.perm,
                 lds_perm + slot * (PBM * 4) + 256 * wave);
    } else if (!BF && wave >= 6) {
      const int half = wave - 6;
      const int blk = MODE == PF_GATE_UP ? (half == 0 ? it.nb : p.N / PBK + it.nb) : 2 * it.nb + half;
      if (lane < KB)
        dma_b32<0>((uint32_t)((it.e * nblk128 + blk) * KB + lane) * 4u, p.sw,
                   lds_swt + (slot * 2 + half) * (kMaxKB * 4));
    }
  };
  // descriptors of item j (its table is in LDS and visible)
  auto desc_a = [&](int j) __attribute__((always_inline)) {
    const PfItem it = pf_item(p, my_slot + j * G);
    const int* perm = s_perm[j % 3];
    auto row_of = [&](int r) __attribute__((always_inline)) {  // operand row of this group's local row r
      const int tr = min(((2 * (r >> 4) + g) << 4) + (r & 15), it.rows - 1);
      return MODE == PF_GATE_UP ? perm[tr] / p.topk : it.row0 + tr;
    };
#pragma unroll
    for (int i = 0; i < P_NA; ++i) a_voff[i] = (uint32_t)(row_of(8 * (wn + 4 * i) + dma_r) * K + dma_lc * 16);
    if constexpr (!BF) sa_voff = (uint32_t)(row_of((PGM / 4) * wn + min(lane, PGM / 4 - 1)) * KB) * 4u;
  };
  auto desc_b = [&](int j) __attribute__((always_inline)) {
    const PfItem it = pf_item(p, my_slot + j * G);
    pb = p.w + ((long)it.e * Nw + (long)it.nb * (MODE == PF_GATE_UP ? 128 : 256)) * K;
  };

  // DMA instruction d of a K block's activations (d == P_NA: their scales) and of its weights.  All
  // of them are issued whatever the tile's rows (those past its end repeat the last row, whose lines
  // are at hand), so that the wait counts are constants.
  auto issue_a = [&](auto dc, uint32_t la, uint32_t lsa) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value;
    if constexpr (d < P_NA) {
      dma_b128<d * 4096>(a_voff[d], pa, la);
    } else if constexpr (!BF) {
      if (lane < PGM / 4) dma_b32<0>(sa_voff, psa, lsa);
    }
  };
  auto issue_b = [&](auto dc, uint32_t lb) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value;
    dma_b128<d * 8192>(b_voff[d], pb, lb);
  };
  auto issue_b_all = [&](uint32_t lb) __attribute__((always_inline)) {
    issue_b(Int<0>{}, lb);
    issue_b(Int<1>{}, lb);
    issue_b(Int<2>{}, lb);
    issue_b(Int<3>{}, lb);
  };
  static_assert(P_NA == 3 && P_NB == 4, "DMA instructions of a wave");
  constexpr int N_A = P_NA + (BF ? 0 : 1);
  // To the block after the one just issued.  Past the last item its blocks are issued over again (into
  // free slots), so that the wait counts stay.
  auto advance_a = [&]() __attribute__((always_inline)) {
    pa += PBK;
    ++psa;
    if (--leftA == 0) {
      leftA = KB;
      pa -= K;
      psa -= KB;
      if (jA + 1 < n_my) desc_a(++jA);
    }
  };
  auto advance_b = [&]() __attribute__((always_inline)) {
    pb += PBK;
    if (--leftB == 0) {
      leftB = KB;
      pb -= K;
      if (jB + 1 < n_my) desc_b(++jB);
    }
  };

  // ---- registers of the compute side ----
  const v4f zero4 = {0.f, 0.f, 0.f, 0.f};

  // MFMA operand order: the weight fragment is the MFMA's A operand and the activation fragment its
  // B operand, so lane l holds weight rows n = 4 (l >> 4) + q, q = 0..3, for token row m = l & 15.
  // First LDS weight row of fragment ni of this wave: gate_up gate rows wn*32 + 16 ni
  // (ni < 2) and the matching up rows 128 + wn*32 + 16 (ni - 2); down wn*64 + 16 ni.
  struct Frags {
    v8i af[PNM], bf[4];
    float sca[PNM], scb[PNM];  // activation scale x weight scale (gate_up: gate, up)
  };
  auto load_frags = [&](auto nmc, Frags& f, int slot_a, int slot_b, int tslot, int kb) __attribute__((always_inline)) {
    constexpr int NM = decltype(nmc)::value;
    const uint8_t* sA = s_a[slot_a][g];
    const uint8_t* sB = s_b[slot_b];
    float sv[NM], w0 = 0.f, w1 = 0.f;
    if constexpr (!BF) {
      if constexpr (MODE == PF_GATE_UP) {
        w0 = s_swt[tslot][0][kb];
        w1 = s_swt[tslot][1][kb];
      } else {
        w0 = s_swt[tslot][wn >> 1][kb];
      }
#pragma unroll
      for (int mi = 0; mi < NM; ++mi) sv[mi] = s_sa[slot_a][g][mi * 16 + lr];
    }
    auto frag = [&](const uint8_t* base) __attribute__((always_inline)) -> v8i {
      const uint4 lo = *(const uint4*)(base + frag_off0), hi = *(const uint4*)(base + frag_off1);
      return (v8i){(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    };
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
      const int brow = MODE == PF_GATE_UP ? (ni < 2 ? wn * 32 + ni * 16 : 128 + wn * 32 + (ni - 2) * 16)
                                          : wn * 64 + ni * 16;
      f.bf[ni] = frag(sB + brow * 128);
    }
#pragma unroll
    for (int mi = 0; mi < NM; ++mi) f.af[mi] = frag(sA + mi * 16 * 128);
    if constexpr (!BF) {
#pragma unroll
      for (int mi = 0; mi < NM; ++mi) {
        f.sca[mi] = sv[mi] * w0;
        if constexpr (MODE == PF_GATE_UP) f.scb[mi] = sv[mi] * w1;
      }
    }
  };

  // The MFMAs of one K block for the first NM activation fragments, fragment by fragment, with its
  // DMA instructions among those of the first and, for FP8, each result folded into its fp32
  // accumulator three MFMAs later.
  auto compute = [&](auto nmc, auto& acc, const Frags& f, uint32_t la, uint32_t lsa, uint32_t lb) __attribute__((always_inline)) {
    constexpr int NM = decltype(nmc)::value;
    v4f t[4];
    auto fold = [&](int mi, int ni) __attribute__((always_inline)) {
      if constexpr (!BF) {
      const float sc = MODE == PF_GATE_UP && ni >= 2 ? f.scb[mi] : f.sca[mi];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[mi][ni][e] = fmaf(t[ni][e], sc, acc[mi][ni][e]);
      asm volatile("" : "+v"(acc[mi][ni][0]), "+v"(acc[mi][ni][1]), "+v"(acc[mi][ni][2]), "+v"(acc[mi][ni][3]));
      }
    };
    // DMA instruction d of this phase (activations, their scales, group 1's weights) goes after
    // MFMA d NT / 8: several at a time hold up the wave's next MFMA
    auto dma_slot = [&](auto itc) __attribute__((always_inline)) {
      constexpr int it = decltype(itc)::value, NT = 4 * NM;
      if constexpr (it == 0 * NT / 8) issue_a(Int<0>{}, la, lsa);
      if constexpr (it == 1 * NT / 8) issue_a(Int<1>{}, la, lsa);
      if constexpr (it == 2 * NT / 8) issue_a(Int<2>{}, la, lsa);
      if constexpr (it == 3 * NT / 8) issue_a(Int<3>{}, la, lsa);
      if constexpr (it >= 4 * NT / 8) {
        if (g == 1) {
          if constexpr (it == 4 * NT / 8) issue_b(Int<0>{}, lb);
          if constexpr (it == 5 * NT / 8) issue_b(Int<1>{}, lb);
          if constexpr (it == 6 * NT / 8) issue_b(Int<2>{}, lb);
          if constexpr (it == 7 * NT / 8) issue_b(Int<3>{}, lb);
        }
      }
    };
    auto tile = [&](auto mic, auto nic) __attribute__((always_inline)) {
      constexpr int mi = decltype(mic)::value, ni = decltype(nic)::value;
      if constexpr (BF) {
        acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag_half(f.bf[ni], 0), frag_half(f.af[mi], 0),
                                                              acc[mi][ni], 0, 0, 0);
      } else {
        t[ni] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(f.bf[ni], f.af[mi], zero4, 0, 0, 0, 0, 0, 0);
        PF_PIN(t[ni]);
      }
      dma_slot(Int<mi * 4 + ni>{});
      if constexpr (!BF) {  // the result of three MFMAs ago
        if constexpr (ni == 3)
          fold(mi, 0);
        else if constexpr (mi > 0)
          fold(mi - 1, ni + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto block = [&](auto mic) __attribute__((always_inline)) {
      constexpr int mi = decltype(mic)::value;
      tile(mic, Int<0>{});
      tile(mic, Int<1>{});
      tile(mic, Int<2>{});
      tile(mic, Int<3>{});
      if constexpr (BF) {
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag_half(f.bf[ni], 1), frag_half(f.af[mi], 1),
                                                                acc[mi][ni], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    block(Int<0>{});
    if constexpr (NM > 1) block(Int<1>{});
    if constexpr (NM > 2) block(Int<2>{});
    if constexpr (NM > 3) block(Int<3>{});
    if constexpr (NM > 4) block(Int<4>{});
    if constexpr (NM > 5) block(Int<5>{});
    fold(NM - 1, 1);
    fold(NM - 1, 2);
    fold(NM - 1, 3);
  };

  // ---- prologue: two tables, the first K blocks ----
  // The weights need no table: block 0 goes out with the tables, and the K loop starts when it has
  // landed with its activations, the next ones in flight (300 tokens of Qwen3-30B-A3B: gate_up 78.2 ->
  // 76.1 us, down 47.1 -> 45.5 us, against waiting for the tables and then for all first blocks).
  auto issue_a_all = [&](int b) __attribute__((always_inline)) {
    const uint32_t la = lds_a + b * (2 * P_ASLOT), lsa = lds_sa + b * (2 * PGM * 4);
    issue_a(Int<0>{}, la, lsa);
    issue_a(Int<1>{}, la, lsa);
    issue_a(Int<2>{}, la, lsa);
    issue_a(Int<3>{}, la, lsa);
    advance_a();
  };
  table(0, 0);
  if (n_my > 1) table(1, 1);
  desc_b(0);
  issue_b_all(lds_b);
  advance_b();
  wait_vm<P_NB>();  // the tables
  lds_wait_barrier();
  desc_a(0);
  issue_a_all(0);
  issue_b_all(lds_b + P_BSLOT);
  advance_b();
  issue_a_all(1);
  if (g == 1) {
    issue_b_all(lds_b + 2 * P_BSLOT);
    advance_b();
    wait_vm<N_A + 2 * P_NB>();  // in flight may be block 1 and these
  } else {
    wait_vm<N_A + P_NB>();  // in flight may be block 1
  }
  lds_wait_barrier();

  int sl = 0, sb = 0;  // slots of the K block in the rings: s & 1, s % 3

  // Item j with its fragment count a constant (one straight-line compute phase and epilogue per
  // count: with the count a run-time value inside them the accumulators were copied and spilled).
  auto item = [&](auto nmc, const PfItem& it, int j) __attribute__((always_inline)) {
    constexpr int NM = decltype(nmc)::value;
    typename AccOf<BF>::type acc[NM][4];
#pragma unroll
    for (int mi = 0; mi < NM; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[mi][ni][q] = 0.f;
#pragma unroll 1
    for (int kb = 0; kb < KB; ++kb) {
      // ---- load phase ----
      Frags f;
      load_frags(nmc, f, sl, sb, j % 3, kb);
      const uint32_t lb = lds_b + (g == 0 && sb == 0 ? 2 : sb - 1 + g) * P_BSLOT;  // slot (s + 2) % 3 or (s + 3) % 3
      const uint32_t la = lds_a + sl * (2 * P_ASLOT), lsa = lds_sa + sl * (2 * PGM * 4);
      if (g == 0) {
        issue_b_all(lb);  // block s + 2
        advance_b();
      } else {
        wait_vm<N_A + P_NB>();  // the weights issued a K block ago (group 0 reads them in its next load phase)
      }
      if (kb == 1 && j + 2 < n_my) table(j + 2, (j + 2) % 3);  // slot (j - 1) % 3: its last reader ended a phase ago
      lds_wait_barrier();
      // ---- compute phase: activations of block s + 2, group 1's weights of block s + 3 ----
      __builtin_amdgcn_s_setprio(1);  // its MFMAs before the other wave's address arithmetic
      compute(nmc, acc, f, la, lsa, lb);
      __builtin_amdgcn_s_setprio(0);
      advance_a();
      if (g == 1) advance_b();
      sl ^= 1;
      sb = sb == 2 ? 0 : sb + 1;
      // the activations issued a K block ago have landed, and group 0's weights with them; in flight
      // may be what was issued since: a block of activations and one (group 1: two) of weights
      if (g == 0)
        wait_vm<N_A + P_NB>();
      else
        wait_vm<N_A + 2 * P_NB>();
      lds_wait_barrier();
    }
    // the epilogue, in the phases before the next item's first loads
    if constexpr (MODE == PF_DOWN) {
      pf_store_pairs<NM>(acc, s_perm[j % 3], p, it, g, wn, lr, lg);
    } else if constexpr (BF) {
      pf_store_h_bf16<NM>(acc, p, it, g, wn, lr, lg);
    } else {
      pf_silu_amax<NM>(acc, s_amax[g][0], PGM, wn, lr, lg);
      lds_wait_barrier();  // both groups run it, one phase apart: they stay half a K block apart
      pf_quant_h<NM>(acc, s_amax[g][0], PGM, p, it, g, wn, lr, lg);
    }
    // the epilogue's divergent branches join here and not where the item cases do: else the pipeline's
    // state, merged there, counts as different from lane to lane and leaves the scalar registers
    asm volatile("");
  };

  if (g == 1) lds_wait_barrier();  // one phase later than group 0
#pragma unroll 1
  for (int j = 0; j < n_my; ++j) {
    const PfItem it = pf_item(p, my_slot + j * G);
    switch (pf_frags(it.rows, g)) {
      case 1: item(Int<1>{}, it, j); break;
      case 2: item(Int<2>{}, it, j); break;
      case 3: item(Int<3>{}, it, j); break;
      case 4: item(Int<4>{}, it, j); break;
      case 5: item(Int<5>{}, it, j); break;
      default: item(Int<6>{}, it, j); break;
    }
  }
  if (g == 0) lds_wait_barrier();  // group 1 runs one phase later
  wait_vm<0>();                    // no DMA may land in LDS after the workgroup has ended
}

template <int MODE, bool BF>
int launch_prefill(PrefillArgs a, int max_tiles, hipStream_t s) {
  MOE_LAUNCH(MODE == PF_GATE_UP ? MOE_PROF_GATE_UP : MOE_PROF_DOWN, s, (grouped_gemm_prefill_kernel<MODE, BF>),
             dim3(pf_grid(a, max_tiles)), dim3(P_THREADS), 0, s, a);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

}  // namespace

int moe_launch_grouped_gemms_prefill_exact(const uint8_t* xq, const float* sx, const uint8_t* w13, const float* s13,
                                           const uint8_t* w2, const float* s2, const int32_t* perm,
                                           const int32_t* tiles, const int32_t* n_tiles, int max_tiles, uint8_t* hq,
                                           float* sh, uint16_t* pairs, int H, int I, int k, hipStream_t s);

// gate_up (with fused SiLU*up and e4m3 re-quantisation of h) then down on tiles of
// moe_prefill_rows(moe_exact_accum(H)) rows, at most max_tiles of them.
int moe_launch_grouped_gemms_prefill(const uint8_t* xq, const float* sx, const uint8_t* w13, const float* s13,
                                     const uint8_t* w2, const float* s2, const int32_t* perm, const int32_t* tiles,
                                     const int32_t* n_tiles, int max_tiles, uint8_t* hq, float* sh, uint16_t* pairs,
                                     int H, int I, int k, hipStream_t s) {
  // the DMA takes 32-bit per-lane byte offsets into the activations; max_tiles counts 128-row tiles
  const long max_rows = 128L * max_tiles;
  if (max_rows * (H > I ? H : I) >= (1L << 32)) return MOE_ERR_INVALID_ARG;
  // the cross-item DMA pipeline needs at least 4 K blocks per GEMM
  if (H / PBK < 4 || I / PBK < 4 || H % PBN != 0) return MOE_ERR_INVALID_ARG;
  if (moe_exact_accum(H))
    return moe_launch_grouped_gemms_prefill_exact(xq, sx, w13, s13, w2, s2, perm, tiles, n_tiles, max_tiles, hq, sh,
                                                  pairs, H, I, k, s);
  PrefillArgs g1{xq, sx, w13, s13, perm, tiles, n_tiles, nullptr, hq, sh, nullptr, H, I, k, I / PBK};
  int rc = launch_prefill<PF_GATE_UP, false>(g1, max_tiles, s);
  if (rc) return rc;
  PrefillArgs g2{hq, sh, w2, s2, perm, tiles, n_tiles, pairs, nullptr, nullptr, nullptr, I, H, k, H / PBN};
  return launch_prefill<PF_DOWN, false>(g2, max_tiles, s);
}

// Whether bf16 experts of this shape can take these tiles (bf16 K blocks are 64 deep).
bool moe_prefill_bf16_ok(int H, int I, long max_rows) {
  return H % PBN == 0 && H / 64 >= 4 && I / 64 >= 4 && I % MOE_GROUP == 0 &&
         max_rows * 2 * (H > I ? H : I) < (1L << 32);
}

// The same pair of GEMMs for bf16 weights: gate_up writes bf16 h [S, I], down bf16(z) pair rows
// (the combine applies the routing weight).
int moe_launch_grouped_gemms_prefill_bf16(const uint16_t* x, const uint16_t* w13, const uint16_t* w2,
                                          const int32_t* perm, const int32_t* tiles, const int32_t* n_tiles,
                                          int max_tiles, uint16_t* h, uint16_t* pairs, int H, int I, int k,
                                          hipStream_t s) {
  if (!moe_prefill_bf16_ok(H, I, 128L * max_tiles)) return MOE_ERR_INVALID_ARG;
  PrefillArgs g1{(const uint8_t*)x, nullptr, (const uint8_t*)w13, nullptr, perm, tiles, n_tiles, nullptr, nullptr,
                 nullptr, h, H, I, k, I / PBK};
  int rc = launch_prefill<PF_GATE_UP, true>(g1, max_tiles, s);
  if (rc) return rc;
  PrefillArgs g2{(const uint8_t*)h, nullptr, (const uint8_t*)w2, nullptr, perm, tiles, n_tiles, pairs, nullptr,
                 nullptr, nullptr, I, H, k, H / PBN};
  return launch_prefill<PF_DOWN, true>(g2, max_tiles, s);
}
