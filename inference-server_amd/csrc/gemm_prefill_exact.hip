// Grouped FP8 GEMMs of the larger batches accumulated exactly (H > 2048, moe_exact_accum) on LDS
// tiles.  Tile, arguments and epilogues: prefill_dev.h.
//
// The codes of both operands are widened to bf16 in registers (e4m3x8_to_bf16) and each 128-deep K
// block is four 32-deep quarters of v_mfma_f32_16x16x32_bf16, chained in the MFMA and folded into the
// fp32 accumulators once, by the scales.  All chains of a wave are live at once, so a quarter of an
// activation fragment is widened once for the four weight fragments and a quarter of a weight
// fragment once for all rows: 16 (NM + 4) conversions per wave and K block beside 16 NM MFMAs of NM
// 16-row fragments.  (With both operands widened a whole K block at a time, one chain after the
// other, a weight fragment was widened again for every pair of row fragments and the conversions took
// longer than the MFMAs.)  Each quarter is read from LDS right after the one before it was widened, into
// its registers.  144 rows per tile: nine 16-row groups, five of wave group 0, whose chains and
// accumulators (160 registers) are what fits; what the K loop can work out anew (fresh_tid, LDS
// addresses) is not kept in registers.
//
// Qwen3-235B-A22B: gate_up 687 -> 522 us and down 362 -> 272 us at 2048 tokens, 468 -> 332 us (1.6 GB of
// weights, 4.8 TB/s) and 237 -> 157 us at 300; bound by the matrix cores (the bf16 MFMAs of 2048 tokens take
// 165 us in gate_up at their full rate) and the waits of each quarter's LDS reads, below about 64 rows
// per expert by the stream of weights.
//
// Operands reach LDS by global->LDS DMA through rings of three K blocks.  One barrier per K block s,
// before its last quarter: by then every wave holds what it still needs of block s in registers, so
// its slots take block s + 3, and block s + 1, issued two K blocks ago, has landed.  (The activation
// scales are read after that barrier and have a fourth slot.)
//
// Persistent grid: one workgroup per CU.  Work items (tile, column block) are handed out so that
// the workgroups on one XCD (hardware places workgroup w on XCD w % 8) take consecutive items:
// they share the expert's weights and the tile's activations in that XCD's L2.  The DMA stream
// runs across items.
#include "prefill_dev.h"

namespace {

constexpr int PBM = moe_prefill_rows(true);  // rows per tile: nine 16-row groups, five of wave group 0
constexpr int PGM = pf_group_row0(PBM, 1);  // rows of wave group 0 (group 1: 64)
constexpr int P_ASLOT = PBM * PBK;     // 18 KB: group 0's rows, then group 1's
constexpr int P_FRAGS1 = pf_group_frags(PBM, 1);  // fragments of a wave of group 1; group 0 has one more
static_assert(PGM == 80 && P_FRAGS1 == 4, "9 row groups");

template <int MODE>
__global__ __launch_bounds__(P_THREADS, 1) void grouped_gemm_prefill_exact_kernel(PrefillArgs p) {
  __shared__ __attribute__((aligned(16))) uint8_t s_b[3][P_BSLOT];
  __shared__ __attribute__((aligned(16))) uint8_t s_a[3][P_ASLOT];
  __shared__ __attribute__((aligned(16))) float s_sa[4][PBM];          // activation scales of K block s in slot s & 3
  __shared__ __attribute__((aligned(16))) int s_perm[3][PBM];          // pairs of the tile's rows, by item mod 3
  __shared__ __attribute__((aligned(16))) float s_swt[3][2][kMaxKB];   // weight scales per K block, as s_perm
  __shared__ float s_amax[2][4][PGM];
  __shared__ uint32_t s_voff2[128], s_savoff[PBM];  // a_voff[2] of the waves that have it, sa_voff

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave >> 2, wn = wave & 3;
  const int K = p.K;
  const int KB = K / PBK;
  const int Nw = MODE == PF_GATE_UP ? 2 * p.N : p.N;
  const int nblk128 = Nw / PBK;
  const int n_items = const_ld(p.n_tiles, 0) * p.n_nblk;
  const int G = gridDim.x;  // a multiple of 8
  const int my_slot = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  if (my_slot >= n_items) return;  // workgroup-uniform
  const int n_my = (n_items - my_slot + G - 1) / G;  // items of this workgroup: my_slot + j G
  const uint32_t lds_b = __builtin_amdgcn_readfirstlane(lds_u32(&s_b[0][0])) + 1024 * wave;
  // wave group g's part of a slot: rows [0, 80) or [80, 144), a quarter of the scales per wave
  const int arow0 = g * PGM, sa_lanes = g == 0 ? PGM / 4 : (PBM - PGM) / 4;
  const uint32_t lds_a = __builtin_amdgcn_readfirstlane(lds_u32(&s_a[0][0])) + arow0 * PBK + 1024 * wn;
  const uint32_t lds_sa = __builtin_amdgcn_readfirstlane(lds_u32(&s_sa[0][0])) + (arow0 + sa_lanes * wn) * 4;
  const bool third_a = g == 0 && wn < 2;  // this wave has a third block of 8 activation rows
  const uint32_t lds_perm = __builtin_amdgcn_readfirstlane(lds_u32(&s_perm[0][0]));
  const uint32_t lds_swt = __builtin_amdgcn_readfirstlane(lds_u32(&s_swt[0][0][0]));

  // DMA lane assignment: one instruction fills 8 rows x 128 B (block jb = rows 8 jb ..).  Lane L
  // writes position L & 7 of row 8 jb + (L >> 3), which holds logical chunk (L & 7) ^ swz_key(row)
  // = (L & 7) ^ ((L >> 3) ^ (jb & 1)).  A wave fills weight blocks wave + 8 i and the blocks
  // wn + 4 i of its group's rows, so jb & 1 = wn & 1 for all of them.
  // The thread's number, and all that is worked out from it, anew: no registers to spare in the K loop,
  // and the reload of a spilled one would wait for every DMA in flight.
  auto fresh_tid = []() __attribute__((always_inline)) -> int {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  // Quarter jj of a lane's 32 codes of a row, chunks 2 lg and 2 lg + 1 (swizzled), lies at
  // (frag_off ^ 16 (jj / 2)) + 8 (jj % 2) within a 16-row fragment group.
  const int frag_off = (lane & 15) * 128 + ((2 * (lane >> 4) ^ swz_key(lane & 15)) << 4);
  // A wave fills weight blocks wave + 8 i: 64 rows apart, the third and fourth of gate_up among the up
  // rows, I rows after the gate rows.
  const long b_64 = 64L * K, b_128 = MODE == PF_GATE_UP ? (long)p.N * K : 128L * K;

  // ---- issue side: where the next K block of the activations and of the weights is read and put ----
  // Per-lane byte offsets of the item whose activations are being issued; the third (third_a) and the
  // scales' (lanes < sa_lanes) wait in LDS, each written and read by its own wave: no registers to
  // spare, and the reload of a spilled one would wait for every DMA in flight.
  uint32_t a_voff[2];
  const uint8_t *pa = p.a, *pb = nullptr;
  const float* psa = p.sa;
  // item (of this workgroup) and its K blocks not yet issued
  int jA = 0, leftA = KB, jB = 0, leftB = KB;
  // tables of item j into slot j % 3: pairs of its rows (rows past its end repeat the last) and the
  // weight scales of its K blocks (gate_up: gate block nb and up block I/128 + nb; down: blocks
  // 2 nb and 2 nb + 1, the two 128-row halves).  At most one instruction per wave.
  auto table = [&](int j, int slot) __attribute__((always_inline)) {
    const PfItem it = pf_item(p, my_slot + j * G);
    if (wave < 3) {
      const int r = fresh_tid();
      if (r < PBM)
        dma_b32<0>((uint32_t)(it.row0 + min(r, it.rows - 1)) * 4u, p.perm, lds_perm + slot * (PBM * 4) + 256 * wave);
    } else if (wave >= 6) {
      const int half = wave - 6;
      const int blk = MODE == PF_GATE_UP ? (half == 0 ? it.nb : p.N / PBK + it.nb) : 2 * it.nb + half;
      const int kb = fresh_tid() & 63;
      if (kb < KB)
        dma_b32<0>((uint32_t)((it.e * nblk128 + blk) * KB + kb) * 4u, p.sw,
                   lds_swt + (slot * 2 + half) * (kMaxKB * 4));
    }
  };
  // descriptors of item j (its table is in LDS and visible)
  auto desc_a = [&](int j) __attribute__((always_inline)) {
    const PfItem it = pf_item(p, my_slot + j * G);
    const int* perm = s_perm[j % 3];
    const int t = fresh_tid(), ln = t & 63, dma_r = ln >> 3;
    const int dma_lc = (ln & 7) ^ ((dma_r ^ (wn & 1)) & 7);
    int topk = p.topk;
    asm volatile("" : "+s"(topk));  // what a division by it needs is worked out here too
    auto row_of = [&](int r) __attribute__((always_inline)) {  // operand row of this group's local row r
      const int tr = min(((2 * (r >> 4) + g) << 4) + (r & 15), it.rows - 1);
      return MODE == PF_GATE_UP ? perm[tr] / topk : it.row0 + tr;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) a_voff[i] = (uint32_t)(row_of(8 * (wn + 4 * i) + dma_r) * K + dma_lc * 16);
    if (third_a) s_voff2[t] = (uint32_t)(row_of(8 * (wn + 8) + dma_r) * K + dma_lc * 16);
    if (ln < sa_lanes) s_savoff[arow0 + sa_lanes * wn + ln] = (uint32_t)(row_of(sa_lanes * wn + ln) * KB) * 4u;
  };
  auto desc_b = [&](int j) __attribute__((always_inline)) {
    const PfItem it = pf_item(p, my_slot + j * G);
    pb = p.w + ((long)it.e * Nw + (long)it.nb * (MODE == PF_GATE_UP ? 128 : 256) + pf_weight_row(8 * wave)) * K;
  };

  // DMA instruction d of a K block's activations (d == 3: their scales) and of its weights.  All of
  // them are issued whatever the tile's rows (those past its end repeat the last row, whose lines
  // are at hand), so that the wait counts are constants of the wave.
  auto issue_a = [&](auto dc, uint32_t la, uint32_t lsa) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value;
    if constexpr (d == 2) {
      if (third_a) dma_b128<2 * 4096>(s_voff2[fresh_tid()], pa, la);
    } else if constexpr (d < 2) {
      dma_b128<d * 4096>(a_voff[d], pa, la);
    } else {
      const int ln = fresh_tid() & 63;
      if (ln < sa_lanes) dma_b32<0>(s_savoff[arow0 + sa_lanes * wn + ln], psa, lsa);
    }
  };
  // A lane's byte offset from its wave's weights: pf_weight_row(8 wave + dma_r) splits into the two sums.
  auto b_voff = [&]() __attribute__((always_inline)) -> uint32_t {
    const uint32_t l = fresh_tid(), r = (l >> 3) & 7;
    return __umul24(pf_weight_row(r), K) + ((((l ^ r) & 7) ^ (wn & 1)) << 4);
  };
  auto issue_b = [&](auto dc, uint32_t v, uint32_t lb) __attribute__((always_inline)) {
    constexpr int d = decltype(dc)::value;
    dma_b128<d * 8192>(v, pb + (d & 1 ? b_64 : 0) + (d & 2 ? b_128 : 0), lb);
  };
  auto issue_b_all = [&](uint32_t lb) __attribute__((always_inline)) {
    const uint32_t v = b_voff();
    issue_b(Int<0>{}, v, lb);
    issue_b(Int<1>{}, v, lb);
    issue_b(Int<2>{}, v, lb);
    issue_b(Int<3>{}, v, lb);
  };
  constexpr int N_B = 4, N_A = 3;  // instructions of a K block; third_a waves: N_A + 1
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

  // ---- prologue: two tables, the first K blocks ----
  // The weights need no table: block 0 goes out with the tables, and the K loop starts when it has
  // landed with its activations.  K >= 4 blocks (launcher): all three of the first item.
  auto issue_a_all = [&](int b) __attribute__((always_inline)) {
    const uint32_t la = lds_a + b * P_ASLOT, lsa = lds_sa + b * (PBM * 4);
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
  wait_vm<N_B>();  // the tables
  lds_wait_barrier();
  desc_a(0);
  issue_a_all(0);
#pragma unroll
  for (int b = 1; b < 3; ++b) {
    issue_b_all(lds_b + b * P_BSLOT);
    advance_b();
    issue_a_all(b);
  }
  if (third_a)  // in flight may be blocks 1 and 2
    wait_vm<2 * (N_A + 1 + N_B)>();
  else
    wait_vm<2 * (N_A + N_B)>();
  lds_wait_barrier();

  int slot = 0, sslot = 0;  // ring slots of K block s: s % 3, and s & 3 (activation scales)

  uint2 ca[5] = {}, cb[4];  // codes of one quarter of the fragments
  auto read_a = [&](int mi, int sl, int off) __attribute__((always_inline)) {
    if (mi < P_FRAGS1 || g == 0)  // group 1's part of the slot ends after four
      ca[mi] = *(const uint2*)(s_a[sl] + arow0 * PBK + mi * 16 * 128 + off);
  };
  auto read_b = [&](int ni, int sl, int off) __attribute__((always_inline)) {
    const int brow = MODE == PF_GATE_UP ? (ni < 2 ? wn * 32 + ni * 16 : 128 + wn * 32 + (ni - 2) * 16)
                                        : wn * 64 + ni * 16;
    cb[ni] = *(const uint2*)(s_b[sl] + brow * 128 + off);
  };
  auto block = [&](auto nmc, auto& acc, int j, int kb) __attribute__((always_inline)) {
    constexpr int NM = decltype(nmc)::value, NT = 4 * NM;
    v4f tx[NM][4];
    float w0, w1, sv[2];
    const int next = slot == 2 ? 0 : slot + 1;
    const uint32_t la = lds_a + slot * P_ASLOT, lsa = lds_sa + ((sslot + 3) & 3) * (PBM * 4), lb = lds_b + slot * P_BSLOT;
    auto widen = [&](uint32_t lo, uint32_t hi) __attribute__((always_inline)) -> v8bf {
      asm volatile("" : "+v"(lo), "+v"(hi));  // not before this point
      return e4m3x8_to_bf16(lo, hi);
    };
    auto fold = [&](int it) __attribute__((always_inline)) {
      const int mi = it >> 2, ni = it & 3;
      const float sc = sv[mi & 1] * (MODE == PF_GATE_UP && ni >= 2 ? w1 : w0);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[mi][ni][e] = fmaf(tx[mi][ni][e], sc, acc[mi][ni][e]);
      asm volatile("" : "+v"(acc[mi][ni][0]), "+v"(acc[mi][ni][1]), "+v"(acc[mi][ni][2]), "+v"(acc[mi][ni][3]));
    };
    auto quarter = [&](auto jjc) __attribute__((always_inline)) {
      constexpr int jj = decltype(jjc)::value;
      const int src = jj == 3 ? next : slot;  // of the quarter read here, the one after jj
      int off = frag_off;
      asm volatile("" : "+v"(off));  // addresses of this quarter only
      off = ((jj + 1) & 2 ? off ^ 16 : off) + 8 * ((jj + 1) & 1);
      v8bf bw[4];
#pragma unroll
      for (int ni = 0; ni < 4; ++ni) {
        bw[ni] = widen(cb[ni].x, cb[ni].y);
        read_b(ni, src, off);
      }
      auto frag = [&](auto mic) __attribute__((always_inline)) {
        constexpr int mi = decltype(mic)::value;
        if constexpr (mi < NM) {
          const v8bf aw = widen(ca[mi].x, ca[mi].y);
          read_a(mi, src, off);
          if (jj == 3) sv[mi & 1] = s_sa[sslot][arow0 + mi * 16 + (fresh_tid() & 15)];  // used three MFMAs on
          auto tile = [&](auto nic) __attribute__((always_inline)) {
            constexpr int ni = decltype(nic)::value, it = 4 * mi + ni;
            tx[mi][ni] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[ni], aw, jj == 0 ? zero4 : tx[mi][ni], 0, 0, 0);
            PF_PIN(tx[mi][ni]);
            if constexpr (jj == 3) {
              if constexpr (it == 0 * NT / 8) issue_a(Int<0>{}, la, lsa);
              if constexpr (it == 1 * NT / 8) issue_a(Int<1>{}, la, lsa);
              if constexpr (it == 2 * NT / 8) issue_a(Int<2>{}, la, lsa);
              if constexpr (it == 3 * NT / 8) issue_a(Int<3>{}, la, lsa);
              if constexpr (it == 4 * NT / 8) issue_b(Int<0>{}, b_voff(), lb);
              if constexpr (it == 5 * NT / 8) issue_b(Int<1>{}, b_voff(), lb);
              if constexpr (it == 6 * NT / 8) issue_b(Int<2>{}, b_voff(), lb);
              if constexpr (it == 7 * NT / 8) issue_b(Int<3>{}, b_voff(), lb);
              if constexpr (it >= 3) fold(it - 3);
            }
            __builtin_amdgcn_sched_barrier(0);
          };
          tile(Int<0>{});
          tile(Int<1>{});
          tile(Int<2>{});
          tile(Int<3>{});
        } else if constexpr (jj == 3) {
          read_a(mi, src, off);  // the next item may have more fragments
        }
      };
      frag(Int<0>{});
      frag(Int<1>{});
      frag(Int<2>{});
      frag(Int<3>{});
      frag(Int<4>{});
      if constexpr (jj == 3) {
        fold(NT - 3);
        fold(NT - 2);
        fold(NT - 1);
      }
    };
    quarter(Int<0>{});
    quarter(Int<1>{});
    w0 = MODE == PF_GATE_UP ? s_swt[j % 3][0][kb] : s_swt[j % 3][wn >> 1][kb];
    w1 = MODE == PF_GATE_UP ? s_swt[j % 3][1][kb] : 0.f;
    quarter(Int<2>{});
    if (third_a)
      wait_vm<N_A + 1 + N_B>();
    else
      wait_vm<N_A + N_B>();
    lds_wait_barrier();
    quarter(Int<3>{});
    if (kb == 1 && j + 2 < n_my) table(j + 2, (j + 2) % 3);  // slot (j - 1) % 3: its last readers are a barrier ago
    advance_a();
    advance_b();
    slot = next;
    sslot = (sslot + 1) & 3;
  };

  // Item j with its fragment count a constant (one straight-line K block and epilogue per count: with
  // the count a run-time value inside them the accumulators were copied and spilled).
  auto item = [&](auto nmc, const PfItem& it, int j) __attribute__((always_inline)) {
    constexpr int NM = decltype(nmc)::value;
    F4 acc[NM][4];
#pragma unroll
    for (int mi = 0; mi < NM; ++mi)
#pragma unroll
      for (int ni = 0; ni < 4; ++ni)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[mi][ni][q] = 0.f;
    // whatever the previous item's epilogue had spilled of the pipeline's registers is back before the K
    // loop, not waited for in each of its steps (behind every DMA in flight)
    asm volatile("" : "+v"(a_voff[0]), "+v"(a_voff[1]));
#pragma unroll
    for (int i = 0; i < 5; ++i) asm volatile("" : "+v"(ca[i].x), "+v"(ca[i].y));
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(cb[i].x), "+v"(cb[i].y));
#pragma unroll 1
    for (int kb = 0; kb < KB; ++kb) block(nmc, acc, j, kb);
    const int ln = fresh_tid() & 63, lr = ln & 15, lg = ln >> 4;
    if constexpr (MODE == PF_DOWN) {
      pf_store_pairs<NM>(acc, s_perm[j % 3], p, it, g, wn, lr, lg);
    } else {
      pf_silu_amax<NM>(acc, s_amax[g][0], PGM, wn, lr, lg);
      lds_wait_barrier();
      pf_quant_h<NM>(acc, s_amax[g][0], PGM, p, it, g, wn, lr, lg);
    }
    // the epilogue's divergent branches join here and not where the item cases do: else the pipeline's
    // state, merged there, counts as different from lane to lane and leaves the scalar registers
    asm volatile("");
  };

#pragma unroll
  for (int ni = 0; ni < 4; ++ni) read_b(ni, 0, frag_off);
#pragma unroll
  for (int mi = 0; mi < 5; ++mi) read_a(mi, 0, frag_off);
#pragma unroll 1
  for (int j = 0; j < n_my; ++j) {
    const PfItem it = pf_item(p, my_slot + j * G);
    switch (pf_frags(it.rows, g)) {
      case 1: item(Int<1>{}, it, j); break;
      case 2: item(Int<2>{}, it, j); break;
      case 3: item(Int<3>{}, it, j); break;
      case 4: item(Int<4>{}, it, j); break;
      default: item(Int<5>{}, it, j); break;
    }
  }
  wait_vm<0>();  // no DMA may land in LDS after the workgroup has ended
}

template <int MODE>
int launch_prefill_exact(PrefillArgs a, int max_tiles, hipStream_t s) {
  MOE_LAUNCH(MODE == PF_GATE_UP ? MOE_PROF_GATE_UP : MOE_PROF_DOWN, s, grouped_gemm_prefill_exact_kernel<MODE>,
             dim3(pf_grid(a, max_tiles)), dim3(P_THREADS), 0, s, a);
  MOE_CHECK_LAUNCH();
  return MOE_OK;
}

}  // namespace

// gate_up (with fused SiLU*up and e4m3 re-quantisation of h) then down on moe_prefill_rows(true)-row
// tiles; the caller (moe_launch_grouped_gemms_prefill) has checked the shape.
int moe_launch_grouped_gemms_prefill_exact(const uint8_t* xq, const float* sx, const uint8_t* w13, const float* s13,
                                           const uint8_t* w2, const float* s2, const int32_t* perm,
                                           const int32_t* tiles, const int32_t* n_tiles, int max_tiles, uint8_t* hq,
                                           float* sh, uint16_t* pairs, int H, int I, int k, hipStream_t s) {
  PrefillArgs g1{xq, sx, w13, s13, perm, tiles, n_tiles, nullptr, hq, sh, nullptr, H, I, k, I / PBK};
  int rc = launch_prefill_exact<PF_GATE_UP>(g1, max_tiles, s);
  if (rc) return rc;
  PrefillArgs g2{hq, sh, w2, s2, perm, tiles, n_tiles, pairs, nullptr, nullptr, nullptr, I, H, k, H / PBN};
  return launch_prefill_exact<PF_DOWN>(g2, max_tiles, s);
}
