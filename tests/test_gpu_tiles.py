"""The combine's forms, and the LDS-tiled grouped GEMMs at the edges of their tiles: experts whose row counts lie around the
16-row fragments, the two wave groups' shares and the 128-, 144- and 192-row tiles, with K loops of 4 and
5 blocks and with rows of a multiple of 4 KB."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe_oracle as orc
from tests.helpers import TOL_MAX_ABS, TOL_MEAN_REL, errors, np_f32, tile_rows, to_bf16, to_dev, to_f8

pytestmark = pytest.mark.gpu

ROWS = [1, 0, 15, 16, 17, 32, 33, 80, 81, 127, 129, 143, 144, 145, 160, 191, 192, 193, 289, 400]


def pairs_of(rng, rows):
    """One slot per token, expert e holding rows[e] of them, tokens in a random order."""
    ids = np.repeat(np.arange(len(rows), dtype=np.int64), rows)
    return rng.permutation(ids)[:, None]


# (repeat: experts rows, rows, .. that many times over, with the same weights each time)
@pytest.mark.parametrize("kind,H,I,rows,repeat", [
    ("fp8", 512, 512, ROWS, 1),                      # 4 K blocks
    ("fp8", 1024, 640, ROWS, 1),                     # 5 K blocks in the down GEMM
    ("fp8", 512, 4096, [145, 0, 17, 400], 1),        # the down GEMM's rows are 4 KB
    ("fp8", 512, 1024, ROWS, 6),                     # 4 K blocks in gate_up, four and more items a workgroup
    ("fp8", 2048, 512, ROWS, 6),                     # the same in the down GEMM
    ("fp8", 2304, 512, [144, 1, 145, 81, 300], 1),   # exact accumulation, 18 K blocks
    ("fp8", 4096, 512, ROWS, 1),                     # exact, gate_up's rows are 4 KB
    ("fp8", 2304, 512, ROWS, 6),                     # exact, 4 K blocks in the down GEMM, its items as above
    ("bf16", 256, 256, ROWS, 1),                     # 4 K blocks
    ("bf16", 512, 384, ROWS, 1),                     # 6 K blocks in the down GEMM
    ("bf16", 2048, 256, ROWS, 1),                    # gate_up's rows are 4 KB
    ("bf16", 256, 2048, [193, 0, 17, 192, 300], 1),  # the down GEMM's rows are 4 KB
    ("bf16", 256, 1024, ROWS, 6),                    # 4 K blocks in gate_up, four and more items a workgroup
    ("bf16", 2048, 256, ROWS, 6),                    # the same in the down GEMM
])
def test_tile_edges(pkg, dev, kind, H, I, rows, repeat):
    """Few experts take 128-row tiles (or 144 for exact sums) and at most one or two work items per workgroup;
    with many experts the tiles have 192 rows, and a workgroup goes from item to item with other row counts."""
    rng = np.random.default_rng(H + I + len(rows))
    E0, E, ids = len(rows), len(rows) * repeat, pairs_of(rng, rows * repeat)
    T = len(ids)
    fp8, exact = int(kind == "fp8"), kind == "fp8" and H > 2048
    lib = pkg._lib.load()
    assert int(lib.moe_mi355x_block_numerics_key(T, H, I, E, 1, fp8)) & 0xFFFF == 128

    height, tile = tile_rows(pkg, rows * repeat, T, H, I, 1, fp8)
    assert height == (144 if exact else 128 if repeat == 1 else 192)
    if repeat > 1:  # more than three rounds of the persistent grid
        tiles = sum(-(-r // h) for r, h in zip(rows * repeat, tile.tolist()))
        assert tiles * max(I // 128, H // 256) > 3 * torch.cuda.get_device_properties(dev).multi_processor_count
    x = orc.gen_normal_bf16(rng, (T, H))
    w = orc.round_bf16(rng.uniform(0.2, 1.0, (T, 1)).astype(np.float32))
    w13 = orc.gen_normal_bf16(rng, (E0, 2 * I, H), 0.02)
    w2 = orc.gen_normal_bf16(rng, (E0, H, I), 0.02)
    if fp8:
        (q13, s13), (q2, s2) = orc.quantize_weight_fp8(w13), orc.quantize_weight_fp8(w2)
        ref = orc.experts_fp8(x, ids % E0, w, q13, s13, q2, s2)
        wd = (to_f8(np.tile(q13, (repeat, 1, 1)), dev), to_dev(np.tile(s13, (repeat, 1, 1)), dev),
              to_f8(np.tile(q2, (repeat, 1, 1)), dev), to_dev(np.tile(s2, (repeat, 1, 1)), dev))
        run = pkg.experts_fp8
    else:
        ref = orc.experts_bf16(x, ids % E0, w, w13, w2, acc=np.float32)
        wd = (to_bf16(w13, dev).repeat(repeat, 1, 1), to_bf16(w2, dev).repeat(repeat, 1, 1))
        run = pkg.experts_bf16
    out = run(to_bf16(x, dev), to_dev(ids, dev), to_bf16(w, dev), *wd)
    max_abs, mean_rel = errors(np_f32(out), ref)
    assert max_abs <= TOL_MAX_ABS and mean_rel <= TOL_MEAN_REL, (max_abs, mean_rel)
    # a row's sums depend on its expert's weights alone: in another place of the tiles it gives the same bits
    p = rng.permutation(T)
    moved = run(to_bf16(x[p], dev), to_dev(ids[p], dev), to_bf16(w[p], dev), *wd)
    assert torch.equal(moved, out[torch.from_numpy(p).to(dev)])


@pytest.mark.parametrize("k", [1, 8, 12, 16])
@pytest.mark.parametrize("id_type", [torch.int32, torch.int64])
@pytest.mark.parametrize("T,H,I", [
    (7, 256, 256),     # pair rows that the GEMM has weighted: streaming tiles
    (130, 2304, 256),  # the same, two column blocks
    (130, 768, 512),   # LDS tiles, whose pair rows the combine weights: one column block of 96 threads
    (130, 2304, 512),  # the same, two column blocks (exact accumulation)
])
def test_combine_forms(pkg, dev, T, H, I, k, id_type):
    """Pair rows weighted already (H or I below the LDS tiles' or few pairs), weights one by one (k % 8 != 0,
    or rows of 8 at an odd address) and eight at a time, one and two passes over the slots, ids of both
    sizes with sentinels on either side of the range (for 64-bit ids also ones whose low word is an
    expert), one and two column blocks with a remainder."""
    rng = np.random.default_rng(T + k)
    E = 16
    key = int(pkg._lib.load().moe_mi355x_block_numerics_key(T, H, I, E, k, 1)) & 0xFFFF
    assert (key == 128) == (I == 512)  # the LDS tiles leave the weights to the combine
    ids = np.argsort(rng.random((T, E)), axis=1)[:, :k].astype(np.int64)
    ids[0, 0], ids[T // 2, -1] = -1, E
    if id_type == torch.int64:
        ids[1, 0], ids[2, 0] = (1 << 32) + 3, -(1 << 32) + 3
    x = orc.gen_normal_bf16(rng, (T, H))
    w = orc.round_bf16(rng.uniform(0.05, 0.5, (T, k)).astype(np.float32))
    q13, s13 = orc.quantize_weight_fp8(orc.gen_normal_bf16(rng, (E, 2 * I, H), 0.02))
    q2, s2 = orc.quantize_weight_fp8(orc.gen_normal_bf16(rng, (E, H, I), 0.02))
    wd = (to_f8(q13, dev), to_dev(s13, dev), to_f8(q2, dev), to_dev(s2, dev))
    ok = (ids >= 0) & (ids < E)
    ref = orc.experts_fp8(x, np.where(ok, ids, 0), np.where(ok, w, 0.0), q13, s13, q2, s2)
    di = torch.from_numpy(ids).to(id_type).to(dev)
    out = pkg.experts_fp8(to_bf16(x, dev), di, to_bf16(w, dev), *wd)
    max_abs, mean_rel = errors(np_f32(out), ref)
    assert max_abs <= TOL_MAX_ABS and mean_rel <= TOL_MEAN_REL, (max_abs, mean_rel)
    # the rows' address alone decides between one by one and eight at a time
    odd = torch.empty(T * k + 1, dtype=torch.bfloat16, device=dev)[1:].view(T, k).copy_(to_bf16(w, dev))
    assert odd.data_ptr() % 16 == 2
    assert torch.equal(pkg.experts_fp8(to_bf16(x, dev), di, odd, *wd), out)


@pytest.mark.parametrize("kind,H,I", [
    ("fp8", 512, 512),
    ("fp8", 512, 4096),   # the down GEMM's rows are 4 KB
    ("fp8", 4096, 512),   # exact accumulation
    ("bf16", 2048, 256),  # gate_up's rows are 4 KB
    ("bf16", 256, 2048),  # the down GEMM's rows are 4 KB
])
def test_expert_index_leaves_the_bits(pkg, dev, kind, H, I):
    """A pair's bits depend on its expert's weights, not on the expert's index in the call: the same
    experts in another order, and a share of them under local indices (sentinels for the others)."""
    rows = [40, 1, 150, 17, 200, 33]
    rng = np.random.default_rng(H + I)
    E, ids = len(rows), pairs_of(rng, rows)
    T = len(ids)
    x = to_bf16(orc.gen_normal_bf16(rng, (T, H)), dev)
    w = to_bf16(orc.round_bf16(rng.uniform(0.2, 1.0, (T, 1)).astype(np.float32)), dev)
    w13 = orc.gen_normal_bf16(rng, (E, 2 * I, H), 0.02)
    w2 = orc.gen_normal_bf16(rng, (E, H, I), 0.02)
    if kind == "fp8":
        (q13, s13), (q2, s2) = orc.quantize_weight_fp8(w13), orc.quantize_weight_fp8(w2)
        wd = (to_f8(q13, dev), to_dev(s13, dev), to_f8(q2, dev), to_dev(s2, dev))
        run = pkg.experts_fp8
    else:
        wd = (to_bf16(w13, dev), to_bf16(w2, dev))
        run = pkg.experts_bf16

    def take(order):
        """The call with the experts of ``order`` alone, in that order."""
        local = np.full(E, -1, dtype=np.int64)
        local[order] = np.arange(len(order))
        sel = torch.as_tensor(order, device=dev)
        part = [t.view(torch.uint8)[sel].view(t.dtype) if t.dtype == torch.float8_e4m3fn else t[sel] for t in wd]
        return run(x, to_dev(local[ids], dev), w, *part)

    whole = take(list(range(E)))
    assert torch.equal(take([3, 0, 5, 1, 2, 4]), whole)
    share = take([2, 4, 5])
    mine = to_dev(np.isin(ids[:, 0], [2, 4, 5]), dev)
    assert torch.equal(share[mine], whole[mine]) and not share[~mine].any()
