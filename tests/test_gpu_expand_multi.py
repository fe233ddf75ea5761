"""lorax_sgmv_expand_multi: several expands of different rank, width and segments in one launch, against one launch
each (bit for bit: every element of the update is one dot product over r whatever the tiling) and against the oracle
formula.  The batches are small enough for the launch to cut its row tiles into pieces of 128, 64 or 32 rows."""

import pytest
import torch

from lorax_amd import _native, sgmv
from tests.helpers import assert_close, ptr_table, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("parts", [
    [(8, 8, [1]), (8, 1160, [31, 0, 33])],                          # one row, one short panel; pieces of 32 rows
    [(64, 4096, [300]), (64, 1024, [300])],                         # a merged remainder: tiles higher than 256 rows
    [(16, 512, [17, 1]), (24, 640, [65]), (128, 1024, [129, 3]), (72, 8, [5])],  # every body of the mixed launch
    [(32, 4096, [700, 256, 511]), (16, 14336, [1000])],             # enough workgroups for higher pieces
])
def test_expands_of_one_launch_equal_single_launches(dtype, planned, parts):
    print(f"case dtype={dtype} planned={planned} parts={parts}", flush=True)
    gen = torch.Generator().manual_seed(sum(r + h for r, h, _ in parts))
    layer, pos, spans = 1, 1, []
    for _, _, lens in parts:  # every problem owns rows of its own
        spans.append([])
        for n in lens:
            spans[-1].append((pos, pos + n))
            pos += n + 1
    T = pos + 2
    width = sum(h for _, h, _ in parts) + 16
    y0 = randn((T, width), 0.5, gen, dtype, DEV)
    problems, weights, off = [], [], 8
    for (r, h_out, lens), seg in zip(parts, spans):
        bt = [randn((2, h_out, r), 0.05, gen, dtype, DEV) for _ in lens]
        v = randn((T, r), 1.0, gen, dtype, DEV)
        s, e = [a for a, _ in seg], [b for _, b in seg]
        tiles = None
        if planned:
            records, rows = _native.plan_tiles(s, e, T, _native.TILES_EXPAND)
            tiles = _native.TilePlan(torch.from_numpy(records.copy()).to(DEV), rows)
        problems.append([None, v, ptr_table(bt, DEV), torch.tensor(s, dtype=torch.int32, device=DEV),
                         torch.tensor(e, dtype=torch.int32, device=DEV), off, h_out, tiles])
        weights.append(bt)
        off += h_out
    for accumulate in (True, False):
        y_a, y_b = y0.clone(), y0.clone()
        _native.sgmv_expand_multi([(y_a, *p[1:]) for p in problems], layer, accumulate)
        for _, v, w, s, e, o, h, tiles in problems:
            tmp = sgmv.get_tmp_tensor_for_size(s.numel(), torch.device(DEV))
            _native.sgmv_expand(y_b, v, w, s, e, tmp, layer, o, h, True, accumulate, tiles)
        torch.cuda.synchronize()
        assert torch.equal(y_a, y_b), f"accumulate={accumulate}"
    want = y0.cpu().clone()
    for p, bt, seg in zip(problems, weights, spans):
        for w, (s, e) in zip(bt, seg):
            want[s:e, p[5]:p[5] + p[6]] = p[1].cpu()[s:e] @ w[layer].cpu().t()  # the last call overwrote
    assert_close(y_a, want, "expands of one launch")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ranks", [[8], [16], [24], [40], [72], [96], [96, 128], [16, 64], [8, 24, 32, 40, 72, 104]])
def test_infinities_of_v_stay_infinities(ranks, dtype):
    """An element of v that overflowed gives an infinite update, as a dot product over the rank does, whether or not the
    rank fills the matrix instruction's steps and whatever other ranks share the launch."""
    print(f"case dtype={dtype} ranks={ranks}", flush=True)
    gen = torch.Generator().manual_seed(sum(ranks))
    h_out, rows = 264, 37
    problems, wants, ys, stacks = [], [], [], []
    for r in ranks:
        v = randn((rows, r), 1.0, gen, dtype, DEV)
        v[3, 0], v[20, r - 1], v[36, 5] = float("inf"), float("-inf"), float("inf")
        bt = randn((1, h_out, r), 0.05, gen, dtype, DEV)
        bt[0, :, [0, 5, r - 1]] = torch.where(bt[0, :, [0, 5, r - 1]] == 0, 0.05, bt[0, :, [0, 5, r - 1]])  # no inf * 0
        s, e = (torch.tensor([t], dtype=torch.int32, device=DEV) for t in (0, rows))
        ys.append(randn((rows, h_out), 0.5, gen, dtype, DEV))
        wants.append((ys[-1].cpu().double() + v.cpu().double() @ bt[0].cpu().double().t()).to(DEV))
        problems.append((ys[-1], v, ptr_table([bt], DEV), s, e, 0, h_out, None))
        stacks.append(bt)
    _native.sgmv_expand_multi(problems, 0)
    torch.cuda.synchronize()
    for r, y, want in zip(ranks, ys, wants):
        inf = torch.isinf(want)
        assert inf[[3, 20, 36]].all() and inf.sum() == 3 * h_out
        assert torch.equal(y.double()[inf], want[inf]), f"rank {r}"
        assert_close(y[~inf], want[~inf].to(dtype), f"rank {r}")


def test_expand_multi_checks_its_problems():
    y = torch.zeros((4, 64), dtype=torch.bfloat16, device=DEV)
    v = torch.zeros((4, 16), dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(1, dtype=torch.int64, device=DEV)
    s = torch.zeros(1, dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match="y_offset=8"):
        _native.sgmv_expand_multi([(y, v, w, s, s, 8, 64, None)], 0)
    with pytest.raises(RuntimeError, match="between 1 and 16 problems"):
        _native.sgmv_expand_multi([(y, v, w, s, s, 0, 64, None)] * 17, 0)


@pytest.mark.parametrize("planned", [False, True])
@pytest.mark.parametrize("h_out", [2048, 2304, 264, 4096])  # 8, 9, 2 and 16 panel groups: dealt out with and without runs
@pytest.mark.parametrize("lens", [[1], [64, 65, 0, 300, 7], [1100, 3], [4400]])  # tile heights of 64, 80 and 256 rows
def test_every_element_of_the_expand_is_written_once(h_out, lens, planned):
    """y += 1 everywhere inside the segments and nowhere else: v and B are such that every update is exactly one."""
    print(f"case h_out={h_out} lens={lens} planned={planned}", flush=True)
    r, off = 16, 8
    starts = [sum(lens[:i]) + i + 1 for i in range(len(lens))]
    ends = [s + n for s, n in zip(starts, lens)]
    T = ends[-1] + 2
    v = torch.zeros((T, r), dtype=torch.bfloat16, device=DEV)
    v[:, 3] = 1.0
    bt = torch.zeros((1, h_out, r), dtype=torch.bfloat16, device=DEV)
    bt[:, :, 3] = 1.0
    tiles = None
    if planned:
        records, rows = _native.plan_tiles(starts, ends, T, _native.TILES_EXPAND_BATCH)
        tiles = _native.TilePlan(torch.from_numpy(records.copy()).to(DEV), rows)
    y = torch.zeros((T, h_out + 2 * off), dtype=torch.bfloat16, device=DEV)
    s, e = (torch.tensor(b, dtype=torch.int32, device=DEV) for b in (starts, ends))
    _native.sgmv_expand(y, v, ptr_table([bt] * len(lens), DEV), s, e, sgmv.get_tmp_tensor_for_size(len(lens), torch.device(DEV)),
                        0, off, h_out, True, True, tiles)
    want = torch.zeros((T, h_out + 2 * off))
    for a, b in zip(starts, ends):
        want[a:b, off:off + h_out] = 1.0
    torch.cuda.synchronize()
    assert torch.equal(y.float().cpu(), want)
