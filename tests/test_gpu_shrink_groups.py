"""lorax_sgmv_shrink_groups: the shrinks of several rank groups over one x in one launch, against fp64 and against one
launch per group.  Sizes at the edges: one-row tiles, 16- and 32-row tiles, every stacked rank, groups without rows, more
tiles than CUs; and launches that cut the hidden dimension into parts, of stages that do not divide among them, of some
groups further than of others and of some not at all.  ROUTES says
what each case has to run as, so that none compares the calls per group with themselves."""

import pytest
import torch

from lorax_amd import _native
from lorax_amd.adapters import _tile_plans
from lorax_amd.sgmv import get_shrink_scratch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _group(rank, count, spans, rows, h_in, dtype, gen):
    stacks = [[torch.randn((2, rank, h_in), generator=gen).mul_(0.02).to(dtype).cuda() for _ in spans] for _ in range(count)]
    tables = [torch.tensor([w.data_ptr() for w in ws], dtype=torch.int64, device=DEV) for ws in stacks]
    starts, ends = [a for a, _ in spans], [b for _, b in spans]
    s, e = (torch.tensor(t, dtype=torch.int32, device=DEV) for t in (starts, ends))
    tiles = _tile_plans(starts, ends, len(spans), DEV, rank)[0]
    v = torch.randn((count, rows, rank), generator=gen).to(dtype).cuda()
    return stacks, tables, s, e, tiles, v


# (rank, projections, row counts of its segments) per group
CASES = {
    "four ranks": (1024, [(8, 3, [100, 1, 33]), (16, 3, [17, 200]), (32, 3, [90, 16]), (64, 2, [130])]),
    "every stacked rank": (384, [(8, 1, [70]), (32, 1, [71]), (24, 2, [72]), (64, 1, [73]), (40, 2, [74]), (48, 2, [75]),
                                 (56, 2, [76]), (128, 1, [77])]),
    "an odd number of stages": (128 * 17, [(16, 1, [300]), (64, 2, [300, 1, 1])]),
    "a group without rows": (512, [(16, 2, [300]), (8, 1, [0]), (32, 1, [250])]),
    "many tiles": (256, [(64, 2, [1500]), (128, 1, [33] * 60)]),
    "32-row tiles": (256, [(128, 1, [4096]), (64, 1, [64])]),
    # 67 stages
    "parts, four ranks": (128 * 67, [(8, 3, [100, 1, 33]), (16, 3, [17, 200]), (32, 3, [90, 16]), (64, 2, [130])]),
    "parts, a group without rows": (128 * 67, [(16, 2, [300]), (8, 1, [0]), (32, 1, [250])]),
    "parts, every stacked rank": (128 * 67, [(8, 1, [700]), (16, 1, [33] * 9), (24, 1, [71]), (40, 2, [9]), (48, 2, [17]),
                                             (56, 2, [31]), (128, 1, [65])]),
    "parts, 32-row tiles": (128 * 67, [(128, 1, [4096]), (64, 1, [64])]),
    "parts, some groups whole": (128 * 67, [(32, 1, [820]), (16, 1, [190]), (64, 1, [730]), (32, 2, [730]), (8, 2, [190])]),
    "parts, the first group whole": (128 * 67, [(16, 1, [190]), (8, 1, [0]), (32, 1, [820]), (64, 1, [730]), (32, 2, [730]),
                                                (8, 2, [190])]),
}
# (parts of every group's hidden dimension, heights of the groups' tiles)
ROUTES = {
    "four ranks": ([1, 1, 1, 1], {16}), "every stacked rank": ([1] * 8, {16}), "an odd number of stages": ([1, 1], {16}),
    "a group without rows": ([1, 0, 1], {16}), "many tiles": ([1, 1], {16}), "32-row tiles": ([1, 1], {16, 32}),
    "parts, four ranks": ([6, 6, 6, 6], {16}), "parts, a group without rows": ([7, 0, 7], {16}),
    "parts, every stacked rank": ([4, 4, 5, 8, 8, 8, 8], {16}), "parts, 32-row tiles": ([3, 2], {16, 32}),
    "parts, some groups whole": ([2, 1, 3, 3, 1], {16}), "parts, the first group whole": ([1, 0, 2, 3, 3, 1], {16}),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("accumulate", [True, False])
@pytest.mark.parametrize("case", list(CASES))
def test_groups_in_one_launch(case, accumulate, dtype):
    h_in, spec = CASES[case]
    gen = torch.Generator().manual_seed(len(case))
    rows = sum(sum(lens) for _, _, lens in spec) + 3  # three rows outside every segment
    assert rows > 512
    x = torch.randn((rows, h_in), generator=gen).to(dtype).cuda()
    groups, pos = [], 0
    for rank, count, lens in spec:
        spans = []
        for n in lens:
            spans.append((pos, pos + n))
            pos += n
        groups.append(_group(rank, count, spans, rows, h_in, dtype, gen))
    tmp = get_shrink_scratch(DEV)
    shrinks = [(list(g[5].unbind(0)), g[1], g[2], g[3], g[4]) for g in groups]
    parts, heights = ROUTES[case]
    assert {g[4].tile_rows for g in groups} == heights
    assert _native.sgmv_shrink_groups_parts_of(shrinks, x, tmp, 1, accumulate) == parts

    def run(apart):
        vs = [g[5].clone() for g in groups]
        calls = [(list(v.unbind(0)), g[1], g[2], g[3], g[4]) for v, g in zip(vs, groups)]
        if apart:
            for ys, tables, s, e, tiles in calls:
                _native.sgmv_shrink_multi(ys, x, tables, s, e, tmp, 1, 0.5, accumulate, tiles)
        else:
            _native.sgmv_shrink_groups(calls, x, tmp, 1, 0.5, accumulate)
        torch.cuda.synchronize()
        return vs

    together, apart = run(False), run(True)
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for (stacks, _, s, e, _, v0), got, other in zip(groups, together, apart):
        want, inside = v0.double(), torch.zeros(rows, dtype=torch.bool, device=DEV)
        for i, (a, b) in enumerate(zip(s.tolist(), e.tolist())):
            inside[a:b] = True
            for p, ws in enumerate(stacks):
                update = (0.5 * (x[a:b].double() @ ws[i][1].double().t())).to(dtype).double()
                want[p, a:b] = update + (want[p, a:b] if accumulate else 0)
        assert torch.equal(got[:, ~inside], v0[:, ~inside])
        # two roundings of the storage type (update, sum), each at most half an ulp, and fp32 sums
        norm = torch.linalg.norm(want)
        assert torch.linalg.norm(got.double() - want) <= 2 * eps * norm
        assert torch.linalg.norm(got.double() - other.double()) <= 2 * eps * norm

    # fixed-order sums do not depend on how the groups are launched
    before = _native.set_fixed_order_shrink(True)
    try:
        assert _native.sgmv_shrink_groups_parts(shrinks, x, tmp, 1, accumulate) == 1
        for a, b in zip(run(False), run(True)):
            assert torch.equal(a, b)
    finally:
        _native.set_fixed_order_shrink(before)


@pytest.mark.parametrize("rank,count", [(10, 4), (12, 2), (18, 4), (12, 4)])
def test_other_ranks_are_refused(rank, count):
    gen = torch.Generator().manual_seed(rank)
    x = torch.randn((600, 256), generator=gen).to(torch.bfloat16).cuda()
    calls = []
    for start in (0, 300):
        _, tables, s, e, tiles, v = _group(rank, count, [(start, start + 300)], 600, 256, torch.bfloat16, gen)
        calls.append((list(v.unbind(0)), tables, s, e, tiles))
    before = [[v.clone() for v in vs] for vs, *_ in calls]
    with pytest.raises(RuntimeError, match="No suitable kernel"):
        _native.sgmv_shrink_groups(calls, x, get_shrink_scratch(DEV), 0)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for vs, old in zip((c[0] for c in calls), before) for a, b in zip(vs, old))
