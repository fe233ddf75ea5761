"""The streaming shrink of a short prefill batch with several projections in one launch (lorax_sgmv_shrink_multi, up to
512 rows) against one launch per projection: the same sums in the same order, so the same bits; and against fp64."""

import pytest
import torch

from lorax_amd import _native
from lorax_amd.sgmv import get_shrink_scratch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,count,lens,h_in", [
    (8, 4, [1], 256), (16, 3, [3, 0, 5, 1], 512), (24, 2, [17, 4], 200), (64, 3, [100, 156, 255], 1024),
    (128, 4, [511, 1], 384), (128, 2, [2, 2, 2], 4096),
])
@pytest.mark.parametrize("accumulate", [True, False])
def test_one_launch_for_several_projections(rank, count, lens, h_in, dtype, accumulate):
    gen = torch.Generator().manual_seed(rank + count)
    rows = sum(lens) + 2  # two rows outside every segment
    assert rows <= 514
    rows = min(rows, 512)
    x = torch.randn((rows, h_in), generator=gen).to(dtype).cuda()
    ends = [min(sum(lens[: i + 1]), rows) for i in range(len(lens))]
    starts = [min(sum(lens[:i]), rows) for i in range(len(lens))]
    s, e = (torch.tensor(t, dtype=torch.int32, device="cuda") for t in (starts, ends))
    stacks = [[torch.randn((2, rank, h_in), generator=gen).mul_(0.02).to(dtype).cuda() for _ in lens] for _ in range(count)]
    tables = [torch.tensor([w.data_ptr() for w in ws], dtype=torch.int64, device="cuda") for ws in stacks]
    v0 = torch.randn((count, rows, rank), generator=gen).to(dtype).cuda()
    tmp = get_shrink_scratch(x.device)
    together, apart = v0.clone(), v0.clone()
    _native.sgmv_shrink_multi(list(together.unbind(0)), x, tables, s, e, tmp, 1, 1.0, accumulate)
    for v, table in zip(apart.unbind(0), tables):
        _native.sgmv_shrink_multi([v], x, [table], s, e, tmp, 1, 1.0, accumulate)
    want = v0.double()
    for p in range(count):
        for i, (a, b) in enumerate(zip(starts, ends)):
            update = (x[a:b].double() @ stacks[p][i][1].double().t()).to(dtype).double()
            want[p, a:b] = update + (want[p, a:b] if accumulate else 0)
    torch.cuda.synchronize()
    # launches of another size may give a workgroup another number of A's rows; a row's sum does not depend on it
    assert torch.equal(together, apart)
    # two roundings of the storage type (update, sum), each at most half an ulp, and fp32 sums
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert torch.linalg.norm(together.double() - want) <= 2 * eps * torch.linalg.norm(want)


@pytest.mark.parametrize("rows,h_in", [(100, 256), (900, 256)])
def test_projections_that_share_their_output_add_up(rows, h_in):
    """Two projections may add into one v: they then go out one after the other, in short and in long batches."""
    gen = torch.Generator().manual_seed(rows)
    dtype, rank = torch.bfloat16, 16
    x = torch.randn((rows, h_in), generator=gen).to(dtype).cuda()
    s, e = (torch.tensor([t], dtype=torch.int32, device="cuda") for t in (0, rows))
    stacks = [torch.randn((1, rank, h_in), generator=gen).mul_(0.02).to(dtype).cuda() for _ in range(3)]
    tables = [torch.tensor([w.data_ptr()], dtype=torch.int64, device="cuda") for w in stacks]
    v0 = torch.randn((2, rows, rank), generator=gen).to(dtype).cuda()
    together, apart = v0.clone(), v0.clone()
    tmp = get_shrink_scratch(x.device)
    _native.sgmv_shrink_multi([together[0], together[1], together[0]], x, tables, s, e, tmp, 0)
    for i, table in zip((0, 1, 0), tables):
        _native.sgmv_shrink_multi([apart[i]], x, [table], s, e, tmp, 0)
    torch.cuda.synchronize()
    assert torch.equal(together, apart)
