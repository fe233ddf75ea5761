"""Launches of up to four problems pass their arguments in a smaller struct than launches of up to sixteen - decode launches
of several ranks only with few routing records: at and beside those edges, several problems in one launch against one
launch each, bit for bit."""

import pytest
import torch

from lorax_amd import _native
from lorax_amd.adapters import build_bgmv_plan
from tests.helpers import ptr_table, randn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
RANKS = (8, 64, 16, 128, 32)


@pytest.mark.parametrize("count", [1, 4, 5, 16])
def test_expands(count):
    gen = torch.Generator().manual_seed(count)
    T, width = 70, 264
    y0 = randn((T, width * count), 0.5, gen, torch.bfloat16, DEV)
    s, e = (torch.tensor(b, dtype=torch.int32, device=DEV) for b in ([0, 33], [33, 70]))
    problems, keep = [], []
    for i in range(count):
        r = RANKS[i % len(RANKS)]
        bt = [randn((1, width, r), 0.05, gen, torch.bfloat16, DEV) for _ in range(2)]
        keep.append(bt)
        problems.append((randn((T, r), 1.0, gen, torch.bfloat16, DEV), ptr_table(bt, DEV), s, e, i * width, width, None))
    together, apart = y0.clone(), y0.clone()
    _native.sgmv_expand_multi([(together, *p) for p in problems], 0)
    for p in problems:
        _native.sgmv_expand_multi([(apart, *p)], 0)
    torch.cuda.synchronize()
    assert torch.equal(together, apart) and not torch.equal(together, y0)


@pytest.mark.parametrize("times", [1, 4, 5, 9])  # 3, 8, 11 and 19 routing records a problem: 32 and 44 in launches of four
@pytest.mark.parametrize("planned", [True, False])
@pytest.mark.parametrize("count", [1, 4, 5, 16])
def test_decode_shrinks_and_expands(count, planned, times):
    gen = torch.Generator().manual_seed(count)
    T, h_in, width = 9 * times, 512, 264
    x = randn((T, h_in), 1.0, gen, torch.bfloat16, DEV)
    y0 = randn((T, width * count), 0.5, gen, torch.bfloat16, DEV)
    slots = [0, 1, -1, 1, 0, 1, 1, 1, 1] * times
    idx = torch.tensor(slots, device=DEV)
    shrinks, expands, plans, keep = [], [], [], []
    for i in range(count):
        r = RANKS[i % len(RANKS)]
        a = [randn((1, r, h_in), 0.05, gen, torch.bfloat16, DEV) for _ in range(2)]
        b = [randn((1, width, r), 0.05, gen, torch.bfloat16, DEV) for _ in range(2)]
        keep.append((a, b))
        records = build_bgmv_plan(slots, [w.data_ptr() for w in a], [w.data_ptr() for w in b])
        plans.append(torch.tensor(records, dtype=torch.int64, device=DEV).reshape(-1, 8))
        v = torch.zeros((T, r), dtype=torch.bfloat16, device=DEV)
        shrinks.append((v, x, ptr_table(a, DEV), idx, 0, None))
        expands.append((v, ptr_table(b, DEV), idx, i * width, width))

    def run(step):
        y = y0.clone()
        for v, *_ in shrinks:
            v.zero_()
        for problems, add in ((shrinks, False), ([(y, *p) for p in expands], True)):
            for i in range(0, count, step):
                _native.bgmv_multi(problems[i:i + step], 0, 1.0, add, plans=plans[i:i + step] if planned else None)
        torch.cuda.synchronize()
        return y

    together = run(16)
    assert torch.equal(together, run(1)) and not torch.equal(together, y0)
