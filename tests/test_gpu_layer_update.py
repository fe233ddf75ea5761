"""lorax_layer_update (a layer's launches from one native call) against the general path of layers.py, which issues the
same launches one by one: the outputs are the same bits."""

import random

import pytest
import torch

from lorax_amd import _native
from lorax_amd.adapters import LORA, AdapterBatchData, LayerAdapterWeights, LoraConfig, LoraWeights
from lorax_amd.layers import TensorParallelMultiAdapterLinear
from lorax_amd.synthetic import make_meta

pytestmark = pytest.mark.gpu

NAMES = ["q_proj", "k_proj", "v_proj"]


def _layer(ranks, h_in, h_out, dtype, gen):
    layer = LayerAdapterWeights()
    for a, r in enumerate(ranks, start=1):
        wa = [torch.randn((h_in, r), generator=gen).mul_(0.02).to(dtype).cuda() for _ in range(2)]
        wb = [torch.randn((r, h_out), generator=gen).mul_(0.02).to(dtype).cuda() for _ in range(2)]
        layer.add_adapter(a, LoraWeights(wa, wb, LoraConfig(r=r)))
    return layer


# (ranks of the adapters, h_in, widths, run lengths; 0 = adapter 0, which has no weights, in every third run)
CASES = {
    "one row": ([16], 512, [512, 128, 128], False, [1]),
    "fused decode": ([8, 16], 512, [512, 128, 128], False, [1] * 23),
    "decode of four ranks, two launches of problems": ([8, 16, 32, 64, 24, 40], 512, [512, 2048, 128], False, [1] * 37),
    "wide projections, 16 records of rank 16": ([16] * 16, 1024, [14336, 128, 128], False, [1] * 24),
    "wide projections, 17 records of rank 16": ([16] * 17, 1024, [14336, 128, 2056], False, [1] * 26),
    "wide projections, rank 8": ([8] * 3, 1024, [16384, 16392, 128], False, [1] * 9),
    "wide projections, two ranks": ([8, 16], 1024, [14336, 128, 4104], False, [1] * 5),
    "short prefill, rank 16": ([16], 1024, [512, 128, 128], True, [3, 1, 40, 17]),
    "prefill of four ranks": ([8, 16, 32, 64], 1024, [512, 136, 128], True, [200, 90, 1, 300, 33]),
    "prefill with decode rows": ([16, 32], 1024, [512, 128, 128], True, [400, 300] + [1] * 90),
    "decode rows only, as prefill": ([32], 512, [512, 128, 128], True, [1, 2] * 25),
    "odd hidden size, rank 24": ([24], 200, [72, 128, 128], True, [100, 50, 7]),
    "odd hidden size, rank 16, many rows": ([16], 200, [72, 128, 128], True, [400, 350, 7]),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", list(CASES))
def test_layer_update_matches_the_general_path(case, dtype):
    ranks, h_in, widths, prefill, lens = CASES[case]
    gen = torch.Generator().manual_seed(len(case))
    rng = random.Random(len(case))
    weights = {n: _layer(ranks, h_in, w, dtype, gen) for n, w in zip(NAMES, widths)}
    weights["k_proj"].remove_adapter(len(ranks) if len(ranks) > 1 else 0)  # projections may differ in their adapters
    owners = [0 if i % 3 == 2 else rng.randrange(1, len(ranks) + 1) for i in range(len(lens))]
    indices = [a for a, n in zip(owners, lens) for _ in range(n)]
    meta = make_meta(indices, torch.device("cuda", 0))
    x = torch.randn((len(indices), h_in), generator=gen).to(dtype).cuda()
    y0 = torch.randn((len(indices), sum(widths)), generator=gen).to(dtype).cuda()

    outs = []
    for native in (True, False):
        data = AdapterBatchData.from_meta(meta, weights, prefill=prefill)
        if not native:
            for per_type in data.data.values():
                assert per_type[LORA].rank_data  # whoever holds the tables gets the general path
        assert all((per_type[LORA].packed_tables is not None) == native for per_type in data.data.values())
        y = y0.clone()
        linear = TensorParallelMultiAdapterLinear.load(lambda x, y=y: y, 1, NAMES, widths)
        taken = linear._native_update(y0.clone(), x, data, [(n, s, s + w) for n, s, w in zip(NAMES, (0, 512, 640), widths)]) \
            if widths[0] == 512 and widths[1] == 128 else None
        assert taken in (None, native)
        linear(x, data)
        outs.append(y)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert not torch.equal(outs[0], y0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,h_out,adapters,tokens", [(16, 14336, 1, 1), (16, 16384, 16, 16), (16, 2056, 5, 23), (8, 16384, 64, 64),
                                                       (8, 4104, 2, 7)])
def test_few_decode_rows_of_wide_projections(rank, h_out, adapters, tokens, dtype):
    """The single-launch update of wide projections of a small decode batch against fp64."""
    gen = torch.Generator().manual_seed(h_out + tokens)
    weights = {"up_proj": _layer([rank] * adapters, 4096, h_out, dtype, gen)}
    owners = [1 + i % adapters for i in range(tokens)]
    meta = make_meta(owners, torch.device("cuda", 0))
    data = AdapterBatchData.from_meta(meta, weights)
    x = torch.randn((tokens, 4096), generator=gen).to(dtype).cuda()
    y0 = torch.randn((tokens, h_out), generator=gen).to(dtype).cuda()
    y = y0.clone()
    TensorParallelMultiAdapterLinear.load(lambda _: y, 1, ["up_proj"], [h_out])(x, data)
    want = y0.double()
    for t, a in enumerate(owners):
        w = weights["up_proj"].adapter_weights[a]
        v = (x[t].double() @ w.weights_a_t[1].double().t()).to(dtype).double()
        want[t] += (v @ w.weights_b_t[1].double().t()).to(dtype).double()
    # roundings of v, of the update and of the sum, each at most half an ulp, and fp32 sums
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert torch.linalg.norm(y.double() - want) <= 2 * eps * torch.linalg.norm(want)


def test_layer_update_leaves_other_operands_to_the_general_path():
    gen = torch.Generator().manual_seed(5)
    weights = {"q_proj": _layer([16], 512, 256, torch.bfloat16, gen)}
    meta = make_meta([1] * 4, torch.device("cuda", 0))
    x = torch.randn((4, 512), generator=gen).to(torch.bfloat16).cuda()
    y = torch.zeros((4, 256), dtype=torch.bfloat16, device="cuda")
    for bad_x, bad_y in [(x.float(), y), (x, y.float()), (x[:3], y), (x.cpu(), y), (x.t().contiguous().t(), y)]:
        data = AdapterBatchData.from_meta(meta, weights)
        linear = TensorParallelMultiAdapterLinear.load(lambda _, out=bad_y: out, 0, ["q_proj"], [256])
        with pytest.raises(RuntimeError):
            linear(bad_x, data)
    assert torch.count_nonzero(y).item() == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,h_in,widths,records", [
    (8, 1024, [8192, 1024, 1024], [16, 16, 16]),    # one-block slices, gaps in the plain grid
    (8, 512, [1024, 8200, 264], [20, 41, 3]),       # projections of different record counts, the wide one not first
    (8, 512, [8192, 1024, 1024], [43, 43, 43]),     # more half slices than CUs: whole ones
    (8, 512, [14336, 1024], [64, 64]),              # more whole slices than CUs
    (16, 1024, [8192, 1024, 1024, 16], [16, 16, 16, 0]),
    (16, 512, [4096, 1024, 1024], [12, 15, 9]),
    (16, 512, [2048, 512, 512], [50, 50, 50]),
])
def test_one_launch_for_unequal_projections(rank, h_in, widths, records, dtype):
    """The single-launch update of wide and narrow projections together, whose workgroups are numbered without gaps,
    against one launch each: the same bits, and nothing outside their columns."""
    print(f"case rank={rank} h_in={h_in} widths={widths} records={records} dtype={dtype}", flush=True)
    gen = torch.Generator().manual_seed(rank + sum(widths))
    tokens = 3 * max(records) + 2
    x = torch.randn((tokens, h_in), generator=gen).to(dtype).cuda()
    y0 = torch.randn((tokens, sum(widths) + 16), generator=gen).to(dtype).cuda()
    problems, keep, off = [], [], 8
    for width, n in zip(widths, records):
        a = torch.randn((max(n, 1), 2, rank, h_in), generator=gen).mul_(0.05).to(dtype).cuda()
        b = torch.randn((max(n, 1), 2, width, rank), generator=gen).mul_(0.05).to(dtype).cuda()
        plan = torch.zeros((n, 8), dtype=torch.int64)
        for i in range(n):  # one to three tokens each; every seventh record is padding
            toks = [3 * i + k for k in range(1 + i % 3)]
            plan[i] = torch.tensor([0 if i % 7 == 6 else len(toks), *toks, *[toks[0]] * (4 - len(toks)), a[i].data_ptr(),
                                    b[i].data_ptr(), 0])
        keep.append((a, b))
        problems.append((plan.cuda(), off, width))
        off += width
    together, apart = y0.clone(), y0.clone()
    _native.bgmv_lora_multi([(together, x, plan, o, w) for plan, o, w in problems], rank, 1)
    for plan, o, w in problems:
        _native.bgmv_lora_multi([(apart, x, plan, o, w)], rank, 1)
    torch.cuda.synchronize()
    # (launches of another size may cut other column slices; an element's sums do not depend on it)
    assert torch.equal(together, apart)
    assert not torch.equal(together, y0)
    assert torch.equal(together[:, :8], y0[:, :8]) and torch.equal(together[:, off:], y0[:, off:])


@pytest.mark.parametrize("native", [True, False])
def test_prefill_layers_on_two_streams(native):
    """Layers of two prefill batches whose shrinks cut the hidden dimension, issued on two streams at once: every call has a
    scratch of its own, so the outputs are the bits of one after the other."""
    gen = torch.Generator().manual_seed(3)
    h_in, width, lens = 4096, 512, [300, 410, 90]
    jobs = []
    for _ in range(2):
        weights = {"q_proj": _layer([64, 32, 16], h_in, width, torch.bfloat16, gen)}
        meta = make_meta([a for a, n in zip((1, 2, 3), lens) for _ in range(n)], torch.device("cuda", 0))
        data = AdapterBatchData.from_meta(meta, weights, prefill=True)
        if not native:
            assert data.data["q_proj"][LORA].rank_data
        x = torch.randn((sum(lens), h_in), generator=gen).to(torch.bfloat16).cuda()
        jobs.append((data, x, torch.randn((sum(lens), width), generator=gen).to(torch.bfloat16).cuda(), weights))

    def run(streams):
        ys = [y0.clone() for _, _, y0, _ in jobs]
        torch.cuda.synchronize()
        for _ in range(10):
            for (data, x, _, _), y, stream in zip(jobs, ys, streams):
                with torch.cuda.stream(stream):
                    TensorParallelMultiAdapterLinear.load(lambda _, y=y: y, 0, ["q_proj"], [width])(x, data)
        torch.cuda.synchronize()
        return ys

    here = torch.cuda.current_stream()
    for a, b in zip(run([here, here]), run([torch.cuda.Stream(), torch.cuda.Stream()])):
        assert torch.equal(a, b)


@pytest.mark.parametrize("ranks,lens", [
    ([64], [500, 40, 160]),          # three groups of one projection in one launch
    ([64], [300, 240]),              # ... of so few tiles that the hidden dimension is cut into parts
    ([48, 64], [300, 17, 1, 290]),   # groups of two ranks
    ([32], [700]),                   # one group of all three projections
    ([128, 64], [400, 200]),         # a rank that fills a group by itself
    ([64], [9000]),                  # tiles of 48 rows and more: launches of their own
    ([64, 32], [9000, 300, 280]),    # ... next to a rank that is then alone
    ([128, 32], [700, 300]),         # a rank above 64
])
def test_prefill_shrinks_of_several_groups(ranks, lens):
    """The groups that a layer's shrinks are cut into, natively and on the general path: the same bits, and the update of
    fp64 within the roundings of v and of the update, 16 rows of a projection at a time."""
    print(f"case ranks={ranks} lens={lens}", flush=True)
    gen = torch.Generator().manual_seed(sum(lens))
    h_in, widths, dtype, rows = 4096, [512, 136, 128], torch.bfloat16, sum(lens)
    weights = {n: _layer(ranks, h_in, w, dtype, gen) for n, w in zip(NAMES, widths)}
    owners = [1 + i % len(ranks) for i in range(len(lens))]
    meta = make_meta([a for a, n in zip(owners, lens) for _ in range(n)], torch.device("cuda", 0))
    x = torch.randn((rows, h_in), generator=gen).to(dtype).cuda()
    y0 = torch.randn((rows, sum(widths)), generator=gen).to(dtype).cuda()

    def run(native, y):
        data = AdapterBatchData.from_meta(meta, weights, prefill=True)
        if not native:
            assert all(per_type[LORA].rank_data for per_type in data.data.values())
        TensorParallelMultiAdapterLinear.load(lambda _: y, 1, NAMES, widths)(x, data)
        torch.cuda.synchronize()
        return y

    added, update = run(True, y0.clone()), run(True, torch.zeros_like(y0))
    assert torch.equal(added, run(False, y0.clone()))
    assert torch.equal(added, y0 + update)  # the update is rounded before it is added
    want, row = torch.zeros(y0.shape, dtype=torch.float64, device="cuda"), 0
    for a, n in zip(owners, lens):
        col = 0
        for name, w in zip(NAMES, widths):
            lw = weights[name].adapter_weights[a]
            v = (x[row:row + n].double() @ lw.weights_a_t[1].double().t()).to(dtype).double()
            want[row:row + n, col:col + w] = (v @ lw.weights_b_t[1].double().t()).to(dtype).double()
            col += w
        row += n
    # v and the update are rounded on both sides, half an ulp (2^-9) each; fp32 sums are far below
    for col, w in zip([0, 512, 648], widths):
        diff, ref = ((t[:, col:col + w].square().sum(1)) for t in (update.double() - want, want))
        blocks = lambda t: torch.nn.functional.pad(t, (0, -rows % 16)).view(-1, 16).sum(1).sqrt()
        assert torch.all(blocks(diff) <= 4 * 2.0**-9 * blocks(ref)), f"columns from {col}"
