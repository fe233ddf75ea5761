"""lorax_layer_update (a layer's launches from one native call) against the general path of layers.py, which issues the
same launches one by one: the outputs are the same bits."""

import random

import pytest
import torch

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
