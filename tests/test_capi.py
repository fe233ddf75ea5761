"""The C-ABI shared library without a GPU: it loads, exports every function include/lorax_hip.h
declares, and rejects bad arguments on the host before anything is launched."""

import ctypes
import re
from pathlib import Path

import pytest

from lorax_amd import _native

ROOT = Path(__file__).resolve().parent.parent
HEADER = (ROOT / "include" / "lorax_hip.h").read_text()


def _declared_functions():
    body = re.sub(r"/\*.*?\*/", "", HEADER, flags=re.S)
    return sorted(set(re.findall(r"\b(lorax_[a-z0-9_]+)\s*\(", body)))


def test_library_loads():
    assert _native.available(), _native.load_error()
    assert "gfx950" in _native.version()


def test_every_declared_symbol_is_exported_and_bound():
    declared = _declared_functions()
    assert "lorax_bgmv" in declared and "lorax_sgmv_shrink" in declared and "lorax_sgmv_expand" in declared
    raw = ctypes.CDLL(str(_native.LIB_PATH))
    for name in declared:
        assert hasattr(raw, name), f"{name} is declared in lorax_hip.h but not exported"
    assert sorted(_native.EXPORTED_SYMBOLS) == declared


def test_tmp_size_is_60_bytes_per_problem():
    lib = _native.lib()
    assert [lib.lorax_sgmv_tmp_size(n) for n in (-1, 0, 1, 32, 257)] == [0, 0, 60, 1920, 15420]
    assert lib.lorax_workspace_bytes() == 8 * 1024 * 1024  # the static scratch of lorax_sgmv_shrink_static


OK, EINVAL, ENOKERNEL, ELAUNCH, ETMPSIZE = 0, 1, 2, 3, 4
P = 0x1000  # a non-null, 16-byte aligned fake address: validation failures return before any launch


def _err():
    return _native.lib().lorax_last_error().decode()


def test_bgmv_validation():
    f = _native.lib().lorax_bgmv
    assert f(None, None, None, None, 0, 4096, 8, 0, 8, 0, 1.0, 1, None) == OK  # nothing to do
    assert f(None, P, P, P, 4, 4096, 8, 0, 8, 0, 1.0, 1, None) == EINVAL and "null" in _err()
    assert f(P, P + 2, P, P, 4, 4096, 8, 0, 8, 0, 1.0, 1, None) == EINVAL and "aligned" in _err()
    assert f(P, P, P, P, 4, 4096, 8, 0, 8, 0, 1.0, 2, None) == ENOKERNEL and "No suitable kernel" in _err()
    for h_in, h_out in [(4096, 12), (4096, 136), (4100, 8), (65536, 8), (8, 1 << 20), (256, 256)]:
        assert f(P, P, P, P, 4, h_in, h_out, 0, h_out, 0, 1.0, 1, None) == ENOKERNEL, (h_in, h_out)
        assert f"h_in={h_in} h_out={h_out}" in _err()
    assert f(P, P, P, P, 4, 8, 4096, 8192, 8192, 0, 1.0, 1, None) == EINVAL  # window outside the row
    assert f(P, P, P, P, -1, 8, 4096, 0, 4096, 0, 1.0, 1, None) == EINVAL
    assert f(P, P, P, P, 4, 8, 4096, 0, 4096, -1, 1.0, 1, None) == EINVAL


def test_sgmv_shrink_validation():
    f = _native.lib().lorax_sgmv_shrink
    big = 8 * 1024 * 1024
    assert f(P, P, P, P, P, 2, 16, 4096, 16, 0, 0, 1.0, P, big - 1, 0, None) == ETMPSIZE and "8 * 1024 * 1024" in _err()
    assert f(P, P, P, P, P, 2, 16, 4096, 8, 1, 0, 1.0, P, 119, 0, None) == ETMPSIZE and "sgmv_tmp_size" in _err()
    assert f(P, P, P, P, P, 0, 16, 4096, 16, 0, 0, 1.0, P, big, 0, None) == OK  # no segments
    assert f(P, P, P, P, P, 2, 16, 4096, 16, 7, 0, 1.0, P, big, 0, None) == EINVAL  # layout
    for r, h_in in ((8, 4104), (24, 4104), (144, 4096), (12, 4096)):
        assert f(P, P, P, P, P, 2, 1000, h_in, r, 0, 0, 1.0, P, big, 0, None) == ENOKERNEL, r
    assert f(P, P, P, P, P, 2, 16, 4100, 16, 0, 0, 1.0, P, big, 0, None) == ENOKERNEL
    assert f(P, P, P, None, P, 2, 16, 4096, 16, 0, 0, 1.0, P, big, 0, None) == EINVAL
    assert f(P, P, P, P, P, 2, 16, 4096, 16, 0, 0, 1.0, P, big, 5, None) == ENOKERNEL  # dtype


def test_sgmv_shrink_multi_validation():
    f = _native.lib().lorax_sgmv_shrink_multi
    big = 8 * 1024 * 1024
    one = (_native.SgmvShrinkProblem * 1)(_native.SgmvShrinkProblem(P, P))
    two = (_native.SgmvShrinkProblem * 2)(_native.SgmvShrinkProblem(P, P), _native.SgmvShrinkProblem(P, P))
    assert f(two, 0, P, P, P, 2, 1000, 4096, 16, 0, 1.0, 1, P, big, None, 1, None) == EINVAL and "num_problems" in _err()
    assert f(two, 5, P, P, P, 2, 1000, 4096, 16, 0, 1.0, 1, P, big, None, 1, None) == EINVAL
    assert f(None, 2, P, P, P, 2, 1000, 4096, 16, 0, 1.0, 1, P, big, None, 1, None) == EINVAL
    # stacked launch (2 x 64 <= 128, h_in a multiple of 128, more than 512 rows): its own checks
    assert f(two, 2, P, P, P, 2, 1000, 4096, 64, 0, 1.0, 1, P, big - 1, None, 1, None) == ETMPSIZE
    assert f(two, 2, P, P, P, 0, 1000, 4096, 64, 0, 1.0, 1, P, big, None, 1, None) == OK  # no segments
    assert f(two, 2, P, P, None, 2, 1000, 4096, 64, 0, 1.0, 1, P, big, None, 1, None) == EINVAL and "null" in _err()
    assert f(two, 2, P, P, P, 2, 1000, 4096, 64, -1, 1.0, 1, P, big, None, 1, None) == EINVAL
    # one launch per projection (summed rank 192; or a single projection): lorax_sgmv_shrink's checks
    assert f(two, 2, P, P, P, 2, 1000, 4096, 96, 0, 1.0, 1, P, big - 1, None, 1, None) == ETMPSIZE
    assert f(one, 1, P, P, P, 2, 1000, 4100, 16, 0, 1.0, 1, P, big, None, 1, None) == ENOKERNEL
    assert f(two, 2, P, P, P, 2, 1000, 4096, 12, 0, 1.0, 1, P, big, None, 1, None) == ENOKERNEL
    assert f(two, 2, P, P, P, 2, 1000, 4096, 64, 0, 1.0, 2, P, big, None, 1, None) == EINVAL and "accumulate" in _err()
    assert f(two, 2, P, P, P, 0, 1000, 4096, 64, 0, 1.0, 0, P, 4 * big, None, 1, None) == OK  # a larger scratch is accepted
    # a row-tile plan: records must be aligned, the height bound at least 1
    bad = _native.SgmvTiles(P + 4, 3, 48)
    assert f(two, 2, P, P, P, 2, 1000, 4096, 64, 0, 1.0, 1, P, big, ctypes.byref(bad), 1, None) == EINVAL and "tile plan" in _err()
    bad = _native.SgmvTiles(P, 3, 0)
    assert f(two, 2, P, P, P, 2, 1000, 4096, 64, 0, 1.0, 1, P, big, ctypes.byref(bad), 1, None) == EINVAL
    empty = _native.SgmvTiles(P, 0, 16)  # a plan without tiles: nothing to do
    assert f(two, 2, P, P, P, 2, 1000, 4096, 64, 0, 1.0, 1, P, big, ctypes.byref(empty), 1, None) == OK


def _shrink_groups(rank, num_problems, num_groups, tile_rows=16, num_tiles=40):
    problems = (_native.SgmvShrinkProblem * num_problems)(*[_native.SgmvShrinkProblem(P, P)] * num_problems)
    tiles = _native.SgmvTiles(P, num_tiles, tile_rows)
    group = _native.SgmvShrinkGroup(problems, num_problems, rank, P, P, 2, ctypes.addressof(tiles))
    return (_native.SgmvShrinkGroup * num_groups)(*[group] * num_groups), (problems, tiles)


@pytest.mark.parametrize("rank", [10, 12, 18, 30, 4, 136])
@pytest.mark.parametrize("num_problems", [2, 4])
def test_sgmv_shrink_groups_refuses_the_ranks_that_shrink_multi_refuses(rank, num_problems):
    """A rank that is no multiple of 8 is refused whatever the summed rank of the group (two problems of rank 12 and four
    of rank 10 or 18 have a sum that is one): a store of four columns would cross into the next row of v."""
    f = _native.lib().lorax_sgmv_shrink_groups
    for num_groups in (1, 2):
        groups, _keep = _shrink_groups(rank, num_problems, num_groups)
        assert f(groups, num_groups, P, 1000, 4096, 0, 1.0, 0, P, 8 * 1024 * 1024, 1, None) == ENOKERNEL
        assert "No suitable kernel" in _err()


@pytest.mark.parametrize("jobs,tokens,h_in,together", [
    # one slice per projection: whatever the batch and the mix of ranks 8 and 16
    ([(8, 4096, 65535), (16, 2048, 3)], 60000, 4096, True),
    ([(8, 4096, 1)], 1, 8192, True), ([(8, 4096, 1)], 1, 8200, False), ([(16, 2048, 1)], 1, 4104, False),  # the slab
    ([(32, 512, 1)], 1, 1024, False), ([(8, 512, 1), (24, 512, 1)], 1, 1024, False), ([], 1, 1024, False),
    # wide projections: few records, one rank
    ([(8, 14336, 64)], 256, 4096, True), ([(8, 14336, 65)], 65, 4096, False),
    ([(16, 2056, 16)], 64, 4096, True), ([(16, 2056, 17)], 17, 4096, False),
    ([(8, 4104, 1), (16, 512, 1)], 1, 1024, False),
    ([(16, 4096, 16), (16, 1024, 17)], 17, 4096, False), ([(8, 8192, 3), (8, 1024, 65)], 65, 4096, False),  # a narrow one's count too
    ([(8, 16384, 1)], 1, 1024, True), ([(8, 16392, 1)], 1, 1024, False), ([(8, 32000, 1), (8, 64, 1)], 1, 1024, False),
    # more slices than CUs: about one token per record and at most half the slab
    ([(8, 14336, 32)] * 2, 128, 8192, True), ([(8, 14336, 33)] * 2, 65, 4096, False), ([(8, 14336, 64)] * 2, 64, 4096, True),
    ([(8, 14336, 64)] * 2, 65, 4096, False), ([(8, 14336, 64)] * 2, 64, 4104, False),
    ([(8, 8192, 64), (8, 1024, 64), (8, 1024, 64)], 256, 8192, True), ([(16, 14336, 16)] * 2, 64, 4096, True),
    ([(16, 14336, 16)] * 3, 64, 2048, False), ([(16, 14336, 16)] * 3, 16, 2048, True),
])
def test_decode_route(jobs, tokens, h_in, together):
    """lorax_decode_in_one_launch at its bounds: the rule that the native layer call, the general path of the layers and the
    stacked-weight operators share."""
    assert _native.decode_in_one_launch(jobs, tokens, h_in) is together


def test_single_launch_rules_for_one_projection():
    for rank, width in ((8, 4096), (16, 2048)):
        assert _native.bgmv_lora_fits(rank, 4096, width) and not _native.bgmv_lora_fits(rank, 4096, width + 8)
    assert not _native.bgmv_lora_fits(32, 1024, 64) and not _native.bgmv_lora_fits(16, 8192, 64)
    for rank, rows in ((8, 512), (16, 128)):
        assert _native.sgmv_lora_fits(rank, 4096, rows, 16384) and not _native.sgmv_lora_fits(rank, 4096, rows + 1)
        assert not _native.sgmv_lora_fits(rank, 4096, 1, 16392) and not _native.sgmv_lora_fits(rank, 65536 // rank + 8, 1)
    assert not _native.sgmv_lora_fits(32, 1024, 1)
    # the short batches that the Python paths know are the C rule's
    from lorax_amd.sgmv import resident_shrink_applies

    short = _native.SGMV_LORA_MAX_TOKENS
    assert _native.sgmv_lora_fits(8, 1024, short) and not _native.sgmv_lora_fits(8, 1024, short + 1)
    assert resident_shrink_applies(24, 200, short) and not resident_shrink_applies(24, 200, short + 1)


@pytest.mark.parametrize("ranks,problems,tile_rows,rows,h_in,one_launch", [
    ((16, 64), 2, 16, 1000, 4096, True), ((8, 128), 1, 32, 513, 256, True), ((16, 32), 4, 16, 1000, 1024, True),
    ((16, 64), 2, 16, 512, 4096, False), ((16, 64), 2, 48, 1000, 4096, False), ((16, 64), 2, 16, 1000, 4104, False),
    ((16, 64), 4, 16, 1000, 4096, False), ((16, 12), 2, 16, 1000, 4096, False), ((16,), 2, 16, 1000, 4096, False),
])
def test_sgmv_shrink_groups_route(ranks, problems, tile_rows, rows, h_in, one_launch):
    f = _native.lib().lorax_sgmv_shrink_groups_parts
    made = [_shrink_groups(r, problems, 1, tile_rows) for r in ranks]
    groups = (_native.SgmvShrinkGroup * len(ranks))(*[g[0] for g, _ in made])
    big = 8 * 1024 * 1024
    assert (f(groups, len(ranks), P, rows, h_in, 0, 0, P, big, 1) > 0) is one_launch
    for layer, accumulate, tmp, size, dtype in ((-1, 0, P, big, 1), (0, 2, P, big, 1), (0, 0, None, big, 1), (0, 0, P + 4, big, 1),
                                                (0, 0, P, big - 1, 1), (0, 0, P, big, 2)):
        assert f(groups, len(ranks), P, rows, h_in, layer, accumulate, tmp, size, dtype) == 0
    # parts only as far as their fp32 sums fit the scratch: 40 tiles of rank 128 take 320 KB each
    made = [_shrink_groups(64, 2, 1, 16) for _ in range(16)]
    groups = (_native.SgmvShrinkGroup * 16)(*[g[0] for g, _ in made])
    for count in range(2, 17):
        assert 1 <= f(groups, count, P, 12000, 128 * 67, 0, 0, P, big, 1) <= max(1, (big - 65536) // (count * 40 * 16 * 128 * 4))


def test_sgmv_shrink_groups_parts_of_every_group():
    """lorax_sgmv_shrink_groups_parts_of: at least one part of at least eight stages each, at most eight of them, their fp32 sums
    in the first 8 MiB (less the counters), and no part for a group without tiles."""
    import random

    average, each = (getattr(_native.lib(), "lorax_sgmv_shrink_groups_parts" + suffix) for suffix in ("", "_of"))
    rng, big, seen = random.Random(5), 8 * 1024 * 1024, set()
    for _ in range(2000):
        n, h_in = rng.randint(2, 16), 128 * rng.choice([3, 16, 32, 64, 67, 112, 224])
        shapes = [(rng.choice([8, 16, 24, 32, 64]), rng.randint(1, 2), rng.choice([0, 1, 9, 40, 90, 170]), rng.choice([16, 32]))
                  for _ in range(n)]
        made = [_shrink_groups(r, count, 1, height, tiles) for r, count, tiles, height in shapes]
        groups = (_native.SgmvShrinkGroup * n)(*[g[0] for g, _ in made])
        parts = (ctypes.c_int32 * n)(*[-1] * n)
        args = (groups, n, P, 12000, h_in, 0, 0, P, big, 1)
        k = average(*args)
        assert each(*args, parts) == k
        if k == 0:
            assert list(parts) == [-1] * n
            continue
        sums = 0
        for (r, count, tiles, height), got in zip(shapes, parts):
            assert got == 0 if tiles == 0 else 1 <= got <= max(1, min(8, h_in // 128 // 8))
            sums += got * tiles * height * ((r * count + 15) // 16 * 16) * 4 if got > 1 else 0
        assert sums <= big - 65536 and (k > 1 or max(parts) == 1)
        seen.add((k > 1, 1 in parts, len(set(parts) - {0}) > 1))
    assert (True, True, True) in seen and (True, False, True) in seen


def test_sgmv_lora_multi_validation():
    f = _native.lib().lorax_sgmv_lora_multi
    one = (_native.SgmvLoraProblem * 1)(_native.SgmvLoraProblem(P, P, P, 0, 4096, 4096))
    assert f(one, 0, P, P, P, 2, 64, 4096, 16, 0, 1.0, 1, None) == EINVAL and "num_problems" in _err()
    assert f(one, 1, P, P, P, 0, 64, 4096, 16, 0, 1.0, 1, None) == OK  # no segments
    assert f(one, 1, P, P, None, 2, 64, 4096, 16, 0, 1.0, 1, None) == EINVAL and "null" in _err()
    assert f(one, 1, P, P, P, 2, 64, 4096, 32, 0, 1.0, 1, None) == ENOKERNEL  # rank
    assert f(one, 1, P, P, P, 2, 513, 4096, 16, 0, 1.0, 1, None) == ENOKERNEL  # too many rows
    assert f(one, 1, P, P, P, 2, 64, 4096, 16, -1, 1.0, 1, None) == EINVAL
    narrow = (_native.SgmvLoraProblem * 1)(_native.SgmvLoraProblem(P, P, P, 8, 4096, 4096))
    assert f(narrow, 1, P, P, P, 2, 64, 4096, 16, 0, 1.0, 1, None) == EINVAL and "y_offset" in _err()
    no_b = (_native.SgmvLoraProblem * 1)(_native.SgmvLoraProblem(P, P, None, 0, 4096, 4096))
    assert f(no_b, 1, P, P, P, 2, 64, 4096, 16, 0, 1.0, 1, None) == EINVAL


def test_sgmv_expand_validation():
    f = _native.lib().lorax_sgmv_expand
    for layout in (_native.B_RH, _native.B_HR):
        assert f(P, P, P, P, P, 2, 16, 16, 4096, layout, 0, 4096, 0, 1, P, 121, 1, None) == ETMPSIZE
        assert f(P, P, P, P, P, 0, 16, 16, 4096, layout, 0, 4096, 0, 1, None, 0, 1, None) == OK
        for r, h in [(4, 4096), (136, 4096), (16, 4100)]:
            assert f(P, P, P, P, P, 2, 16, r, h, layout, 0, h, 0, 1, P, 120, 1, None) == ENOKERNEL, (r, h)
        assert f(P, P, P, P, P, 2, 16, 16, 4096, layout, 4, 8192, 0, 1, P, 120, 1, None) == EINVAL  # unaligned window
        assert f(P, P, P, P, P, 2, 16, 16, 4096, layout, 4096, 4096, 0, 1, P, 120, 1, None) == EINVAL  # too wide
        assert f(P, P, P, P, P, 2, 16, 16, 4096, layout, 0, 1 << 24, 0, 1, P, 120, 1, None) == EINVAL  # row pitch
        assert "2^24" in _err()
    assert f(P, P, P, P, P, 2, 16, 16, 4096, 2, 0, 4096, 0, 1, P, 120, 1, None) == EINVAL  # unknown layout


@pytest.mark.parametrize("num_segments,num_tokens", [(-1, 0), (-1, 16), (2, -1), (0, -1)])
def test_sgmv_expand_refuses_negative_sizes_whatever_else_is_empty(num_segments, num_tokens):
    lib = _native.lib()
    for layout in (_native.B_RH, _native.B_HR):
        assert lib.lorax_sgmv_expand(P, P, P, P, P, num_segments, num_tokens, 16, 4096, layout, 0, 4096, 0, 1, P,
                                     60 * max(num_segments, 0), 1, None) == EINVAL, layout
    assert lib.lorax_sgmv_expand_planned(P, P, P, P, P, num_segments, num_tokens, 16, 4096, 0, 4096, 0, 1, None, 1, None) == EINVAL
    one = (_native.SgmvExpandProblem * 1)(_native.SgmvExpandProblem(P, P, P, P, P, num_segments, 16, 4096, 0, 4096, None))
    assert lib.lorax_sgmv_expand_multi(one, 1, num_tokens, 0, 1, 1, None) == EINVAL and "negative" in _err()


def test_sgmv_expand_planned_validation():
    f = _native.lib().lorax_sgmv_expand_planned
    assert f(P, P, P, P, P, 0, 16, 16, 4096, 0, 4096, 0, 1, None, 1, None) == OK  # no segments
    assert f(P, P, P, P, P, 2, 16, 12, 4096, 0, 4096, 0, 1, None, 1, None) == ENOKERNEL
    assert f(P, P, P, P, None, 2, 16, 16, 4096, 0, 4096, 0, 1, None, 1, None) == EINVAL
    bad = _native.SgmvTiles(P, -1, 256)
    assert f(P, P, P, P, P, 2, 16, 16, 4096, 0, 4096, 0, 1, ctypes.byref(bad), 1, None) == EINVAL and "tile plan" in _err()
    empty = _native.SgmvTiles(P, 0, 256)
    assert f(P, P, P, P, P, 2, 16, 16, 4096, 0, 4096, 0, 1, ctypes.byref(empty), 1, None) == OK


def test_stacked_update_validation():
    f = _native.lib().lorax_stacked_update
    pack = lambda *slices: b"".join(_native._STACKED_SLICES[1].pack(*s) for s in slices)
    one = pack((P, P, 0, 16, 256))
    call = lambda s, n, rows=4, records=2, v_bytes=1 << 20, plan=P: f(s, n, plan, records, P, 256, P, rows, 512, P, v_bytes, 1, 0, None)
    assert call(one, 0) == call(one, 1, rows=0) == call(one, 1, records=0) == OK  # nothing to do
    # no row to route: nothing is launched, but a window beyond y, a width the kernels do not take and a misaligned stack are refused
    assert call(pack((P, P, 8, 16, 256)), 1, records=0) == EINVAL and "do not hold" in _err()
    assert call(pack((P, P, 0, 16, 252)), 1, records=0) == ENOKERNEL
    assert call(pack((P, P + 2, 0, 16, 256)), 1, records=0) == EINVAL and "aligned" in _err()
    assert call(one, 17) == call(one, -1) == call(one, 1, rows=-1) == call(one, 1, records=-1) == EINVAL and "out of range" in _err()
    assert call(one, 1, plan=None) == EINVAL and "null" in _err()
    for rank in (4, 12, 136):
        assert call(pack((P, P, 0, rank, 256)), 1) == _native.EROUTE
    assert call(pack((0, P, 0, 16, 256)), 1) == _native.EROUTE
    assert call(pack((P, P, 0, 16, 256), (P, P, 256, 8, 256)), 2, v_bytes=4 * 24 * 2 - 1) == 5 and "workspace" in _err()


def test_plan_tiles_cuts_every_row_once():
    """lorax_sgmv_plan_tiles (host only): every row of every non-empty segment in exactly one tile, tiles inside
    their segment and no higher than the bound, numbered inside the segment; empty and negative segments get none."""
    starts = [5, 100, 100, -1, 400, 2000]
    ends = [47, 100, 90, -1, 1500, 2003]
    T = 2500
    for kind, limit in ((_native.TILES_SHRINK, 64), (_native.TILES_EXPAND, 256 + 32 + 16), (_native.TILES_EXPAND_BATCH, 256 + 32 + 16)):
        records, tile_rows = _native.plan_tiles(starts, ends, T, kind)
        assert tile_rows <= limit
        covered = {}
        last_index = {}
        for seg, row0, row_end, index in records.tolist():
            assert starts[seg] <= row0 < row_end <= ends[seg] and row_end - row0 <= tile_rows
            assert index == last_index.get(seg, -1) + 1
            last_index[seg] = index
            for row in range(row0, row_end):
                assert row not in covered
                covered[row] = seg
        want = {row: seg for seg, (s, e) in enumerate(zip(starts, ends)) for row in range(max(s, 0), min(e, T))}
        assert covered == want
    # bounds beyond the batch are clamped; a table without rows gives an empty plan
    records, _ = _native.plan_tiles([10], [100], 50, _native.TILES_SHRINK)
    assert records[:, 2].max() == 50
    records, _ = _native.plan_tiles([3, -1], [3, -1], 50, _native.TILES_EXPAND)
    assert records.shape == (0, 4)
    # a thousand rows in ten segments: low tiles (the launch also cuts the hidden dimension); a long batch: 64 rows
    records, tile_rows = _native.plan_tiles(list(range(0, 1000, 100)), list(range(100, 1100, 100)), 1000, _native.TILES_SHRINK)
    assert tile_rows == 16 and len(records) == 70
    records, tile_rows = _native.plan_tiles([0], [40000], 40000, _native.TILES_SHRINK)
    assert tile_rows == 64 and len(records) == 625
    # tiles are not lowered below a quarter of the rank: 4096 rows at rank 128 stay at 32 rows (128 tiles), at rank
    # 64 they go down to 16 (256 tiles, one per CU)
    assert _native.plan_tiles([0], [4096], 4096, _native.TILES_SHRINK, 128)[1] == 32
    assert _native.plan_tiles([0], [4096], 4096, _native.TILES_SHRINK, 64)[1] == 16


def test_shrink_summed_rank_looks_at_the_whole_call():
    """lorax_shrink_summed_rank: 64 only where every group of the call can be in one launch, several are, and none is higher."""
    from types import SimpleNamespace

    def rule(*groups, rows=2000, h_in=4096):
        return _native.shrink_summed_rank([(r, n, SimpleNamespace(num_tiles=t, tile_rows=h) if t else None) for r, n, t, h in groups],
                                          rows, h_in)

    assert rule((64, 3, 120, 16)) == rule((32, 3, 60, 16), (64, 3, 60, 32)) == rule((8, 3, 9, 16), (16, 3, 9, 16)) == 64
    assert rule((32, 3, 60, 16)) == rule((64, 2, 100, 16)) == 128            # one group of up to 128
    assert rule((32, 3, 60, 16), (64, 3, 60, 48)) == 128                     # another group's tiles are too high ...
    assert rule((32, 3, 60, 16), (64, 3, 0, 0)) == 128                       # ... or it has no plan
    assert rule((32, 3, 60, 16), (128, 3, 60, 32)) == rule((64, 3, 60, 16), (72, 3, 60, 32)) == 128
    assert rule((64, 3, 120, 16), rows=512) == rule((64, 3, 120, 16), h_in=2752) == rule() == 128
    assert rule(*[(40 + 8 * (i % 4), 4, 20, 16) for i in range(4)]) == 64    # 16 groups ...
    assert rule(*[(40 + 8 * (i % 4), 4, 20, 16) for i in range(5)]) == 128   # ... and more than one call takes


def test_expand_tile_counts_of_smaller_batches():
    """What a caller that sized its records, or captured a launch, for its largest batch relies on: with LORAX_TILES_EXPAND
    shorter segments never make more records; plans for one batch stay below the bound that the header names."""
    import random

    def count(lens, kind):
        bounds = [sum(lens[:i]) for i in range(len(lens) + 1)]
        return len(_native.plan_tiles(bounds[:-1], bounds[1:], bounds[-1], kind)[0])

    most = 0
    for n in range(4500):
        now = count([n], _native.TILES_EXPAND)
        assert most <= now <= n // 256 + 1
        most = now
    rng = random.Random(3)
    for _ in range(400):
        lens = [rng.choice([0, 1, 15, 64, 65, 200, 256, 289, 700, 1025, 2100]) for _ in range(rng.randrange(1, 12))]
        shorter = [rng.randint(0, n) for n in lens]
        assert count(shorter, _native.TILES_EXPAND) <= count(lens, _native.TILES_EXPAND) <= sum(lens) // 256 + len(lens)
        for batch in (lens, shorter):
            bound = max(16, sum(batch) // 256) + sum(n > 0 for n in batch)
            assert count(batch, _native.TILES_EXPAND_BATCH) <= bound
    assert count([1024], _native.TILES_EXPAND_BATCH) == 16 and count([1025], _native.TILES_EXPAND_BATCH) == 12


def test_python_binding_rejects_cpu_tensors():
    import torch

    y = torch.zeros(2, 8, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        _native.dispatch_bgmv(y, y, torch.zeros(1, dtype=torch.int64), torch.zeros(2, dtype=torch.int64), 0, 1.0)
