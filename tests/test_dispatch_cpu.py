"""Which kernel takes dk and dv, by sizes: the tests that run on the GPU name the form that they are written for, and this file
holds them to it, so that a rule that moves does not leave them green on another kernel."""
import ctypes

import pytest
import torch

from flash_mi355 import _cabi
from tests._forms import dkdv_form

bf16, fp16, f32 = torch.bfloat16, torch.float16, torch.float32


def test_invalid_parameters_have_no_form():
    assert _cabi.lib().fa_bwd_form(None, 1) == -1
    p = _cabi.FaParams()
    assert _cabi.lib().fa_bwd_form(ctypes.byref(p), 1) == -2 and _cabi.lib().fa_bwd_form(ctypes.byref(p), 0) == -2


@pytest.mark.parametrize("args,kw,form", [
    ((1, 2, 2, 300, 300, 32, bf16, True), {}, ("keys", False)), ((1, 1, 1, 300, 300, 64, bf16, True), {}, ("small", True)),
    ((1, 32, 32, 16384, 16384, 128, bf16, True), {}, ("pipe", False)), ((1, 32, 32, 16384, 16384, 128, bf16, True), {"window": 1024}, ("keys", False)),
    ((1, 32, 32, 16384, 16384, 128, bf16, True), {"kind": "doc"}, ("keys", False)), ((8, 8, 8, 1024, 8192, 128, fp16, True), {"kind": "doc"}, ("cols", False)),
    ((1, 8, 8, 1088, 1088, 128, bf16, True), {"kind": "block"}, ("keys", True)), ((1, 8, 8, 1088, 1088, 128, bf16, True), {"whole": False}, ("keys", False)),
    ((2, 32, 8, 1100, 1100, 64, bf16, True), {}, ("rows", True)), ((2, 4, 4, 512, 512, 64, f32, True), {"kind": "doc"}, ("fp32", True)),
    # (the diagnostic flag of the pair wait keeps fa_bwd_dkdv off the form without pairs)
    ((1, 8, 1, 520, 520, 128, bf16, True), {"whole": False}, ("small", False)), ((1, 8, 1, 520, 520, 128, bf16, True), {"whole": False, "no_pair_wait": True}, ("pipe", False)),
])
def test_forms(args, kw, form):
    assert dkdv_form(*args, **kw) == form


@pytest.mark.parametrize("args,kw", [
    ((4, 8, 8, 115, 429, 64, bf16, False), {}), ((1, 64, 64, 205, 205, 64, fp16, True), {"kind": "doc"}), ((1, 16, 16, 186, 989, 64, bf16, True), {"kind": "block"}),
    ((2, 4, 4, 1711, 1870, 64, bf16, True), {"window": 100}), ((1, 4, 4, 425, 3031, 64, fp16, True), {}), ((3, 2, 2, 815, 2624, 64, fp16, True), {}),
    ((2, 4, 4, 125, 1871, 64, bf16, True), {"prefix": 535}), ((1, 8, 8, 118, 1892, 64, bf16, True), {}),
])
def test_the_small_form_stops_where_its_workgroups_share_cus(args, kw):
    """D = 64, 340 to 512 workgroups of 32 keys with short chains of rows or equal ones: 1.1 to 1.4 times the time of the form with 128 keys to a workgroup."""
    assert dkdv_form(*args, **kw)[0] != "small"


@pytest.mark.parametrize("args,kw", [((1, 8, 8, 1252, 1252, 64, bf16, True), {}), ((3, 2, 2, 1780, 1780, 64, bf16, True), {}), ((4, 64, 8, 470, 470, 64, bf16, True), {}),
                                     ((1, 64, 8, 1856, 1856, 64, fp16, True), {"window": 62}), ((1, 8, 8, 96, 1925, 64, fp16, True), {"window": 51}), ((1, 4, 4, 2591, 3124, 64, bf16, True), {"kind": "doc"}),
                                     ((1, 16, 2, 2196, 2196, 64, fp16, True), {"kind": "packed", "nseq": 35}), ((4, 64, 8, 147, 147, 128, fp16, False), {})])
def test_long_chains_keep_the_small_form(args, kw):
    """... up to two workgroups of 32 keys to a CU: 1.2 to 1.8 times faster than the other forms."""
    assert dkdv_form(*args, **kw)[0] == "small"


@pytest.mark.parametrize("args,kw,form", [
    *(((B, H, Hk, M, N, 128, bf16, True), kw, ("small", True)) for B, H, Hk, M, N, kw in (
        (1, 16, 2, 2374, 2374, {}), (1, 8, 1, 5156, 5156, {}), (1, 32, 4, 1127, 1181, {}), (2, 8, 1, 2623, 2623, {}), (3, 8, 1, 1742, 1742, {}), (1, 32, 4, 1236, 1236, {"window": 188}), (3, 8, 1, 1786, 1786, {"prefix": 320}))),
    *(((B, H, H, M, N, 128, bf16, True), {}, ("keys", True)) for B, H, M, N in ((2, 8, 3844, 4546), (1, 16, 3452, 4997), (4, 4, 3723, 5483), (3, 4, 5127, 6263), (1, 5, 12000, 14982))),
    ((1, 16, 2, 2417, 2417, 128, bf16, True), {"whole": False}, ("small", False)),
])
def test_query_tiles_of_64_rows_do_not_move_the_backwards_form(args, kw, form):
    """Causal problems of one to two workgroups of 128 rows to a CU, whose dq may take 64-row tiles: counted in those, the backward took 1.2 to 1.3 times as long
    in the form it moved to."""
    assert dkdv_form(*args, **kw) == form


@pytest.mark.parametrize("args", [(1, 32, 8, 151, 614, 128, bf16, False), (2, 64, 16, 38, 149, 128, bf16, False)])
def test_the_small_form_stops_earlier_without_a_mask(args):
    """D = 128, several query heads to a key head, 160 workgroups of 32 keys, chains of 8 and 20 blocks: 1.17 to 1.26 times the time of the other form."""
    assert dkdv_form(*args)[0] == "keys"


@pytest.mark.parametrize("args,kw", [
    ((1, 16, 16, 2425, 2425, 64, bf16, True), {}), ((1, 16, 16, 2021, 2021, 64, fp16, False), {}), ((2, 8, 8, 2854, 2854, 64, bf16, True), {"prefix": 100}),
    ((1, 16, 16, 2138, 2225, 64, fp16, True), {"kind": "block"}), ((3, 16, 8, 2474, 2474, 64, bf16, False), {}),
])
def test_rows_are_shared_only_where_cus_are_free(args, kw):
    """D = 64, 256 to 480 workgroups of 128 keys: 1.05 to 1.28 times the time of the form whose waves own their keys."""
    assert dkdv_form(*args, **kw)[0] == "keys"


@pytest.mark.parametrize("args,kw", [
    ((1, 16, 16, 2500, 2500, 64, bf16, False), {}), ((1, 6, 6, 6400, 6400, 64, bf16, True), {}), ((2, 64, 8, 3000, 3000, 64, fp16, True), {"window": 900}),
    ((2, 4, 4, 1789, 6128, 64, bf16, True), {"window": 1156}), ((1, 16, 16, 2011, 2011, 64, bf16, True), {"kind": "block"}), ((1, 64, 8, 1302, 5000, 64, bf16, True), {"kind": "block"}),
])
def test_long_chains_share_their_rows_beyond_a_workgroup_to_a_cu(args, kw):
    """... up to 512 workgroups (1024 with a block map), where every one of them walks many tiles."""
    assert dkdv_form(*args, **kw)[0] == "rows"


@pytest.mark.parametrize("args,kw", [
    ((8, 32, 32, 32, 32, 64, f32, True), {"kind": "doc"}), ((4, 64, 64, 25, 25, 128, f32, True), {"kind": "doc"}), ((4, 64, 64, 92, 274, 128, f32, True), {"kind": "doc"}),
    ((8, 32, 32, 98, 98, 128, f32, False), {}), ((2, 64, 64, 209, 209, 128, f32, False), {}),
])
def test_short_fp32_rows_are_not_cut_among_eight_waves(args, kw):
    """Many short rows: 1.2 to 2.5 times the time in dq where eight waves shared 16 rows, most of the workgroups of them empty with ids."""
    form, dq, _ = dkdv_form(*args, **kw)
    assert form == "fp32" and dq != 0


def test_fp32_shapes_without_a_mask_follow_the_rounds_of_workgroups():
    """D = 128: 640 workgroups of 32 rows are three rounds of one to a CU or two of two, which take 1.9 times as long; 512 are two or one."""
    assert dkdv_form(1, 40, 40, 490, 490, 128, f32, False) == ("fp32", 1, 1) and dkdv_form(1, 32, 32, 500, 500, 128, f32, False) == ("fp32", 2, 2)
    assert dkdv_form(4, 1, 1, 1754, 1754, 64, f32, False)[1] is not True   # (440 workgroups of 32: two launches)
    for args in ((2, 4, 1, 1219, 1219, 128), (1, 2, 2, 4240, 2436, 128), (3, 1, 1, 2419, 2419, 16)):   # (dk/dv's chains longer or shorter than dq's: one)
        assert dkdv_form(*args, f32, False) == ("fp32", True)


def test_fp32_backward_in_one_launch_up_to_two_workgroups_to_a_cu():
    """... under a causal mask, and without one where the chains are short; padded places of ids count against eight to a CU."""
    assert dkdv_form(8, 8, 8, 128, 128, 64, f32, True) == ("fp32", True) and dkdv_form(4, 8, 8, 250, 250, 64, f32, False) == ("fp32", True)
    assert dkdv_form(8, 8, 8, 129, 129, 64, f32, True)[1] is not True and dkdv_form(8, 32, 32, 29, 29, 64, f32, True, kind="doc")[1] is not True


def _kind(k):
    return k if k in ("doc", "heads", "qpos", "block") else "plain"


def _form(case, D, window, prefix, **kw):
    """(B, H, Hk, M, N, dtype, causal, kind) with a window or prefix of the given size where the kind says so"""
    B, H, Hk, M, N, dtype, causal, kind = case
    return dkdv_form(B, H, Hk, M, N, D, dtype, causal, _kind(kind), window=window if kind == "window" else 0, prefix=prefix if kind == "prefix" else 0, **kw)


def test_gpu_cases_reach_the_form_they_are_written_for():
    from tests import test_gpu_launch_forms as F, test_gpu_parity as P
    assert {_form(c, 64, 500, 270)[0] for c in F.ROWS_CASES} == {"rows"}
    assert {_form(c, 64, 500, 270)[1] for c in F.ROWS_CASES} == {True, False}
    assert {_form(c, 64, 500, 270)[0] for c in F.ROWS_BEYOND_CASES} == {"keys"}
    for lens in ([1000, 833, 961, 64, 1, 532, 990], [700, 0, 1211, 130]):
        assert dkdv_form(1, 32, 8, sum(lens), sum(lens), 64, bf16, True, "packed", nseq=len(lens))[0] == "rows"
    for B, H, Hk, M, N, D, causal, form in F.LAYOUT_CASES:
        assert dkdv_form(B, H, Hk, M, N, D, bf16, causal)[0] == form
    for B, H, Hk, M, N, dtype, causal, window, prefix in F.PIPE_CASES:
        assert dkdv_form(B, H, Hk, M, N, 128, dtype, causal, window=window, prefix=prefix, whole=False, no_pair_wait=True)[0] == "pipe"
    for i, (B, H, Hk, M, N, D, dtype, causal, kind) in enumerate(F.SMALL_BWD_CASES):   # (the second half: runs of key tiles next to the column form)
        assert _form((B, H, Hk, M, N, dtype, causal, kind), D, 37, 21)[0] == ("small" if i < 11 else "cols")
    alone = [{dkdv_form(B, H, Hk, M, N, D, dtype, causal, _kind(kind), window=170 if kind == "window" else 0, prefix=170 if kind == "prefix" else 0, whole=w)[0]
              for w in (True, False)} for B, H, Hk, M, N, D, dtype, causal, kind in F.SHARED_CASES]
    assert {"keys", "pipe"} in alone and {"rows"} in alone and {"keys"} in alone and {"small"} in alone
    unseen = {dkdv_form(1, H, H, M, N, D, bf16, True, _kind(kind), window=2000 if kind == "window" else 0, whole=w)[0] for D, H, M, N, kind in F.UNSEEN_CASES for w in (True, False)}
    assert unseen == {"keys", "rows", "small", "pipe", "cols"}
    for B, H, Hk, M, N, D, dtype, causal, doc in P.KEYS_CASES:
        assert dkdv_form(B, H, Hk, M, N, D, dtype, causal, "doc" if doc else "plain")[0] == "keys"
    for B, H, Hk, M, N, D, dtype, causal, window, _, _ in P.KEYS_BLOCK_CASES:
        assert dkdv_form(B, H, Hk, M, N, D, dtype, causal, "block", window=window)[0] == "keys"
    for B, H, Hk, M, N, D, dtype, doc, window, prefix in P.KEYS_BAND_CASES:
        assert dkdv_form(B, H, Hk, M, N, D, dtype, True, "doc" if doc else "plain", window=window, prefix=prefix)[0] == "keys"
    for B, H, Hk, M, N, D, dtype, causal, _, window in P.COLS_BIG_CASES:
        assert dkdv_form(B, H, Hk, M, N, D, dtype, causal, "doc", window=window)[0] == "cols"
    for B, H, Hk, M, N, causal, kw in ((1, 4, 2, 243, 1419, True, {"window": 876}), (2, 2, 1, 651, 617, False, {}), (2, 4, 2, 248, 1297, True, {"prefix": 530})):
        assert dkdv_form(B, H, Hk, M, N, 128, bf16, causal, "doc", **kw)[0] == "small"
        assert dkdv_form(6 * B, H, Hk, M, N, 128, bf16, causal, "doc", **kw)[0] in ("keys", "cols")   # (P crosses between the waves of a pair)
    shapes = [dkdv_form(B, H, Hk, M, N, D, f32, causal, _kind(kind), window=37 if kind == "window" else 0, prefix=21 if kind == "prefix" else 0)[1:]
              for B, H, Hk, M, N, D, causal, kind in F.FP32_SHAPE_CASES]
    assert shapes[:3] == [(0, 0)] * 3 and {s[0] for s in shapes} == {s[1] for s in shapes} == {0, 1, 2}
