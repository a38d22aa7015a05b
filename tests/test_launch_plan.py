"""The split counts the library tells against the ones it runs, on the CPU: fa2_launch_splits and
fa2_num_splits (include/fa2_fwd.h) and the native call's policy against the plan of the launch itself (fa2_ablate_plan: the
library's planning code, without a GPU call).
"""

import random

import pytest

from fa2 import _lib
from test_schedule import needs_ablate

WAVE_SPLIT = "fa2::attn_wave_split_kernel"


def _plan(*sizes, **kw):
    from ablation import launch_plan
    return launch_plan(*sizes, **kw)


def _launch_splits(B, h_q, h_kv, n_q, n_kv, D, num_splits, cus=256):
    return int(_lib.lib().fa2_launch_splits(B, h_q, h_kv, n_q, n_kv, D, 0, 128, 0, cus, num_splits))


def _ranges(plan, n_kv):
    """First and last key of every range of a launch."""
    per = plan["split_tiles"] * plan["keys"] or n_kv
    return [(x, min(x + per, n_kv)) for x in range(0, n_kv, per)]


def _calls(n, seed):
    rnd = random.Random(seed)
    for _ in range(n):
        h_kv, group = rnd.choice([1, 2, 4, 8, 16]), rnd.choice([1, 1, 2, 4, 5, 7, 8, 16, 56])
        yield (rnd.choice([1, 1, 2, 3, 8, 20]), h_kv * group, h_kv, rnd.choice([1, 1, 2, 7, 16, 40, 150, 700]),
               rnd.choice([1, 100, 129, 513, 1000, 1088, 1536, 2112, 3000, 4097, 8192, 16483, 32000, 40001]),
               rnd.choice([16, 32, 64, 128]))


@needs_ablate
@pytest.mark.parametrize("cus,xcds", [(256, 8), (304, 8), (96, 4)])
def test_launch_splits_is_the_count_that_runs(cus, xcds):
    """Over key counts that are no multiple of a tile and every num_splits: the count told is the
    count of the plan, passing it back makes the same ranges with its own workspace, and every range
    holds keys. A workspace of the requested count, and of the least count accepted."""
    lib = _lib.lib()
    seen = set()
    for sizes in _calls(500, cus):
        B, h_q, h_kv, n_q, n_kv, D = sizes
        for n in (2, 3, 5, 7, 8, 12, 16):
            told = _launch_splits(*sizes, n, cus)
            ws = lib.fa2_workspace_bytes(B, h_q, n_q, D, n)
            plan = _plan(*sizes, 0, False, num_splits=n, workspace_bytes=ws, cus=cus, xcds=xcds)
            assert told == plan["splits"], (sizes, n, told, plan)
            again = _plan(*sizes, 0, False, num_splits=told, cus=cus, xcds=xcds,
                          workspace_bytes=lib.fa2_workspace_bytes(B, h_q, n_q, D, told))
            assert again == plan and _launch_splits(*sizes, told, cus) == told, (sizes, n, plan, again)
            assert len(_ranges(plan, n_kv)) == told <= n
            seen.add((plan["kernel"], told))
            # the least workspace accepted holds the general kernel's ranges: no kernel runs more
            tiles = -(-n_kv // (128 if D == 16 else 64))
            least = -(-tiles // -(-tiles // n))
            if least > 1:
                tight = _plan(*sizes, 0, False, num_splits=n, cus=cus, xcds=xcds,
                              workspace_bytes=lib.fa2_workspace_bytes(B, h_q, n_q, D, least))
                assert tight == plan and plan["splits"] <= least
                with pytest.raises(RuntimeError, match="workspace"):
                    _plan(*sizes, 0, False, num_splits=n, cus=cus, xcds=xcds,
                          workspace_bytes=lib.fa2_workspace_bytes(B, h_q, n_q, D, least) - 256)
    assert len({k for k, _ in seen}) == 2 and {k for k, s in seen if s > 8} >= {WAVE_SPLIT}


@needs_ablate
@pytest.mark.parametrize("n_kv,n,want", [(1088, 16, 6), (1088, 8, 6), (1088, 6, 6), (2112, 16, 11),
                                         (2112, 12, 11), (4096, 16, 16), (4096, 3, 3), (31987, 16, 16)])
def test_wave_split_ranges(n_kv, n, want):
    """B1 H32/8 head_dim 128, one query, 32-key tiles: the count that leaves no range empty in them and
    in 64-key tiles (1088 keys are 34 or 17 of them), whatever larger count was asked for."""
    plan = _plan(1, 32, 8, 1, n_kv, 128, 1, False, num_splits=n,
                 workspace_bytes=_lib.lib().fa2_workspace_bytes(1, 32, 1, 128, n))
    assert plan["kernel"] == WAVE_SPLIT and plan["keys"] == 32 and plan["splits"] == want
    assert _launch_splits(1, 32, 8, 1, n_kv, 128, n) == want


@needs_ablate
def test_default_count_covers_what_the_launch_runs():
    """fa2_num_splits: the workspace of its count is accepted, and a larger one changes nothing."""
    lib = _lib.lib()
    for sizes in _calls(600, 5):
        B, h_q, h_kv, n_q, n_kv, D = sizes
        n = _lib.num_splits(*sizes, False, 128, 0, 256)
        ws = lib.fa2_workspace_bytes(B, h_q, n_q, D, n)
        plan = _plan(*sizes, 0, False, num_splits=n, workspace_bytes=ws)
        assert plan["splits"] <= n
        if plan["kernel"] == WAVE_SPLIT:
            more = _plan(*sizes, 0, False, num_splits=16,
                         workspace_bytes=lib.fa2_workspace_bytes(B, h_q, n_q, D, 16))
            assert more == plan, (sizes, plan, more)


@needs_ablate
def test_native_call_plans_attentions_launch():
    """The native call's packing, splits and workspace (fa2/_torch_call.so) give the launch that
    attention()'s Python gives with fa2_num_splits's count, also where the key-norm table pays and the
    wave-split kernel would take fewer splits (B1 H56/1, 150 queries of 32768 keys in bf16)."""
    from fa2._torch_call import policy
    from fa2.kernel import should_pack_gqa

    lib = _lib.lib()
    calls = list(_calls(1500, 7)) + [(1, g, 1, n_q, n_kv, D) for g in (48, 56, 60) for D in (64, 128)
                                     for n_q in (130, 150, 170) for n_kv in (8192, 32768, 65536)]
    tables = 0
    for sizes in calls:
        B, h_q, h_kv, n_q, n_kv, D = sizes
        for dtype in (0, 1):
            for causal in (False, True) if n_q == n_kv else (False,):
                n = 1 if causal else _lib.num_splits(*sizes, causal, 128, 0, 256)
                ws = lib.fa2_workspace_bytes_for(*sizes, dtype, int(causal), n)
                pack = h_q // h_kv if should_pack_gqa(n_q, h_q // h_kv, 128) else 1
                want = _plan(*sizes, dtype, causal, pack=pack, num_splits=n, workspace_bytes=ws)
                got_pack, got_n, got_ws = policy(*sizes, dtype, int(causal), 256)
                got = _plan(*sizes, dtype, causal, pack=got_pack, num_splits=got_n, workspace_bytes=got_ws)
                assert got == want and got_pack == pack and got_ws <= ws, (sizes, dtype, want, got)
                tables += want["key_table"] and n > _launch_splits(*sizes, n)
    assert tables >= 3
    assert policy(1, 56, 1, 150, 32768, 128, 1, 0, 256)[1] == 4


# H16 on 256 CUs: batch and length, and whether 256-row programs pay. At head_dim 32 the launch lasts as
# long as the CU with the most programs: 8 x 1024 is 2 per CU, 10 x 1024 2.5 (3 for 5 of 128 rows), 12 3,
# 14 3.5 (4 for 7), 15 3.75, 18 4.5 (5 for 9), 28 7, 22 5.5 (6 for 11), 25 6.25 (7 for 13). At 64 it is
# the last round of two per CU that matters. Rows past the last (3186) and short key ranges never pay.
@needs_ablate
@pytest.mark.parametrize("D,B,n,n_kv,wide", [
    (32, 8, 1024, 1024, False), (32, 10, 1024, 1024, False), (32, 12, 1024, 1024, True),
    (32, 14, 1024, 1024, False), (32, 15, 1024, 1024, True), (32, 18, 1024, 1024, False),
    (32, 22, 1024, 1024, False), (32, 25, 1024, 1024, True), (32, 28, 1024, 1024, True),
    (32, 12, 1024, 1000, False), (32, 12, 3186, 3186, False), (64, 8, 1024, 1024, True),
    (64, 9, 1024, 1024, False), (64, 14, 1024, 1024, True), (64, 25, 1024, 1024, True),
    (64, 12, 1024, 1000, False), (64, 12, 3186, 3186, False), (128, 12, 1024, 1024, False)])
def test_wide_kernel_where_it_pays(D, B, n, n_kv, wide):
    for dtype in (0, 1):
        plan = _plan(B, 16, 16, n, n_kv, D, dtype, False)
        assert (plan["kernel"] == "fa2::attn_wide_kernel") == wide, plan
        assert not wide or plan["rows"] == 256


def _kernel(B, h_q, h_kv, n_q, n_kv, D, causal=False):
    """The kernel of the default call (fp16: no key-norm table at these sizes), rows per workgroup."""
    n = 1 if causal else _lib.num_splits(B, h_q, h_kv, n_q, n_kv, D, causal, 128, 0, 256)
    plan = _plan(B, h_q, h_kv, n_q, n_kv, D, 0, causal, num_splits=n,
                 workspace_bytes=_lib.lib().fa2_workspace_bytes(B, h_q, n_q, D, n))
    return plan["rows"] if plan["kernel"] == WAVE_SPLIT else 0


# Full calls on both sides of the short-key line: rows per wave-split workgroup, 0 for the general kernel
@needs_ablate
@pytest.mark.parametrize("shape,rows", [
    ((6, 16, 16, 67, 150, 64), 0), ((9, 16, 8, 60, 320, 64), 0), ((3, 8, 2, 184, 370, 64), 32),
    ((7, 16, 8, 93, 204, 64), 0), ((37, 6, 2, 60, 206, 64), 32), ((11, 12, 12, 76, 310, 64), 0),
    ((36, 4, 4, 73, 464, 64), 64), ((9, 4, 4, 402, 239, 64), 64),
    ((49, 8, 2, 24, 250, 128), 0), ((21, 16, 8, 45, 250, 128), 0), ((24, 20, 4, 26, 209, 128), 0),
    ((12, 32, 8, 21, 407, 128), 0), ((14, 4, 4, 164, 467, 128), 32), ((30, 28, 4, 14, 372, 128), 64),
    ((24, 6, 2, 68, 140, 16), 0), ((10, 28, 4, 49, 214, 16), 32),
    ((3, 20, 4, 141, 244, 32), 0), ((8, 28, 4, 61, 302, 32), 0), ((3, 20, 4, 138, 381, 32), 32),
    ((8, 16, 1, 1, 162, 32), 0), ((33, 6, 2, 37, 129, 32), 0), ((45, 6, 2, 27, 177, 32), 0),
    ((41, 28, 4, 12, 179, 32), 32), ((53, 6, 2, 1, 186, 32), 32), ((8, 16, 1, 1, 194, 32), 32)])
def test_short_keys(shape, rows):
    assert _kernel(*shape) == rows


# Causal calls of 64-row workgroups with more than one per CU, on both sides of 192 keys
@needs_ablate
@pytest.mark.parametrize("shape,rows", [
    ((4, 32, 1, 165, 165, 32), 0), ((7, 16, 2, 184, 184, 32), 0), ((7, 16, 2, 193, 193, 32), 64),
    ((10, 12, 12, 192, 192, 64), 0), ((10, 12, 12, 193, 193, 64), 64), ((10, 12, 12, 184, 184, 16), 64),
    ((5, 16, 4, 184, 184, 32), 64), ((9, 16, 16, 191, 191, 64), 64), ((10, 20, 4, 133, 133, 32), 64),
    ((12, 16, 8, 134, 134, 64), 0), ((2, 8, 2, 184, 184, 32), 32)])
def test_short_causal_prompts(shape, rows):
    assert _kernel(*shape, causal=True) == rows


# More than 64 rows on at most half the CUs, one range of the wave-split kernel's against the general
# kernel's eight splits: both sides of 2560 keys, of 32 general programs and of half the CUs
@needs_ablate
@pytest.mark.parametrize("shape,rows", [
    ((3, 32, 4, 31, 2560, 64), 0), ((3, 32, 4, 31, 2559, 64), 32), ((3, 32, 8, 22, 3531, 32), 0),
    ((9, 8, 2, 36, 2984, 64), 32), ((3, 32, 8, 36, 3164, 64), 32), ((3, 16, 8, 39, 3600, 64), 32),
    ((1, 28, 4, 103, 3388, 32), 0), ((3, 16, 8, 39, 2736, 16), 32), ((2, 8, 8, 32, 2736, 64), 32)])
def test_long_keys_of_grids_that_leave_cus_idle(shape, rows):
    assert _kernel(*shape) == rows
    if rows == 0:
        _only_with_its_splits(shape)


def _only_with_its_splits(shape):
    """A call that the general kernel takes for its splits: the wave-split kernel keeps it where the
    caller allows fewer (fa2_attn_fwd: one), and the count told makes the same launch again."""
    lib = _lib.lib()
    B, h_q, h_kv, n_q, n_kv, D = shape
    assert _plan(*shape, 0, False)["kernel"] == WAVE_SPLIT
    for n in range(2, 17):
        told = _launch_splits(*shape, n)
        plans = [_plan(*shape, 0, False, num_splits=x,
                       workspace_bytes=lib.fa2_workspace_bytes(B, h_q, n_q, D, x)) for x in (n, told)]
        assert plans[0] == plans[1] and plans[0]["splits"] == told, (n, told, plans)
        assert n >= _lib.num_splits(*shape, False, 128, 0, 256) or plans[0]["kernel"] == WAVE_SPLIT


# 33 to 64 rows at head_dim 128: two row tiles whose splits leave CUs idle against one general program
# with splits for all of them, on both sides of 544 keys a general split (660 of four, 2048 where seven in eight CUs
# have a workgroup); never where the wave-split kernel's fill the CUs, the group does not pack, or at 64
@needs_ablate
@pytest.mark.parametrize("shape,rows", [
    ((6, 32, 4, 6, 8264, 128), 32), ((6, 32, 4, 6, 8704, 128), 0), ((3, 12, 12, 41, 4351, 128), 32),
    ((3, 12, 12, 41, 4352, 128), 0), ((6, 12, 12, 44, 2639, 128), 32), ((6, 12, 12, 44, 2640, 128), 0),
    ((30, 32, 4, 5, 8191, 128), 32), ((30, 32, 4, 5, 8192, 128), 0), ((8, 8, 8, 46, 20000, 128), 32),
    ((3, 12, 12, 41, 20000, 64), 32), ((9, 28, 4, 7, 20000, 128), 32), ((3, 12, 12, 32, 20000, 128), 32)])
def test_two_row_tiles_of_long_keys(shape, rows):
    assert _kernel(*shape) == rows
    if rows == 0:
        _only_with_its_splits(shape)


# 65 to 128 rows on one to two 32-row workgroups per CU: both sides of 1700 / 2900 keys, of 128 rows and
# of 1.4 workgroups per CU
@needs_ablate
@pytest.mark.parametrize("shape,rows", [
    ((6, 16, 16, 72, 1700, 128), 0), ((6, 16, 16, 72, 1699, 128), 32), ((10, 8, 8, 124, 2029, 128), 0),
    ((63, 16, 2, 10, 1784, 128), 64), ((8, 8, 8, 160, 1877, 128), 32), ((12, 32, 8, 18, 2900, 64), 0),
    ((12, 32, 8, 18, 2899, 64), 32), ((31, 32, 4, 11, 3259, 64), 64), ((3, 28, 4, 18, 1900, 128), 32)])
def test_one_general_program_for_three_row_tiles(shape, rows):
    assert _kernel(*shape) == rows
    if rows == 0:
        _only_with_its_splits(shape)


# Which kernel the default-tile calls of the GPU tests run (tests/test_gpu_wavesplit.py,
# tests/test_gpu_splitkv.py), so that a change of the rule cannot take them off it unseen: rows per
# wave-split workgroup and whether its splits merge, per head_dim
@needs_ablate
@pytest.mark.parametrize("shape,causal,want", [
    ((2, 8, 2, 1, 129), False, {16: (32, 0), 64: (32, 0), 128: (32, 0)}),
    ((2, 6, 2, 11, 193), False, {D: (32, 0) for D in (16, 32, 64, 128)}),
    ((2, 5, 1, 13, 4100), False, {D: (32, 1) for D in (16, 32, 64, 128)}),
    ((2, 2, 2, 64, 9000), False, {D: (32, 1) for D in (16, 32, 64, 128)}),
    ((2, 8, 2, 65, 2048), False, {D: (32, 1) for D in (16, 32, 64, 128)}),
    ((2, 8, 2, 64, 2048), False, {D: (32, 1) for D in (16, 32, 64, 128)}),
    ((17, 8, 8, 40, 300), False, {D: (64, 0) for D in (16, 32, 64, 128)}),
    ((33, 28, 4, 7, 700), False, {D: (64, 0) for D in (16, 32, 64, 128)}),
    ((8, 28, 4, 40, 6200), False, {16: (32, 0), 32: (32, 0), 64: (64, 1), 128: (64, 1)}),
    ((20, 28, 4, 30, 4200), False, {D: (64, 0) for D in (16, 32, 64, 128)}),
    ((4, 8, 8, 1201, 520), False, {16: (64, 0), 32: (64, 0)}),
    ((1, 4, 1, 256, 256), True, {D: (32, 0) for D in (16, 32, 64, 128)}),
    ((2, 16, 16, 520, 520), True, {D: (64, 0) for D in (16, 32, 64, 128)})])
def test_gpu_tests_reach_the_wave_split_kernel(shape, causal, want):
    B, h_q, h_kv, n_q, n_kv = shape
    for D, (rows, merged) in want.items():
        n = 1 if causal else _lib.num_splits(B, h_q, h_kv, n_q, n_kv, D, causal, 128, 0, 256)
        plan = _plan(B, h_q, h_kv, n_q, n_kv, D, 0, causal, num_splits=n,
                     workspace_bytes=_lib.lib().fa2_workspace_bytes(B, h_q, n_q, D, n))
        assert plan["kernel"] == WAVE_SPLIT and plan["rows"] == rows and (plan["splits"] > 1) == merged, plan
