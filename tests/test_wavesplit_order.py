"""The wave-split kernel's program order, checked on the CPU: every row tile of every (batch, KV
head) runs exactly once, on any device topology, and whatever the caller's packing.

split_program (csrc/attn_fwd_schedule.hpp) is __host__ __device__; the measurement library runs the
kernel's own code for a whole launch (fa2_ablate_program_map, static_order 2: the library's own
choice of kernel). No GPU call.
"""

import ctypes
import random

import numpy as np
import pytest

from test_schedule import INFO_WORDS, TOPOLOGIES, _map_fn, needs_ablate

I32P = ctypes.POINTER(ctypes.c_int32)


def library_map(fn, shape):
    """(programs, info) of a launch; a wave-split grid has up to four workgroups per 128 rows."""
    B, hq, hkv, n, d, causal, pack, bm, cus, xcds, static = shape
    cap = 3 * (5 * B * hq * -(-n // 32) + 4096)
    out = np.full(cap, -7, dtype=np.int32)
    info = np.zeros(INFO_WORDS, dtype=np.int32)
    rc = fn(B, hq, hkv, n, d, causal, pack, bm, cus, xcds, static, -1, 0,
            out.ctypes.data_as(I32P), cap, info.ctypes.data_as(I32P), INFO_WORDS)
    assert rc == 0, shape
    return out[: 3 * int(info[0])].reshape(-1, 3), info


def _shapes(n, seed):
    rnd = random.Random(seed)
    for _ in range(n):
        h_kv = rnd.choice([1, 2, 3, 4, 5, 8, 16, 32])
        group = rnd.choice([1, 1, 2, 4, 5, 7, 8])
        pack = rnd.choice([1, group]) if 128 % group == 0 else 1
        yield (rnd.choice([1, 1, 2, 3, 5, 9]), h_kv * group, h_kv,
               rnd.choice([129, 191, 193, 200, 256, 383, 384, 500, 512, 777, 1000, 1500, 2048, 3333]),
               rnd.choice([16, 32, 64, 128]), rnd.random() < 0.6, pack)


@needs_ablate
@pytest.mark.parametrize("cus,xcds", TOPOLOGIES)
def test_every_row_tile_runs_once(cus, xcds):
    fn = _map_fn()
    taken = set()
    for B, hq, hkv, n, d, causal, pack in _shapes(400, cus * 100 + xcds):
        shape = (B, hq, hkv, n, d, int(causal), pack, 128, cus, xcds)
        progs, info = library_map(fn, shape + (2,))
        general, ginfo = library_map(fn, shape + (1,))
        if np.array_equal(info, ginfo):
            continue  # the general kernel (tests/test_schedule.py)
        rows = info[6]
        taken.add((bool(causal), int(rows)))
        group = hq // hkv
        tiles = -(-n * group // rows)
        assert rows in (32, 64) and info[9] == tiles and info[10] == B * hkv
        assert info[0] == tiles * B * hkv == len(progs), shape
        seen = {tuple(x) for x in progs.tolist()}
        assert seen == {(t, b, h * group) for t in range(tiles) for b in range(B)
                        for h in range(hkv)}, shape
        # the choice and the order do not depend on the packing
        other = 1 if pack > 1 else (group if 128 % group == 0 else 1)
        progs2, info2 = library_map(fn, shape[:6] + (other,) + shape[7:] + (2,))
        assert np.array_equal(progs, progs2) and np.array_equal(info[[0, 6, 9, 10]],
                                                                info2[[0, 6, 9, 10]])
    if cus >= 128:
        assert taken >= {(True, 32), (True, 64), (False, 32)}, taken


@needs_ablate
def test_causal_tiles_pair_heavy_with_light():
    """B1 H32/8 N1024 head_dim 128: 512 workgroups on 256 CUs; XCD-local slots s and s + 32 meet on
    a CU, and their row tiles (keys walked grow with the tile) add up to the same everywhere."""
    progs, info = library_map(_map_fn(), (1, 32, 8, 1024, 128, 1, 1, 128, 256, 8, 2))
    assert info[0] == 512 and info[6] == 64
    tile = np.asarray(progs)[:, 0].reshape(64, 8)  # block = slot * 8 + XCD
    assert (tile[:32] + tile[32:] == 63).all()
