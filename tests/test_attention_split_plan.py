"""How the planner cuts a query tile's KV range (nsg_attn_plan).  Host only."""
import ctypes as C

import numpy as np
import pytest

from nanosglang_amd import _native
from nanosglang_amd._native import NSG_ATTN_WORK_INTS, AttnPlan


def _plan(q, L, B, Hq, Hkv, D, P=16, cus=256):
    lib = _native.load()
    npg = -(-L // P)
    qo = (np.arange(B + 1) * q).astype(np.int32)
    kvp = (np.arange(B + 1) * npg).astype(np.int32)
    last = np.full(B, (L % P) or P, np.int32)
    cap = 1 << 16
    work = np.zeros((cap, NSG_ATTN_WORK_INTS), np.int32)
    pl = AttnPlan()
    rc = lib.nsg_attn_plan(qo.ctypes.data, kvp.ctypes.data, last.ctypes.data, B, Hq, Hkv, D, P, 1,
                           cus, work.ctypes.data, cap, C.byref(pl))
    assert rc == 0, lib.nsg_last_error()
    return pl, work[:pl.num_work]


# (case, KV groups, split?, steps of the first tile's items)
CASES = [
    # several KV groups, 288 workgroups (a second round either way), three
    # splits or more: whole chunks and a rest
    ((48, 1200, 1, 32, 32, 128), 2, [16, 16, 5]),
    ((64, 16000, 1, 12, 12, 64), 4, [96, 96, 96, 96, 96, 19]),
    # ... also with a rest of one step in the list's last tile
    ((64, 2000, 1, 32, 32, 128), 2, [31, 30]),
    # ... no tile with more than two splits: even shares
    ((48, 4000, 1, 64, 8, 128), 2, None),
    # all workgroups at once: even shares
    ((64, 1100, 1, 14, 2, 64), 4, [16, 17]),
    # one KV group: even shares
    ((24, 4000, 64, 14, 2, 64), 1, None),
    ((16, 4000, 16, 64, 8, 128), 1, None),
]


@pytest.mark.parametrize("case,groups,steps", CASES)
def test_shares(case, groups, steps):
    pl, work = _plan(*case)
    q, L, B = case[:3]
    assert pl.kv_groups == groups and pl.max_splits > 1 and pl.row_tiles <= 4
    tiles = {}
    for w in work.tolist():
        tiles.setdefault(w[0], []).append((w[4], w[5], w[6]))
    for qs, items in tiles.items():
        end = L - q + qs % q + pl.q_tile_tokens if qs % q + pl.q_tile_tokens <= q else L
        assert items[0][0] == 0 and items[-1][1] == end
        assert all(a[1] == b[0] for a, b in zip(items, items[1:]))       # no gap, no overlap
        assert all(i[0] % 32 == 0 and i[2] == len(items) for i in items)
    first = [-(-(e - s) // 32) for s, e, _ in tiles[0]]
    if L == 2000:
        last = [-(-(e - s) // 32) for s, e, _ in list(tiles.values())[-1]]
        assert last == [31, 31, 1]
    if steps is None:
        assert max(first) - min(first) <= 1
    else:
        assert first == steps
