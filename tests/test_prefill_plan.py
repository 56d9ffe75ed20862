"""The planner's prefill tiles (nsg_attn_plan, csrc/prefill_attention.hip): which
batches get them, and that they cover every query row once.  Host only."""
import ctypes as C

import numpy as np
import pytest

from nanosglang_amd import _native
from nanosglang_amd._native import NSG_ATTN_WORK_INTS, AttnPlan


def _plan(q_lens, kv_lens, Hq, Hkv, D, P=16, causal=1, cus=256):
    lib = _native.load()
    npg = [(L + P - 1) // P for L in kv_lens]
    qo = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    kvp = np.concatenate([[0], np.cumsum(npg)]).astype(np.int32)
    last = np.asarray([(L % P) or P for L in kv_lens], np.int32)
    cap = 1 << 16
    work = np.zeros((cap, NSG_ATTN_WORK_INTS), np.int32)
    pl = AttnPlan()
    rc = lib.nsg_attn_plan(qo.ctypes.data, kvp.ctypes.data, last.ctypes.data, len(q_lens), Hq, Hkv,
                           D, P, causal, cus, work.ctypes.data, cap, C.byref(pl))
    assert rc == 0, lib.nsg_last_error()
    return pl, work[:pl.num_work], qo, kvp


@pytest.mark.parametrize("Hq,Hkv,D,rows", [(14, 2, 64, 128), (32, 8, 128, 256), (8, 8, 64, 128),
                                           (64, 1, 128, 256)])
@pytest.mark.parametrize("causal", [0, 1])
def test_tiles_cover_every_row_once_longest_first(Hq, Hkv, D, rows, causal):
    rng = np.random.default_rng(Hq + causal)
    kv = list(rng.integers(64, 513, 300)) + [1, 2000]
    ql = [max(1, int(L * f)) for L, f in zip(kv, rng.choice([1.0, 0.9], len(kv)))]
    pl, work, qo, kvp = _plan(ql, kv, Hq, Hkv, D, causal=causal)
    G = Hq // Hkv
    T = rows // G
    assert (pl.row_tiles, pl.q_tile_tokens, pl.kv_groups) == (rows // 16, T, 1)
    assert pl.num_merge == 0 and pl.max_splits == 1 and pl.workspace_bytes == 256
    want = []
    for b, (q, L) in enumerate(zip(ql, kv)):
        for qb in range(0, q, T):
            qn = min(T, q - qb)
            end = L - q + qb + qn if causal else L
            want.append((qo[b] + qb, qn, L - q + qb if causal else L - 1, kvp[b], 0, end, 1, 0))
    assert sorted(map(tuple, work.tolist())) == sorted(want)
    assert (np.diff((work[:, 5] + 63) // 64) <= 0).all()      # in 64-token steps


@pytest.mark.parametrize("q,kv,heads,prefill", [
    ([5] * 64, [500] * 64, (14, 2, 64), False),          # verify rows: tiles mostly padding
    ([9] * 64, [5000] * 64, (32, 8, 128), False),
    ([300], [300], (14, 2, 64), False),                  # too few workgroups
    ([512] * 2, [8000] * 2, (14, 2, 64), False),         # few and long: needs the KV split
    ([300] * 4, [300] * 4, (14, 2, 64), True),
    ([1000], [1000], (32, 8, 128), True),
    ([512] * 16, [8000] * 16, (14, 2, 64), True),
    ([20000], [20000], (14, 2, 64), False),              # more pages than an item holds
])
def test_which_batches_get_prefill_tiles(q, kv, heads, prefill):
    pl, _, _, _ = _plan(q, kv, *heads)
    assert (pl.row_tiles >= 8) == prefill
    if not prefill:      # the verify kernel's forms are what they were
        assert pl.row_tiles <= 4 and pl.q_tile_tokens * (heads[0] // heads[1]) <= 64


@pytest.mark.parametrize("P", [1, 2, 4, 8, 16, 32])
@pytest.mark.parametrize("Hq,Hkv,D", [(14, 2, 64), (32, 8, 128)])
def test_items_are_never_split_up_to_the_page_list(Hq, Hkv, D, P):
    """The prefill kernel sweeps an item's whole KV range and merges nothing, so
    every query tile is one item up to the 1022 pages an item's list holds (also
    where 1022 pages are no whole number of 32-token steps); past them the batch
    is the verify kernel's."""
    full = 1022 * P
    for L in (full, full - 1, full // 32 * 32, min(full, full // 32 * 32 + 1)):
        B = max(2, 16384 // L)
        pl, work, qo, kvp = _plan([L] * B, [L] * B, Hq, Hkv, D, P=P)
        T = pl.q_tile_tokens
        assert pl.row_tiles >= 8 and pl.max_splits == 1 and pl.num_merge == 0, (P, L)
        assert len(work) == B * -(-L // T), (P, L)
        assert sorted(zip(work[:, 0], work[:, 1], work[:, 4], work[:, 5])) == [
            (b * L + q, min(T, L - q), 0, min(q + T, L)) for b in range(B) for q in range(0, L, T)]
    pl, _, _, _ = _plan([full + 1] * 16, [full + 1] * 16, Hq, Hkv, D, P=P)
    assert pl.row_tiles <= 4


def test_a_prefill_plan_with_splits_is_refused():
    """A record that claims prefill tiles and KV splits is no plan of this
    library: nsg_attn_run answers with an error and launches nothing (the pointers
    here are never followed)."""
    pl, _, _, _ = _plan([300] * 4, [300] * 4, 14, 2, 64)
    assert pl.row_tiles == 8
    lib = _native.load()
    dummy = C.create_string_buffer(256)
    ptr = [C.cast(dummy, C.c_void_p)] * 9
    for field, value in (("max_splits", 2), ("num_merge", 1)):
        bad = AttnPlan.from_buffer_copy(pl)
        setattr(bad, field, value)
        rc = lib.nsg_attn_run(C.byref(bad), *ptr, 16, 100, 0.125, 1, ptr[0], 256, None)
        assert rc != 0 and b"prefill" in lib.nsg_last_error() and b"split" in lib.nsg_last_error()


@pytest.mark.parametrize("q,kv,heads,row_tiles", [
    # fewer than two workgroups per CU, measured ahead on the verify kernel
    ([16] * 16, [600] * 16, (64, 1, 128), 0),
    ([256], [300], (64, 1, 128), 0),
    ([256], [2040], (40, 8, 128), 0),
    ([1024], [2040], (16, 2, 128), 0),
    ([1024], [1200], (12, 12, 64), 0),
    # ... and on the prefill kernel
    ([1000], [1000], (32, 8, 128), 16),
    ([500], [500], (32, 8, 128), 8),
    ([48] * 16, [1200] * 16, (32, 8, 128), 16),
    ([512] * 2, [512] * 2, (14, 2, 64), 8),
    # many rounds of short contexts: 128 rows
    ([128] * 64, [128] * 64, (32, 8, 128), 8),
    ([256] * 16, [256] * 16, (64, 8, 128), 8),
    ([512] * 32, [512] * 32, (32, 8, 128), 16),
])
def test_which_kernel_a_batch_gets(q, kv, heads, row_tiles):
    """Row tiles of the prefill kernel (0: the verify kernel's 1 .. 4), as measured
    on both."""
    pl, _, _, _ = _plan(q, kv, *heads)
    assert pl.row_tiles == row_tiles if row_tiles else pl.row_tiles <= 4


@pytest.mark.parametrize("P", [1, 4])
@pytest.mark.parametrize("L,B,heads,prefill", [
    (32, 16, (32, 8, 128), False), (100, 4, (32, 8, 128), False), (32, 32, (14, 2, 64), False),
    (960, 1, (32, 8, 128), True), (256, 32, (14, 2, 64), True)])
def test_small_pages_without_kv_groups(L, B, heads, prefill, P):
    """Pages below 16 tokens: the verify kernel has one KV group only, which a few
    short prompts still run faster on."""
    pl, _, _, _ = _plan([L] * B, [L] * B, *heads, P=P)
    assert (pl.row_tiles >= 8) == prefill
