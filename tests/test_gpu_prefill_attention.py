"""The prefill attention kernel (csrc/prefill_attention.hip) against the float64
oracle, at the edges of its tiles: bounds as in test_gpu_attention.py (bf16
output and probabilities).  ``num_cus=8`` makes the planner take its tiles for
small batches too."""
import numpy as np
import pytest
import torch

from nanosglang_amd import workloads
from nanosglang_amd.kernels import BatchPrefillWithPagedKVCacheWrapper
from oracle.verify_attention import verify_attention

pytestmark = pytest.mark.gpu


def _run(c, Hq, Hkv, D, causal, row_tiles=None):
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda().bfloat16()  # noqa: E731
    w = BatchPrefillWithPagedKVCacheWrapper(
        torch.empty(1 << 20, dtype=torch.uint8, device="cuda"), "NHD", num_cus=8)
    w.plan(c["qo_indptr"], c["kv_indptr"], c["kv_indices"], c["kv_last_page_len"], Hq, Hkv, D,
           c["page_size"], causal=causal)
    assert w.plan_info.row_tiles >= 8, "not the prefill kernel"
    assert row_tiles in (None, w.plan_info.row_tiles)
    out = w.run(dev(c["q"]), (dev(c["k"]), dev(c["v"])))
    return out.float().cpu().numpy(), w


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Hq,Hkv,D,P", [(14, 2, 64, 16), (4, 4, 64, 1), (32, 8, 128, 16),
                                        (16, 2, 128, 128), (64, 8, 128, 4), (12, 4, 64, 64)])
def test_prefill_tile_edges(Hq, Hkv, D, P, causal):
    # KV lengths around the 64-token step, the ring's depth and the tile; query
    # lengths equal to the context and shorter (a cached prefix)
    kv = [63, 64, 65, 127, 128, 129, 193, 257, 320, 449, 600]
    ql = [63, 64, 65, 127, 100, 129, 193, 250, 256, 449, 511]
    c = workloads.verify_attention_batch(batch=len(kv), kv_lens=kv, q_lens=ql, page_size=P,
                                         num_qo_heads=Hq, num_kv_heads=Hkv, head_dim=D,
                                         num_pages=sum(-(-L // P) for L in kv) + 3, seed=D + P)
    print(f"case: {Hq}/{Hkv} x {D}, pages of {P}, causal {causal}", flush=True)
    got, w = _run(c, Hq, Hkv, D, causal, row_tiles=8 if D == 64 else 16)
    ref = verify_attention(c["q"], c["k"], c["v"], c["qo_indptr"], c["kv_indptr"],
                           c["kv_indices"], c["kv_last_page_len"], c["sm_scale"], causal)
    assert w.check_flags() == 0
    assert (np.abs(got - ref) <= 2e-3 + 2.0 ** -8 * np.abs(ref)).all()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Hq,Hkv,P,ql", [
    (32, 8, 16, [30, 31, 32, 25, 30, 32, 28, 31, 32, 30, 29]),      # chunks over a cached prefix
    (4, 4, 1, [127, 100, 120, 128, 126, 97, 125, 128, 119, 128, 120]),
    (64, 8, 128, [15, 16, 14, 12, 16, 15, 16, 13, 16, 15, 16]),
    (16, 2, 4, None)])                                              # short prompts, many rounds
def test_128_row_tiles_at_head_dim_128(Hq, Hkv, P, ql, causal):
    """The two-slot ring of 128 rows at head dim 128: contexts around one, two and
    three of its 64-token steps and long ones."""
    kv = [63, 64, 65, 127, 128, 129, 193, 257, 320, 349, 384]
    ql, kv = (kv, kv) if ql is None else (
        [min(q, L) for q, L in zip(ql, kv)] + ql[:2], kv + [1000, 1009])
    c = workloads.verify_attention_batch(batch=len(kv), kv_lens=kv, q_lens=ql, page_size=P,
                                         num_qo_heads=Hq, num_kv_heads=Hkv, head_dim=128,
                                         num_pages=sum(-(-L // P) for L in kv) + 3, seed=P)
    print(f"case: {Hq}/{Hkv} x 128, pages of {P}, causal {causal}", flush=True)
    got, w = _run(c, Hq, Hkv, 128, causal, row_tiles=8)
    ref = verify_attention(c["q"], c["k"], c["v"], c["qo_indptr"], c["kv_indptr"],
                           c["kv_indices"], c["kv_last_page_len"], c["sm_scale"], causal)
    assert w.check_flags() == 0
    assert (np.abs(got - ref) <= 2e-3 + 2.0 ** -8 * np.abs(ref)).all()


@pytest.mark.parametrize("Hq,Hkv,D", [(14, 2, 64), (32, 8, 128)])
def test_prefill_at_the_end_of_the_page_list(Hq, Hkv, D):
    """Pages of one token, contexts around the 992 tokens that are whole 32-token
    steps of the 1022 an item's page list holds: one item per tile to the end."""
    kv = [992, 993, 1010, 1022]
    c = workloads.verify_attention_batch(batch=4, kv_lens=kv, q_lens=kv, page_size=1,
                                         num_qo_heads=Hq, num_kv_heads=Hkv, head_dim=D,
                                         num_pages=sum(kv) + 3, seed=D)
    print(f"case: {Hq}/{Hkv} x {D}, pages of 1, contexts {kv}", flush=True)
    got, w = _run(c, Hq, Hkv, D, True)
    assert w.plan_info.max_splits == 1
    ref = verify_attention(c["q"], c["k"], c["v"], c["qo_indptr"], c["kv_indptr"],
                           c["kv_indices"], c["kv_last_page_len"], c["sm_scale"], True)
    assert w.check_flags() == 0
    assert (np.abs(got - ref) <= 2e-3 + 2.0 ** -8 * np.abs(ref)).all()


@pytest.mark.parametrize("Hq,Hkv,D", [(14, 2, 64), (32, 8, 128)])
def test_prefill_growing_scores_and_bad_page(Hq, Hkv, D):
    """Scores that grow along the context rescale the running sums often; a page
    id outside the pool raises the flag and leaves other requests alone."""
    kv = [400, 130, 300]
    c = workloads.verify_attention_batch(batch=3, kv_lens=kv, q_lens=kv, num_qo_heads=Hq,
                                         num_kv_heads=Hkv, head_dim=D, num_pages=60, seed=9)
    for place, page in enumerate(c["kv_indices"]):
        c["k"][page] *= 1.0 + 0.5 * place
    c["k"] = torch.from_numpy(c["k"]).bfloat16().float().numpy()
    got, w = _run(c, Hq, Hkv, D, True)
    ref = verify_attention(c["q"], c["k"], c["v"], c["qo_indptr"], c["kv_indptr"],
                           c["kv_indices"], c["kv_last_page_len"], c["sm_scale"], True)
    # P in bf16 near one-hot rows: 2^-8 of the largest |v| (about 2) beside the usual bound
    assert (np.abs(got - ref) <= 1e-2 + 2.0 ** -8 * np.abs(ref)).all()
    assert w.check_flags() == 0
    bad = dict(c, kv_indices=c["kv_indices"].copy())
    bad["kv_indices"][26] = 10 ** 6                      # request 1's second page
    got2, w2 = _run(bad, Hq, Hkv, D, True)
    assert w2.check_flags() == 1
    a, z = c["qo_indptr"][1], c["qo_indptr"][2]
    assert np.array_equal(got2[:a], got[:a]) and np.array_equal(got2[z:], got[z:])
