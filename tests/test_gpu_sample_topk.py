"""The one-launch top-k sampler (topk_kernel in csrc/sample.hip) at its edges:
against the oracle wherever the draw is more than 1e-6 of the mass from a
boundary (the two sides' exp2 differ in the last bit), as test_gpu_sample.py."""
import numpy as np
import pytest
import torch

from nanosglang_amd import kernels
from oracle import sampling as osm

pytestmark = pytest.mark.gpu
MARGIN = 1e-6
DTYPES = [torch.bfloat16, torch.float32]


def _np(x):
    return x.cpu().view(torch.int16).numpy().view(np.uint16) if x.dtype == torch.bfloat16 \
        else x.cpu().numpy()


def _check(x, T, K, P, u):
    got = kernels.sample(x, T, K, P, u).cpu().tolist()
    rows, uu, n = _np(x.contiguous()), u.cpu().tolist(), 0
    for r, tok in enumerate(got):
        want, margin = osm.sample(rows[r], T, K, P, uu[r])
        if margin >= MARGIN:
            assert tok == want, (r, K, P, tok, want, margin)
            n += 1
    assert n >= 0.5 * len(got)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V", [9, 64, 1023, 8193, 155640, 155649, 160001])
def test_lengths_and_unaligned_rows(dtype, V):
    print(f"case: V {V} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(V)
    base = torch.randn(6, V + 3, generator=g, device="cuda").mul(2).to(dtype)
    u = torch.rand(6, generator=g, device="cuda")
    for off in (0, 1, 3):                       # rows at every alignment
        x = base[:, off:off + V]
        for K, P in ((1, 0.9), (1, 1.0), (8, 0.9), (50, 0.9), (128, 0.95), (256, 0.95), (257, 0.95)):
            _check(x, 0.8, K, P, u)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V", [155640, 160001])
def test_many_kept(dtype, V):
    """Top-k above 128: the one launch takes it from 2^20 elements (bf16 above 200,
    2^22: 28 rows)."""
    print(f"case: many kept, V {V} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(V + 1)
    x = torch.randn(28, V, generator=g, device="cuda").mul(2).to(dtype)
    u = torch.rand(28, generator=g, device="cuda")
    for K, P in ((129, 0.9), (200, 1.0), (256, 0.95), (256, 1.0)):
        _check(x, 0.8, K, P, u)


@pytest.mark.parametrize("dtype", DTYPES)
def test_ties_masks_and_signed_zeros(dtype):
    V = 20000
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(8, V, generator=g, device="cuda") * 2
    x[0] = torch.round(x[0])                                 # thousands of ties below the top
    x[1, 30:] = float("-inf")                                # a grammar mask: fewer than K left
    x[2] = torch.where(x[2] > 0, 0.0, -0.0)                  # -0 == +0
    x[3, :] = 0.25                                           # more ties than the lists hold
    x[4, 1:] = x[4, 0] - 1                                   # one above them
    x[5] = torch.round(x[5] / 4)
    x = x.to(dtype)
    for K, P in ((50, 0.9), (50, 1.0), (1, 0.5), (128, 0.95), (200, 0.99)):
        for u0 in (0.05, 0.37, 0.93):
            print(f"case: ties {dtype} K {K} P {P} u {u0}", flush=True)
            _check(x, 0.8, K, P, torch.full((8,), u0, device="cuda"))


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_without_mass_give_minus_one(dtype):
    x = torch.randn(4, 5000, device="cuda").to(dtype)
    x[0, 7], x[1, 9] = float("inf"), float("nan")
    x[2] = float("-inf")
    got = kernels.sample(x, 0.8, 50, 0.9, torch.rand(4, device="cuda")).tolist()
    assert got[:3] == [-1, -1, -1] and got[3] >= 0


def test_old_workspace_size_still_works():
    """A workspace without room for the row marks (the size before they were
    added) runs the staged launches alone, with the same tokens."""
    from nanosglang_amd import _native
    lib = _native.load()
    R, V = 5, 30000
    x = torch.randn(R, V, device="cuda").bfloat16()
    u = torch.rand(R, device="cuda")
    ws = torch.zeros(lib.nsg_sample_workspace_bytes(R, V), dtype=torch.uint8, device="cuda")
    out = [torch.full((R,), -7, dtype=torch.int64, device="cuda") for _ in range(2)]
    for o, n in zip(out, (ws.numel(), ws.numel() - 256)):
        kernels.check(lib.nsg_sample(x.data_ptr(), V, 0, R, V, 0.8, 40, 0.9, u.data_ptr(), 1,
                                     o.data_ptr(), ws.data_ptr(), n,
                                     torch.cuda.current_stream().cuda_stream), "nsg_sample")
    assert torch.equal(out[0], out[1]) and (out[0] >= 0).all()
