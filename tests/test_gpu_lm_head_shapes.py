"""The lm_head kernel's argmax form at the borders of its workgroup shapes: the
tokens are the first argmax of the logits form's rows, bit for bit, and no key
is written past the stated workspace."""
import ctypes as C

import pytest
import torch

from nanosglang_amd import _native, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 16, 33, 64, 65, 80, 81, 96, 97, 129, 160])
@pytest.mark.parametrize("N", [4, 32, 164, 65532, 65536, 65700])
def test_tokens_match_the_logits_form(M, N):
    print(f"case: {M} rows x {N} columns", flush=True)
    K = 256
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).bfloat16()
    ss = kernels.row_sumsq(x)
    y = kernels.lm_head_fold(x, w, ss, 1e-6)
    # the first index of the largest value (torch.argmax leaves ties open)
    want = (y == y.amax(-1, keepdim=True)).int().argmax(-1)
    lib = _native.load()
    need = lib.nsg_linear_argmax_workspace_bytes(M, N)
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    tok = torch.empty(M, dtype=torch.int64, device="cuda")
    kernels.check(lib.nsg_lm_head_fold_argmax(
        x.data_ptr(), K, w.data_ptr(), K, M, N, K, ss.data_ptr(), K // 16, K, 1e-6,
        ws.data_ptr(), need, tok.data_ptr(), 1, torch.cuda.current_stream().cuda_stream),
        "nsg_lm_head_fold_argmax")
    assert torch.equal(tok, want)
    assert (ws[need:] == 0x5A).all()
    kc = C.c_int32(0)
    kernels.check(lib.nsg_lm_head_fold_keys(
        x.data_ptr(), K, w.data_ptr(), K, M, N, K, ss.data_ptr(), K // 16, K, 1e-6,
        ws.data_ptr(), need, C.byref(kc), torch.cuda.current_stream().cuda_stream),
        "nsg_lm_head_fold_keys")
    assert kc.value <= 4 * -(-N // 128) and M * kc.value * 8 <= need


@pytest.mark.parametrize("M,N", [(1, 4), (16, 32), (81, 48), (160, 20)])
def test_plain_argmax_needs_one_key_per_16_columns(M, N):
    """nsg_linear_argmax of few columns: its kernel writes a key per 16 columns, and
    a workspace of that size (less than the folded form's) is enough."""
    print(f"case: plain argmax, {M} rows x {N} columns", flush=True)
    K = 256
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(N, K, generator=g, device="cuda").bfloat16()
    y = kernels.linear(x, w, force=True)
    need = M * -(-N // 16) * 8
    ws = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
    tok = torch.empty(M, dtype=torch.int64, device="cuda")
    kernels.check(_native.load().nsg_linear_argmax(
        x.data_ptr(), K, w.data_ptr(), K, None, M, N, K, ws.data_ptr(), need, tok.data_ptr(), 1,
        torch.cuda.current_stream().cuda_stream), "nsg_linear_argmax")
    assert torch.equal(tok, (y == y.amax(-1, keepdim=True)).int().argmax(-1))
    assert (ws[need:] == 0x5A).all()
