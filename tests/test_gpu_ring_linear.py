"""The 8B-class linear kernel (csrc/ring_linear.hip) at the edges of its tiles,
against torch fp32 on the dequantised weights: bf16 rounding of one fp32 sum
(2^-8 relative, 2^-6 through SwiGLU's three roundings) plus the sums'
reordering (2e-3 absolute at these magnitudes, as in test_gpu_linear.py), and
FP8 against bf16 weights bit for bit."""
import pytest
import torch

from nanosglang_amd import _native, kernels
from nanosglang_amd.model.quantization import fp8_quantize_rows

pytestmark = pytest.mark.gpu


def _weights(blocks, K, seed, pad=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(sum(blocks), K, generator=g, device="cuda") * K ** -0.5
    w8, s = fp8_quantize_rows(w, blocks)
    if pad:                                  # rows further apart than they are long
        wide = torch.zeros(sum(blocks), K + pad, dtype=torch.uint8, device="cuda")
        wide[:, :K] = w8.view(torch.uint8)
        w8 = wide.view(torch.float8_e4m3fn)[:, :K]
    return w8, s


@pytest.mark.parametrize("M", [1, 16, 17, 33, 48, 49, 65, 97, 129, 160])
@pytest.mark.parametrize("I,K", [(10244, 2048), (8192, 2176)])
def test_swiglu_ragged_columns(M, I, K):
    print(f"case: SwiGLU {M} x {I} x {K}", flush=True)
    w8, s = _weights([I, I], K, M)
    wd = kernels.dequant_fp8(w8, s)
    x = torch.randn(M, K + 8, device="cuda").bfloat16()[:, :K]      # strided rows
    out = torch.full((M, I + 4), 7.0, dtype=torch.bfloat16, device="cuda")
    y = kernels.linear(x, w8, swiglu=True, w_scale=s, out=out[:, :I])
    gate, up = (x.float() @ wd.float().T).chunk(2, -1)
    ref = torch.nn.functional.silu(gate) * up
    assert ((y.float() - ref).abs() <= 2.0 ** -6 * ref.abs() + 2e-3).all()
    assert (out[:, I:] == 7).all()
    if I >= 154 * 64 or M > 32:              # both weight types on this kernel
        assert torch.equal(y, kernels.linear(x, wd, swiglu=True, force=True))


@pytest.mark.parametrize("M", [16, 17, 32, 33, 49, 65, 97, 129, 160])
@pytest.mark.parametrize("N,K,pad", [(4100, 6400, 0), (6144, 4096, 16), (1028, 25600, 0),
                                     (4100, 6400, 8), (33000, 768, 0)])
def test_bias_split_k(M, N, K, pad):
    """pad 8: FP8 rows that are not 16-byte aligned stay on the weight-streaming
    kernel; 33000 columns: K is not split, and up to 32 rows (its 258 column
    tiles, K below 1024) the weight-streaming kernel is ahead."""
    print(f"case: bias {M} x {N} x {K}, row pad {pad}", flush=True)
    lib = _native.load()
    need = lib.nsg_linear_workspace_bytes(M, N, K, 0)
    assert (need > 0) == (M >= 17 and N != 33000)
    w8, s = _weights([N], K, M + N, pad)
    wd = kernels.dequant_fp8(w8, s)
    x = torch.randn(M, K, device="cuda").bfloat16()
    b = torch.randn(N, device="cuda").bfloat16()
    y = kernels.linear(x, w8, b, w_scale=s)
    ref = x.float() @ wd.float().T + b.float()
    assert ((y.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2e-3).all()
    twin = kernels.linear(x, wd, b, force=True)
    if pad != 8:
        assert torch.equal(y, twin)
    else:                                    # another order of the fp32 sums
        assert ((y.float() - twin.float()).abs() <= 2.0 ** -7 * ref.abs() + 2e-3).all()
    # without the workspace: the weight-streaming kernel, within rounding of it
    y0 = torch.empty_like(y)
    kernels.check(lib.nsg_linear_fp8(
        x.data_ptr(), x.stride(0), w8.data_ptr(), w8.stride(0), s.data_ptr(), b.data_ptr(),
        y0.data_ptr(), N, M, N, K, 0, torch.cuda.current_stream().cuda_stream), "nsg_linear_fp8")
    assert ((y.float() - y0.float()).abs() <= 2.0 ** -7 * ref.abs() + 2e-3).all()
