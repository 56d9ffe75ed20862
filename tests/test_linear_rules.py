"""nsg_linear_workspace_bytes: which bias layers split K.  Host only."""
import pytest

from nanosglang_amd import _native


@pytest.mark.parametrize("N,K,splits", [
    (4096, 14336, 8),        # few columns: K split over idle CUs
    (6144, 4096, 5),
    (1028, 25600, 8),
    (512, 51200, 8),
    (16384, 4096, 2),
    (16388, 4096, 1),        # more column tiles than half the CUs: no split, no memory
    (33000, 768, 1),
    (28672, 4096, 1),
    (65532, 512, 1),
])
def test_bytes_are_the_split_partials(N, K, splits):
    lib = _native.load()
    for M in (33, 64, 160):
        want = splits * M * N * 4 if splits > 1 else 0
        assert lib.nsg_linear_workspace_bytes(M, N, K, 0) == want
        assert lib.nsg_linear_workspace_bytes(M, N, K, 1) == 0          # SwiGLU
    assert lib.nsg_linear_workspace_bytes(16, N, K, 0) == 0
    assert lib.nsg_linear_workspace_bytes(161, N, K, 0) == 0


@pytest.mark.parametrize("N,K,few", [
    (4096, 14336, True), (6144, 4096, True),
    (12288, 2048, False), (8192, 3072, False), (16384, 1536, False),    # short rows
    (16384, 2048, True),                                                # 32 M elements
    (4096, 4096, None),                                                 # below 24 M
])
def test_few_rows_need_long_rows_or_more_weight(N, K, few):
    """17 - 32 rows: measured slower than the weight-streaming kernel with K under
    4096 and weights under 32 M elements."""
    lib = _native.load()
    assert (lib.nsg_linear_workspace_bytes(17, N, K, 0) > 0) == bool(few)
    assert (lib.nsg_linear_workspace_bytes(32, N, K, 0) > 0) == bool(few)
    assert (lib.nsg_linear_workspace_bytes(33, N, K, 0) > 0) == (few is not None)
