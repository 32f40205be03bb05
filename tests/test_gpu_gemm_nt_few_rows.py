"""The 32-bit product at few rows: tiles of 32 x 32 and 64 x 64 whose steps of K overlap."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 16, 63, 64, 65, 128, 191, 192, 256, 320, 1000])
def test_few_rows_at_the_edges_of_tiles_and_steps(K):
    """No whole step of 64, one, an odd and an even number, with and without a rest, at rows and columns around a wavefront's half of a tile: a
    chain of K fused multiply-adds is off by at most K 2^-24 times the sum of the magnitudes (the first order of the bound), and a row alone
    has the bits that it has in a batch."""
    from ginfer_amd.kernels import ops
    g = torch.Generator().manual_seed(K)
    for M, N in ((1, 16), (15, 33), (17, 31), (32, 96), (33, 15), (64, 1500), (65, 40)):
        a, w, b = (torch.randn(s, generator=g).cuda() for s in ((M, K), (N, K), (N,)))
        got = ops.gemm_nt(a, w, b)
        want = a.double() @ w.double().t() + b.double()
        bound = (K + 2) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().t() + b.double().abs()) * 1.01
        assert bool(((got.double() - want).abs() <= bound).all()), (M, N)
        for r in {0, M // 2, M - 1}:
            assert torch.equal(ops.gemm_nt(a[r:r + 1], w, b)[0], got[r]), (M, N, r)


def test_one_row_of_any_stride_is_taken_by_the_bfloat16_product():
    """A single row has no next one: a stride beyond what offsets between rows may be is not looked at."""
    from ginfer_amd.kernels import ops
    a, w = torch.randn((1, 128), device="cuda").bfloat16(), torch.randn((48, 128), device="cuda").bfloat16()
    far = a.as_strided((1, 128), (1 << 28, 1))
    assert ops.gemm_skinny_supported(far, w)
    assert torch.equal(ops.gemm_skinny(far, w), ops.gemm_skinny(a, w))
