"""Batched products of few rows, one matrix a head, against 64 bits."""
import pytest
import torch

from tests.test_kernels_gpu import DEV, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("B,K,N", [(1, 16, 8), (3, 264, 40), (16, 512, 128), (40, 1024, 136), (130, 64, 24)])
def test_heads(ops, M, B, K, N):
    """Both sides token by token, as the mixer has them. K additions in 32-bit and one rounding to bfloat16."""
    a = rnd(M, B, K + 8, dtype=BF, seed=1)[:, :, :K].transpose(0, 1)
    w = rnd(B, K, N, dtype=BF, seed=2)
    wide = torch.full((M, B, N + 3), 7.0, dtype=BF, device=DEV)
    assert ops.lib.ra_gemm_heads_fits(B, M, N, K)
    out = ops.batched_product(a, w, out=wide[:, :, :N].transpose(0, 1))
    want = a.double() @ w.double()
    bound = 2.0 ** -8 * want.abs() + K * 2.0 ** -24 * (a.double().abs() @ w.double().abs())
    assert bool(((out.double() - want).abs() <= bound).all()) and bool((wide[:, :, N:] == 7.0).all())
    assert torch.equal(ops.batched_product(a, w), out)


def test_heads_that_go_to_the_library(ops):
    fits = ops.lib.ra_gemm_heads_fits
    assert not fits(4, 9, 8, 64) and not fits(4, 8, 12, 64) and not fits(4, 8, 8, 60) and not fits(4, 8, 8, 1032)
    flat, w = rnd(1 + 2 * 3 * 64, dtype=BF, seed=3), rnd(2, 64, 16, dtype=BF, seed=4)
    a = flat[1:].view(2, 3, 64)                                    # not 16-byte aligned
    torch.testing.assert_close(ops.batched_product(a, w).double(), a.double() @ w.double(), atol=0.1, rtol=2e-2)
