"""Products of a few float32 rows, x from the cache and x in LDS, at the edges of their tiles."""
import pytest
import torch

from return_amd.kernels.hip_ops import _ptr
from tests.test_kernels_gpu import DEV, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(1, 4), (15, 252), (17, 256), (1000, 260), (33, 1004), (4096, 512), (4097, 768), (40, 1280),
                                 (65535, 8), (65537, 36), (8192, 260), (8208, 260), (24576, 4096), (24592, 4096), (4112, 300)])
def test_few_rows(ops, M, N, K):
    """Against 64 bits: a sum of K products in 32 bits, the lanes' chains of K / 64 and a tree of 64, is off by at
    most (K / 64 + 8) 2^-24 of the sum of magnitudes. The padding behind y stays as it is."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    y = torch.full((M * N + 64,), 7.0, device=DEV)
    ops._check(ops.lib.ra_gemm_nt(_ptr(x), _ptr(w), _ptr(y), M, N, K, 0, 0, ops._stream()), "gemm_nt")
    want = x.double() @ w.double().t()
    bound = (K / 64 + 8) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert bool(((y[:M * N].view(M, N).double() - want).abs() <= bound).all())
    assert bool((y[M * N:] == 7.0).all())
