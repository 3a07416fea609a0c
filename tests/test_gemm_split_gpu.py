"""float32 products of many rows from the operands' bfloat16 parts."""
import pytest
import torch

from tests.test_kernels_gpu import ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


def by_parts(ops, x, w):
    return ops._linear_by_parts(x, w)


@pytest.mark.parametrize("M", [1, 63, 64, 65, 127, 129, 300])
@pytest.mark.parametrize("N,K", [(4, 32), (128, 64), (132, 96), (260, 544), (1000, 4096), (384, 2080)])
def test_products_from_parts(ops, M, N, K):
    """Against 64 bits: one rounding in 16 columns and what the products of parts leave out, 3 x 2^-24 of each, with the
    matrix unit's own sums of 16 taken for two roundings: (K / 16 + 8) 2^-23 of the sum of magnitudes."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    x[:, ::7] *= 300.0
    want = x.double() @ w.double().t()
    bound = (K / 16 + 8) * 2.0 ** -23 * (x.double().abs() @ w.double().abs().t())
    assert bool(((by_parts(ops, x, w).double() - want).abs() <= bound).all())


@pytest.mark.parametrize("M,K", [(40, 256), (200, 64)])
def test_products_from_parts_of_values_that_have_none(ops, M, K):
    """Infinite values and no numbers come out as a product of 32-bit multiplications gives them; very large and very
    small rows keep their accuracy."""
    x, w = rnd(M, K, seed=3), rnd(68, K, seed=4)
    x[3, 5], x[7, 9], w[11, K // 2] = float("inf"), float("nan"), -float("inf")
    x[20] = 1e36
    x[21] *= 1e-30
    x[22] *= 1e-36
    got, want = by_parts(ops, x, w).cpu(), x.cpu() @ w.cpu().t()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    both = got.isfinite()
    assert torch.equal(got[got.isinf()] > 0, want[want.isinf()] > 0)
    exact = x.cpu().double() @ w.cpu().double().t()
    bound = (K / 16 + 8) * 2.0 ** -23 * (x.cpu().double().abs() @ w.cpu().double().abs().t())
    assert bool(((got.double() - exact).abs() <= bound)[both].all())


def test_rows_are_taken_apart_in_pieces(ops, monkeypatch):
    x, w = rnd(700, 512, seed=5), rnd(516, 512, seed=6)
    whole = by_parts(ops, x, w)
    monkeypatch.setattr(ops, "SPLIT_ROWS", 128)
    torch.testing.assert_close(by_parts(ops, x, w), whole, atol=1e-4, rtol=1e-5)
