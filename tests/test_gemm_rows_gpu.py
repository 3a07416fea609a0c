"""Products of 17 to 64 rows whose W is streamed through LDS: plain, gated and in pieces of K."""
import pytest
import torch

from tests.test_kernels_gpu import ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
CUS = [256, 3]                   # with few CUs the widest tiles are chosen, with many the narrowest


@pytest.mark.parametrize("cus", CUS)
@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(1, 128), (48, 384), (130, 1280), (1000, 640), (2049, 256), (388, 12288)])
def test_rows_against_64_bits(ops, monkeypatch, M, N, K, cus):
    """fp32 results: K additions in some order, K 2^-24 of the sum of magnitudes at the most; bfloat16: one rounding more."""
    monkeypatch.setattr(ops, "cu_count", cus)
    x, w = rnd(M, K, dtype=BF, seed=1), rnd(2 * N, K, dtype=BF, seed=2, scale=0.2)
    want = x.double() @ w.double().t()
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-30
    y = ops._linear_by("rows", x, w, torch.float32)
    assert bool(((y.double() - want).abs() <= bound).all())
    z = ops._linear_by("rows", x, w, BF)
    assert torch.equal(z, y.to(BF))                                        # the same sums, rounded
    g, u = y[:, :N].double(), y[:, N:].double()
    gated = ops._gated_by("rows", x, w)
    want = g * torch.sigmoid(g) * u
    assert bool(((gated.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * K ** 0.5 * (1 + u.abs())).all())
    for pieces in (2, 3, 8):
        if K % (128 * pieces) == 0:
            shares = ops._split_product(x, w, pieces).tensor
            assert tuple(shares.shape) == (pieces, M, 2 * N)
            part = K // pieces
            for i in range(pieces):
                a, b = x[:, i * part:(i + 1) * part].double(), w[:, i * part:(i + 1) * part].double()
                assert bool(((shares[i].double() - a @ b.t()).abs() <= K * 2.0 ** -24 * (a.abs() @ b.abs().t()) + 1e-30).all())


def test_rows_that_are_not_taken(ops):
    fits = ops.lib.ra_gemm_rows_fits
    assert fits(17, 8, 128) and fits(64, 8, 128) and not fits(16, 8, 128) and not fits(65, 8, 128) and not fits(32, 8, 192)
    assert ops.route_gated(64, 12288, 4096) == "rows" and ops.route_linear(64, 151936, 4096, torch.float32) == "rows"
    assert ops.route_linear(64, 6144, 4096, BF) != "rows" and ops.route_gated(65, 12288, 4096) != "rows"
    # operands that are not 16-byte aligned go to a product that takes them
    flat = rnd(1 + 32 * 256, dtype=BF, seed=3)
    x, w = flat[1:].view(32, 256), rnd(96, 256, dtype=BF, seed=4)
    want = (x.double() @ w.double().t()).float()
    torch.testing.assert_close(ops._linear_by("rows", x, w, BF).float(), want, atol=0.2, rtol=2e-2)
    torch.testing.assert_close(ops._linear_by("rows", x, w, torch.float32), want, atol=2e-3, rtol=1e-4)
    g, u = want[:, :48], want[:, 48:]
    torch.testing.assert_close(ops._gated_by("rows", x, w).float(), g * torch.sigmoid(g) * u, atol=1.0, rtol=3e-2)
