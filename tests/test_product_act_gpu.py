"""A product and the row kernel behind it as one kernel: bit for bit what the two give, at edges of tiles, rounds and spans of K."""
import pytest
import torch

from tests.test_kernels_gpu import ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def sweep(ops, x, w, gated, act, limit, slope, bias):
    M, K, N = x.shape[0], x.shape[1], w.shape[0] // (2 if gated else 1)
    y = torch.full((M, N), float("nan"), dtype=BF, device=x.device)
    ops._check(ops.lib.ra_gemm_sweep_act_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, 1 if gated else 0, ops.cu_count, act, limit, slope,
                                              None if bias is None else bias.data_ptr(), ops._stream()), "")
    return y


def two(ops, x, w, gated, act, limit, slope, bias, product):
    y = product(x, w)
    if not gated:
        return ops.relu_sq(y) if act == 2 else ops.add_bias(y, bias)
    out = torch.empty(y.shape[0], y.shape[1] // 2, dtype=BF, device=x.device)
    if act == 1:
        ops.gated_rows(y, out, "clamped", limit, slope)
    else:
        ops.silu_mul(y, out, bias=bias)
    return out


FORMS = [(False, 2, False), (False, 0, True), (True, 0, True), (True, 1, False)]


@pytest.mark.parametrize("gated,act,biased", FORMS)
@pytest.mark.parametrize("M", [1, 3, 16])
@pytest.mark.parametrize("N,K", [(24, 64), (256, 1536), (4104, 512), (520, 4096), (264, 8192), (5000, 2048), (2056, 12296), (300, 16384)])
def test_few_rows(ops, gated, act, biased, M, N, K):
    """One round of columns and more, one span of K, two that are held, several; columns that end inside a tile."""
    x, w = rnd(M, K, dtype=BF, seed=M), rnd((2 if gated else 1) * N, K, dtype=BF, seed=N, scale=2.0 * K ** -0.5)
    bias = rnd(w.shape[0], seed=5) if biased else None
    got = sweep(ops, x, w, gated, act, 1.5, 1.702, bias)
    # (each half of a gated product has its sums formed as the plain product's are)
    want = two(ops, x, w, gated, act, 1.5, 1.702, bias, lambda x, w: ops._linear_by("sweep", x, w, BF))
    assert torch.equal(got, want)


@pytest.mark.parametrize("gated,act,biased", FORMS)
@pytest.mark.parametrize("tile", [0, 3, 6, 9, 11])
@pytest.mark.parametrize("M,N,K", [(65, 8, 64), (300, 264, 192)])
def test_many_rows(ops, gated, act, biased, tile, M, N, K):
    x, w = rnd(M, K, dtype=BF, seed=M), rnd((2 if gated else 1) * N, K, dtype=BF, seed=N, scale=2.0 * K ** -0.5)
    bias = rnd(w.shape[0], seed=5) if biased else None
    got = ops._block_product(x, w, gated, tile + 16, BF, act, 1.5, 1.702, bias)
    want = two(ops, x, w, gated, act, 1.5, 1.702, bias, lambda x, w: ops._block_product(x, w, False, tile + 16, BF))
    assert torch.equal(got, want)


def test_entries_at_sizes_of_either_way(ops):
    """The public entries, where one kernel forms both and where two do (17 to 64 rows, operands at odd places)."""
    w, b = rnd(4096, 1024, dtype=BF, seed=1, scale=0.05), rnd(4096, seed=2)
    for M in (2, 40, 600):
        for odd in (0, 1):
            x = torch.empty(M * 1024 + odd, dtype=BF, device=w.device)[odd:].view(M, 1024).copy_(rnd(M, 1024, dtype=BF, seed=M))
            y = x.double() @ w.double().t()
            torch.testing.assert_close(ops.linear_bias(x, w, b).double(), y + b, atol=2e-2, rtol=2e-2)
            torch.testing.assert_close(ops.linear_relu_sq(x, w).double(), y.clamp(min=0) ** 2, atol=4e-2, rtol=3e-2)
            g, u = (y + b)[:, :2048], (y + b)[:, 2048:]
            torch.testing.assert_close(ops.linear_gated_bias(x, w, b).double(), g * torch.sigmoid(g) * u, atol=6e-2, rtol=3e-2)
            g, u = y[:, :2048].clamp(max=1.5), y[:, 2048:].clamp(-1.5, 1.5)
            torch.testing.assert_close(ops.linear_clamped(x, w, 1.5).double(), g * torch.sigmoid(1.702 * g) * (u + 1), atol=6e-2, rtol=3e-2)


def test_what_is_refused(ops):
    from return_amd.kernels.hip_ops import KernelError
    x, w = rnd(2, 64, dtype=BF), rnd(32, 64, dtype=BF)
    with pytest.raises(KernelError):
        ops.linear_bias(x, w, torch.zeros(31, device=x.device))
    with pytest.raises(KernelError):
        ops.linear_bias(x, rnd(32, 72, dtype=BF), torch.zeros(32, device=x.device))
    with pytest.raises(KernelError):
        ops.linear_clamped(x, w, 0.0)
    for gated, act, limit in [(1, 2, 0.0), (0, 1, 1.0), (1, 1, 0.0), (0, 3, 0.0)]:
        assert ops.lib.ra_gemm_sweep_act_bf16(x.data_ptr(), w.data_ptr(), x.data_ptr(), 2, 16, 64, gated, 256, act, limit, 1.0, None, ops._stream()) != 0
