"""A norm and the convolution behind it in one kernel, for steps of single tokens: the bits of the two kernels."""
import pytest
import torch

from tests.test_kernels_gpu import DEV, ops, rnd  # noqa: F401
from tests.test_kofipel_gpu import state_step

BF = torch.bfloat16


@pytest.mark.gpu
@pytest.mark.parametrize("H,taps,n", [(4, 2, 1), (1024, 3, 3), (1028, 4, 64), (2048, 4, 2), (2052, 2, 5), (4096, 4, 8), (4092, 3, 1)])
@pytest.mark.parametrize("with_delta", [True, False])
def test_single_tokens(ops, H, taps, n, with_delta):
    slots = torch.randperm(n + 1, generator=torch.Generator().manual_seed(n)).tolist()[:n]
    w, nw, step = rnd(H, taps, seed=1, scale=0.5), 1 + rnd(H, seed=2, scale=0.1), state_step([1] * n, slots)
    h_a, tail_a = rnd(n, H, seed=3), rnd(n + 1, taps - 1, H, dtype=BF, seed=4)
    h_b, tail_b = h_a.clone(), tail_a.clone()
    for r in range(taps + 1):                                   # until the tails hold rows of these steps alone
        delta = rnd(n, H, dtype=BF, seed=5 + r) if with_delta else None
        a = ops.norm_conv(h_a, delta, nw, 1e-6, w, tail_a, step)
        x, b = torch.empty(n, H, dtype=BF, device=DEV), torch.empty(n, H, dtype=BF, device=DEV)
        ops.add_rmsnorm(h_b, delta, nw, 1e-6, x)
        ops.causal_conv(x, w, tail_b, step, b, add_input=True)
        assert torch.equal(a, b) and torch.equal(h_a, h_b) and torch.equal(tail_a, tail_b)


@pytest.mark.gpu
def test_what_goes_by_the_two_kernels(ops):
    """Steps and sizes of neither kind are left alone: None, and nothing is written."""
    h, w, nw = rnd(2, 64, seed=1), rnd(64, 4, seed=2), rnd(64, seed=3)
    one, tail = state_step([1, 1], [0, 1]), rnd(2, 3, 64, dtype=BF, seed=4)
    was = h.clone()
    assert ops.norm_conv(h, None, nw, 1e-6, w, tail, state_step([2], [0])) is None
    assert ops.norm_conv(h, None, nw, 1e-6, w, tail.float(), one) is None
    assert ops.norm_conv(h, None, nw, 1e-6, rnd(64, 5), rnd(2, 4, 64, dtype=BF), one) is None
    assert ops.norm_conv(rnd(2, 66), None, rnd(66), 1e-6, rnd(66, 4), rnd(2, 3, 66, dtype=BF), one) is None
    assert ops.norm_conv(rnd(2, 4100), None, rnd(4100), 1e-6, rnd(4100, 4), rnd(2, 3, 4100, dtype=BF), one) is None
    odd = torch.empty(129, dtype=torch.float32, device=DEV)[1:].view(2, 64).copy_(h)
    assert ops.norm_conv(odd, None, nw, 1e-6, w, tail, one) is None
    assert torch.equal(h, was)
    from return_amd.kernels.hip_ops import KernelError
    with pytest.raises(KernelError):
        ops.norm_conv(h, rnd(3, 64, dtype=BF), nw, 1e-6, w, tail, one)
    with pytest.raises(KernelError):
        ops.norm_conv(h, None, nw, 1e-6, w, tail, state_step([1, 1], [0, 2]))
