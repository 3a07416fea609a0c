"""The rule that puts a mixed step's two attention kernels on two streams, on both sides of its line."""
import pytest
import torch

from tests.test_kernels_gpu import DEV, _step, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, keys, window, beside", [(1, 300, 0, False), (63, 8192, 0, False), (64, 8191, 0, False),
                                                     (64, 8192, 0, True), (64, 8300, 8192, True), (64, 8300, 100, False)])
def test_rule_and_results(ops, monkeypatch, n, keys, window, beside):
    """The kernels are the same on one stream and on two: the same bits, call after call."""
    P, Hq, Hkv, D = 16, 4, 1, 32
    need = [-(-keys // P)] * n + [7]
    starts = [sum(need[:i]) for i in range(len(need))]
    step = _step([1] * n + [90], [keys - 1] * n + [20], P, [list(range(s, s + k)) for s, k in zip(starts, need)])
    assert ops.overlap_attention is None and ops._side_by_side(step, window) is beside
    kp, vp = (rnd(sum(need), Hkv, P, D, dtype=torch.bfloat16, seed=s) for s in (1, 2))
    for it in range(3):
        q = rnd(n + 90, Hq, D, dtype=torch.bfloat16, seed=10 + it)
        outs = []
        for overlap in (None, False, True):
            monkeypatch.setattr(ops, "overlap_attention", overlap)
            o = torch.zeros_like(q)
            ops.attention(q, o, kp, vp, step, 0, D ** -0.5, window)
            outs.append(o * 1)
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), f"call {it}"
