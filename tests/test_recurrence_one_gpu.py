"""Steps of single tokens: the recurrence with its read-out's norm and gate in one kernel has the bits of the two kernels."""
import pytest
import torch

from tests.test_kernels_gpu import DEV, ops, rnd  # noqa: F401
from tests.test_kofipel_gpu import state_step

BF = torch.bfloat16


def run(ops, rule, H, G, D, V, n, odd):
    """Two steps in a row over slots that hold something; odd: gates at places that only the two kernels take."""
    slots = torch.randperm(n + 1, generator=torch.Generator().manual_seed(n)).tolist()[:n]
    state, outs = rnd(n + 1, H, V, D, seed=8, scale=0.3), []
    for r in range(2):
        qkv = rnd(n, 2 * (G if rule != 1 else H) * D + H * V + 8, dtype=BF, seed=10 + r)[:, :2 * (G if rule != 1 else H) * D + H * V]
        wide = torch.zeros(n, H * D + H * V + 4 + odd, dtype=BF, device=DEV)
        wide[:, :H * D + H * V] = rnd(n, H * D + H * V, dtype=BF, seed=20 + r)
        ag, z = wide[:, :H * D + H * V], rnd(n, 2 * H, dtype=BF, seed=30 + r)
        a_log, norm_w, step = rnd(H, seed=5), 1 + rnd(V, seed=7, scale=0.1), state_step([1] * n, slots)
        out = torch.empty(n, H * V, dtype=BF, device=DEV)
        if rule == 0:
            ops.delta_rule(qkv, z[:, H:], ag, a_log, rnd(H * D, seed=6) - 1.0, norm_w, 1e-5, state, step, out, H, G, D, V)
        elif rule == 1:
            ops.outer_rule(qkv, ag[:, :H * D], ag[:, H * D:], rnd(H * D, seed=6), 16.0, norm_w, 1e-5, state, step, out, H, D, V)
        else:
            ops.delta_rule_head(qkv, z[:, H:], z[:, :H], ag[:, H * D:], a_log, rnd(H, seed=6), norm_w, 1e-5, state, step, out, H, G, D, V)
        outs.append(out)
    return outs, state


@pytest.mark.gpu
@pytest.mark.parametrize("rule", [0, 1, 3])
@pytest.mark.parametrize("H,G,D,V,n", [(1, 1, 128, 128, 1), (32, 8, 128, 128, 8), (6, 3, 64, 64, 3), (5, 5, 60, 128, 2), (2, 1, 100, 64, 7), (4, 2, 68, 64, 64)])
def test_single_tokens_in_one_kernel(ops, rule, H, G, D, V, n):
    assert ops.lib.ra_delta_rule_form(D, V, 1) == 1
    (a, sa), (b, sb) = (run(ops, rule, H, G, D, V, n, odd) for odd in (0, 1))
    assert all(torch.equal(x, y) for x, y in zip(a, b)) and torch.equal(sa, sb)


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,V,n", [(1, 1, 128, 64, 1), (64, 8, 128, 64, 8), (6, 3, 64, 128, 70), (4, 1, 60, 64, 3)])
def test_scalar_rule_of_single_tokens(ops, H, G, D, V, n):
    """Read-outs that a kernel of their own norms: the same bits as from the walk (states at an odd place)."""
    got = []
    for odd in (0, 1):
        state = torch.empty((n + 1) * H * V * D + odd, device=DEV)[odd:].view(n + 1, H, V, D).copy_(rnd(n + 1, H, V, D, seed=8, scale=0.3))
        for r in range(2):
            qkv, z = rnd(n, 2 * G * D + H * V, dtype=BF, seed=10 + r), rnd(n, H * V + H, dtype=BF, seed=20 + r)
            out = torch.empty(n, H * V, dtype=BF, device=DEV)
            ops.scalar_rule(qkv, z[:, H * V:], rnd(H, seed=5), rnd(H, seed=6), rnd(H, seed=4), z[:, :H * V], 1 + rnd(H * V, seed=7, scale=0.1), 1, 1e-5,
                            state, state_step([1] * n, list(range(n))), out, H, G, D, V)
            got.append(out)
        got.append(state)
    assert all(torch.equal(a, b) for a, b in zip(got[:3], got[3:]))


def test_which_heads_go_by_one_kernel():
    """(D, V, dtype) on either side of the rule's lines."""
    from return_amd.kernels.hip_ops import load_library
    form = load_library().ra_delta_rule_form
    for D, V, dtype, want in [(128, 128, 1, 1), (128, 128, 0, 0), (130, 128, 1, 0), (132, 128, 1, 0), (56, 64, 1, 0), (60, 64, 1, 1), (128, 256, 1, 0),
                              (128, 96, 1, 0)]:
        assert form(D, V, dtype) == want, (D, V)
