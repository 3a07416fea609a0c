"""The sampler's searches at the edges of their ranges: several workgroups a row against one, and the searches of few
passes against the distribution in 64 bits."""
import pytest
import torch

from return_amd.kernels.hip_ops import _ptr
from tests.test_kernels_gpu import DEV, ops  # noqa: F401

pytestmark = pytest.mark.gpu

KINDS = ["flat", "peaked", "very flat", "ties", "one value", "masked", "two far apart", "crowded", "all -inf", "inf"]


def _rows(V, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(len(KINDS), V, generator=g)
    x[1, torch.randint(0, V, (300,), generator=g)] = 14 + 8 * torch.rand(300, generator=g)
    x[2] *= 0.02
    x[3] = torch.randint(-2, 3, (V,), generator=g).float()
    x[4] = 1.5
    x[5, torch.rand(V, generator=g) < 0.9] = float("-inf")
    x[6] = -1e4
    x[6, V // 3], x[6, V - 1] = 3.0, 2.9
    x[7, 777:777 + 600] = 9 + torch.rand(600, generator=g)
    x[8] = float("-inf")
    x[9, 5] = float("inf")
    return x


def _options(M, seed):
    g = torch.Generator().manual_seed(seed)
    pick = lambda values, dt: torch.tensor(values, dtype=dt)[torch.randint(0, len(values), (M,), generator=g)].to(DEV)
    return (pick([0.0, 0.3, 0.7, 1.0, 1.0, 4.0], torch.float32), pick([0, 0, 0, 1, 50, 3000], torch.int32),
            pick([0.0, 0.01, 0.5, 0.9, 0.999, 1.0], torch.float32), torch.rand(M, generator=g).to(DEV))


@pytest.mark.parametrize("M", [1, 8, 9, 25, 32])
@pytest.mark.parametrize("V", [98304, 98305, 131075, 151936, 262144])
def test_several_workgroups_a_row_draw_what_one_draws(ops, V, M):
    """Whole numbers are added, and masses in the same order: the same tokens, from the same search. The
    log-probabilities' sum of exp is formed in another order (2^-24 a step of some dozens)."""
    assert ops.lib.ra_sample_scratch(M, V) > 0
    base = _rows(V, V).to(DEV)
    for seed in range(3 if M > 1 else 24):
        kinds = torch.randperm(len(KINDS), generator=torch.Generator().manual_seed(seed))
        x = base[kinds.repeat(4)[:M]].contiguous()
        t, k, p, u = _options(M, seed)
        path = [torch.full((M,), -1, dtype=torch.int32, device=DEV) for _ in range(2)]
        one = torch.empty(M, 2, dtype=torch.int32, device=DEV)
        got = ops.sample(x, t, k, p, u, path=path[0])
        ops._check(ops.lib.ra_sample_traced(_ptr(x), M, V, _ptr(t), _ptr(k), _ptr(p), _ptr(u), _ptr(one), _ptr(path[1]),
                                            None, 0, ops._stream()), "sample")
        assert got[:, 0].tolist() == one[:, 0].tolist(), (seed, [KINDS[i] for i in kinds.repeat(4)[:M]])
        assert path[0].tolist() == path[1].tolist()
        torch.testing.assert_close(got[:, 1].contiguous().view(torch.float32), one[:, 1].contiguous().view(torch.float32),
                                   atol=2e-5, rtol=1e-6, equal_nan=True)


@pytest.mark.parametrize("V", [63, 4096, 8193, 20001, 98303, 98304])
def test_kept_tokens_are_those_of_the_distribution(ops, V):
    """Every kind of row under every option: the token is where the running sum of the plain distribution (64 bits),
    in vocabulary order, passes the uniform number. 2^-24 of a weight and a running sum in float32 over runs
    of 256: 1e-4, the bound that the other tests of the sampler have."""
    from tests.plain import qwen3_plain as plain
    x = _rows(V, V) if V > 4096 else torch.randn(len(KINDS), V, generator=torch.Generator().manual_seed(V)) * torch.arange(1, 11)[:, None]
    x = x[:8]                                      # (without a finite largest logit there is no distribution)
    for seed in range(4):
        t, k, p, u = _options(8, 100 + seed)
        out = ops.sample(x.to(DEV), t, k, p, u).cpu()
        for r in range(8):
            tok = int(out[r, 0])
            if float(t[r]) == 0.0:
                assert tok == int(x[r].argmax())
                continue
            d = plain.sample_distribution(x[r], float(t[r]), int(k[r]), float(p[r])).double()
            assert d[tok] > 0, (KINDS[r], seed, tok, float(t[r]), int(k[r]), float(p[r]))
            c = d.cumsum(0)
            before = float(c[tok - 1]) if tok else 0.0
            assert before - 1e-4 <= float(u[r]) <= float(c[tok]) + 1e-4, (KINDS[r], seed, tok)


def test_captured_and_replayed(ops):
    """Several workgroups a row in a graph: every replay gives what a call gives, other logits and calls between."""
    V, M = 131072, 8
    x = torch.empty(M, V, device=DEV)
    t, k, p, u = _options(M, 5)
    t[:] = 0.8
    base = _rows(V, 3).to(DEV)
    x.copy_(base[:M])
    ops.sample(x, t, k, p, u)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.sample(x, t, k, p, u)
    for it in range(4):
        x.copy_(base[:M].roll(it, 0) * (1.0 + 0.1 * it))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.sample(x, t, k, p, u)), f"replay {it}"


@pytest.mark.parametrize("V,M", [(63, 7), (4096, 7), (20001, 7), (98304, 7), (151936, 7), (151936, 40)])
def test_log_probabilities_of_masked_rows(ops, V, M):
    """Tokens of logit -inf weigh nothing, wherever they stand: the log-probability is log_softmax's. A sum of V numbers in
    32 bits, chains of V / 1024 and a tree: (V / 1024 + 16) 2^-24, and a rounding of the logit and of the logarithm."""
    g = torch.Generator().manual_seed(V)
    x = 4 * torch.randn(M, V, generator=g)
    low = float("-inf")
    for r in range(M):
        kind = r % 7
        if kind == 0:
            x[r, torch.rand(V, generator=g) < 0.9] = low
        elif kind == 1:
            x[r, :V // 2] = low
        elif kind == 2:
            x[r, V // 2:] = low
        elif kind == 3:
            x[r, :V - 1] = low
        elif kind == 4:
            x[r, 1:] = low
        elif kind == 5:
            x[r, : V // 2] = torch.finfo(torch.float32).min
        # (kind 6: nothing masked)
    rows = x.to(DEV)
    want = torch.log_softmax(x.double(), -1)
    u = torch.rand(M, generator=g).to(DEV)
    for temperature, top_k, top_p in ((0.0, 0, 1.0), (0.8, 0, 1.0), (0.8, 0, 0.9), (0.8, 40, 0.9), (1.0, 3000, 1.0)):
        t = torch.full((M,), temperature, device=DEV)
        k = torch.full((M,), top_k, dtype=torch.int32, device=DEV)
        p = torch.full((M,), top_p, device=DEV)
        path = torch.zeros(M, dtype=torch.int32, device=DEV)
        one = torch.empty(M, 2, dtype=torch.int32, device=DEV)
        got = ops.sample(rows, t, k, p, u)
        ops._check(ops.lib.ra_sample_traced(_ptr(rows), M, V, _ptr(t), _ptr(k), _ptr(p), _ptr(u), _ptr(one), _ptr(path), None, 0,
                                            ops._stream()), "sample")
        for out in (got, one):
            tokens, logs = out[:, 0].cpu(), out[:, 1].contiguous().view(torch.float32).cpu().double()
            chosen = want[torch.arange(M), tokens]
            assert bool(chosen.isfinite().all()), tokens
            bound = (V / 1024 + 16) * 2.0 ** -24 + 2.0 ** -23 * (chosen.abs() + x.double().clamp(min=-100).abs().max())
            assert bool(((logs - chosen).abs() <= bound).all()), (logs, chosen)


def test_a_row_draws_the_same_whatever_stands_beside_it(ops):
    """Rows whose top-p boundary lies within a few roundings of a tie: K tokens of one value and a tail beyond the list, top-p
    within a rounding of m / (K + tail), so that whether m or m + 1 of them stay hangs on the tail's sum. Every number of rows
    (four, two, one workgroup a wave's run, and one block) keeps the same."""
    V, R = 151936, 96
    g = torch.Generator().manual_seed(7)
    x = (-16.01 - 0.002 * torch.arange(R))[:, None].repeat(1, V)
    m = 1.0 + torch.arange(R) % 3
    for r in range(R):
        x[r, torch.randperm(V, generator=g)[:2 + r % 3]] = 0.0       # (one more than m)
    p = (m.double() / torch.exp(x.double()).sum(-1)).float()
    assert bool((p < 1).all())
    x, p = x.to(DEV), p.to(DEV)
    t, k, u = torch.ones(R, device=DEV), torch.zeros(R, dtype=torch.int32, device=DEV), torch.full((R,), 0.999999, device=DEV)

    def draw(M):
        return [tok for i in range(0, R, M)
                for tok in ops.sample(x[i:i + M].contiguous(), t[i:i + M], k[i:i + M], p[i:i + M].contiguous(), u[i:i + M])[:, 0].tolist()]
    want = draw(1)
    for M in (8, 12, 24, 32, 48):
        assert draw(M) == want, M
