"""Kernels over rows that take 16-byte pieces where sizes and addresses allow: the same bits as element by element."""
import pytest
import torch

from tests.test_kofipel_gpu import DEV, ops, ref, rnd, state_step  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("C,q_lens", [(8, [8]), (1032, [1, 2, 3, 9]), (1024, [16, 7, 15]), (2056, [37, 1, 33])])
@pytest.mark.parametrize("with_bias", [False, True])
def test_convolution_by_pieces_has_the_bits_of_the_one_by_channels(ops, C, taps, q_lens, with_bias):
    n, T = len(q_lens), sum(q_lens)
    w = rnd(C, taps, seed=1, scale=0.5)
    bias, in_bias = (rnd(C, seed=5), rnd(C, seed=6)) if with_bias else (None, None)
    tails = [rnd(n + 1, taps - 1, C, dtype=BF, seed=2) for _ in range(2)]
    slots = list(range(n, 0, -1))
    for r in range(2):
        x = rnd(T, C, dtype=BF, seed=3 + r)
        wide = torch.zeros(T, C + 9, dtype=BF, device=DEV)
        wide[:, 1:C + 1] = x                                     # an address that is no multiple of 16 bytes
        outs = [torch.zeros(T, C, dtype=BF, device=DEV) for _ in range(2)]
        for src, tail, out in zip((x, wide[:, 1:C + 1]), tails, outs):
            ops.causal_conv(src, w, tail, state_step(q_lens, slots), out, add_input=r == 0, silu=True, bias=bias, in_bias=in_bias)
        assert torch.equal(outs[0], outs[1]) and torch.equal(tails[0], tails[1])


@pytest.mark.parametrize("T,N", [(1, 8), (3, 264), (130, 4096)])
def test_rows_by_pieces(ops, T, N):
    x, b = rnd(T, N, dtype=BF, seed=1, scale=3.0), rnd(N, seed=2)
    r = torch.relu(x.float())
    assert torch.equal(ops.relu_sq(x.clone()), (r * r).to(BF))
    assert torch.equal(ops.add_bias(x.clone(), b), (x.float() + b).to(BF))
    gu, b2 = rnd(T, 2 * N, dtype=BF, seed=3), rnd(2 * N, seed=4)
    out = torch.empty(T, N, dtype=BF, device=DEV)
    ops.silu_mul(gu, out, bias=b2)
    g, u = (gu.double() + b2.double()).chunk(2, -1)
    want = g * torch.sigmoid(g) * u
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * u.abs() + 1e-30).all())


@pytest.mark.parametrize("V", [64, 128, 256])
def test_read_outs_by_pieces(ops, V):
    """The gated norm behind the recurrence: bfloat16 rows by pieces of four have the bits of the same rows at an odd place."""
    H, D, T = 3, 64, 21
    qkv = rnd(T, 2 * H * D + H * V, dtype=BF, seed=1)
    beta, a_log, dt_bias, norm_w = rnd(T, H, dtype=BF, seed=2), rnd(H, seed=3), rnd(H * D, seed=4) - 1.0, 1 + rnd(V, seed=5, scale=0.1)
    ag = rnd(T, H * D + H * V, dtype=BF, seed=6)
    wide = torch.zeros(T, ag.shape[1] + 1, dtype=BF, device=DEV)
    wide[:, :-1] = ag
    got = []
    for src in (ag, wide[:, :-1]):
        state, out = rnd(2, H, V, D, seed=8, scale=0.3), torch.empty(T, H * V, dtype=BF, device=DEV)
        ops.delta_rule(qkv, beta, src, a_log, dt_bias, norm_w, 1e-5, state, state_step([T], [1]), out, H, H, D, V)
        got.append(out)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("H,V,parts", [(8, 64, 1), (8, 64, 8), (6, 20, 2), (6, 64, 1), (16, 64, 1), (7, 12, 1)])
def test_grouped_read_outs_by_pieces(ops, H, V, parts):
    G, D, T = H, 64, 19
    c = 2 * G * D + H * V
    qkv, gate, dt = rnd(T, c, dtype=BF, seed=1), rnd(T, H * V, dtype=BF, seed=2), rnd(T, H, dtype=BF, seed=3)
    a_log, dt_bias, skip = rnd(H, seed=4, scale=0.5) - 0.5, rnd(H, seed=5) - 1.0, 1 + rnd(H, seed=6, scale=0.3)
    norm_w = 1 + rnd(H * V, seed=7, scale=0.1)
    wide = torch.zeros(T, H * V + 1, dtype=BF, device=DEV)
    wide[:, :-1] = gate
    got = []
    for src in (gate, wide[:, :-1]):
        state, out = rnd(2, H, V, D, seed=8, scale=0.3), torch.empty(T, H * V, dtype=BF, device=DEV)
        ops.scalar_rule(qkv, dt, a_log, dt_bias, skip, src, norm_w, parts, 1e-5, state, state_step([T], [1]), out, H, G, D, V)
        got.append(out)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("T,H,S", [(1, 8, 8), (3, 2048, 32), (5, 2056, 24), (2, 4096, 32), (7, 4088, 16),       # a row a workgroup
                                   (768, 2048, 32), (769, 4096, 24), (770, 1000, 8), (771, 2056, 32)])          # four
@pytest.mark.parametrize("with_delta", [False, True])
def test_token_input_in_its_forms(ops, ref, T, H, S, with_delta):
    table = rnd(50, 2 * S + 3, dtype=BF, seed=1)
    gate, proj, w = rnd(S, H, dtype=BF, seed=2, scale=H ** -0.5), rnd(H, S, dtype=BF, seed=3), rnd(H, seed=4).abs()
    ids = torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(5)).int().to(DEV)
    delta = rnd(T, H, dtype=BF, seed=6) if with_delta else None
    a = rnd(T, H, seed=7)
    b = a.clone()
    ops.token_side(a, delta, ids, table, S + 1, gate, proj, w, 1e-5)
    ref.token_side(b, delta, ids, table, S + 1, gate, proj, w, 1e-5)
    torch.testing.assert_close(a, b, atol=1e-4, rtol=1e-4)
