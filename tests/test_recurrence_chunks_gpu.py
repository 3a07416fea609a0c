"""The recurrences by chunks of rows on the matrix cores (bf16, requests of 16 or 24 rows and more) against the stand-ins that
walk the rows, at the edges of chunks and halves, of tiles of channels and columns, of runs of chunks and groups of requests,
with decays from one to zero, and with rows that begin at unaligned addresses."""
import ctypes

import pytest
import torch

from return_amd.kernels.hip_ops import _ptr
from tests.test_kofipel_gpu import DEV, i32, ops, ref, rnd, state_step  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def both(ops, ref, rule, q_lens, H, G, D, V, shift=0.0, offset=0, rounds=2):
    """Two steps in a row from a state that holds something; every input is a column slice of wider rows that begins
    `offset` elements in. Sums of 32-bit products in another order: the states agree to 1e-4 (rows of a unit's size,
    up to 200 of them in sight), the outputs to bf16's rounding (2^-8) and its doubling where the norm divides."""
    n, T = len(q_lens), sum(q_lens)
    slots = torch.randperm(n + 1, generator=torch.Generator().manual_seed(n)).tolist()[:n]
    cut = lambda width, seed: rnd(T, width + 8, dtype=BF, seed=seed)[:, offset:offset + width]
    qkv, gate, beta = cut(2 * G * D + H * V, 1), cut(H * V, 2), cut(H, 3)
    per = H * D if rule in ("channel", "outer") else H
    a, a_log = cut(per + (H * V if rule == "channel" else 0), 4), rnd(H, seed=5, scale=0.5) - 1.0
    bias, norm_w = rnd(per, seed=6) - 1.0 + shift, 1 + rnd(V, seed=7, scale=0.1)
    states = [rnd(n + 1, H, V, D, seed=8, scale=0.3)]
    states.append(states[0].clone())
    for _ in range(rounds):
        step, outs = state_step(q_lens, slots), []
        for o, state in zip((ops, ref), states):
            out = torch.empty(T, H * V, dtype=BF, device=DEV)
            if rule == "channel":
                o.delta_rule(qkv, beta, a, a_log, bias, norm_w, 1e-5, state, step, out, H, G, D, V)
            elif rule == "head":
                o.delta_rule_head(qkv, beta, a, gate, a_log, bias, norm_w, 1e-5, state, step, out, H, G, D, V)
            elif rule == "outer":
                o.outer_rule(qkv, a, gate, 2.0 - bias, 4.0, norm_w, 1e-5, state, step, out, H, D, V)
            else:
                o.scalar_rule(qkv, a, a_log, bias, norm_w[:1].expand(H).contiguous(), gate, norm_w.repeat(H), 1, 1e-5, state,
                              step, out, H, G, D, V)
            outs.append(out.float())
        torch.testing.assert_close(outs[0], outs[1], atol=2e-2, rtol=2e-2)
        torch.testing.assert_close(states[0], states[1], atol=1e-4, rtol=1e-4)


RULES = ["channel", "head", "outer", "scalar"]


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("H,G,D,V,q_lens,offset", [
    (2, 1, 128, 128, [16, 17, 15, 1, 31], 0), (3, 3, 64, 16, [32, 33, 2, 64], 0), (2, 2, 80, 40, [65, 96, 97], 0),
    (4, 2, 24, 8, [127], 8), (2, 1, 128, 130, [47, 16], 0), (2, 2, 33, 17, [48, 20], 1), (1, 1, 1, 1, [18], 3),
    (2, 1, 66, 34, [40], 2), (8, 2, 128, 64, [9, 40] * 35, 0), (2, 1, 128, 128, [24, 23, 31, 32], 0), (2, 2, 48, 24, [25, 26], 0),
    (96, 1, 128, 128, [25] * 33, 0)])
def test_against_the_walk(ops, ref, rule, H, G, D, V, q_lens, offset):
    both(ops, ref, rule, q_lens, H, H if rule == "outer" else G, D, V, offset=offset)


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("shift", [-12.0, 4.0, 40.0], ids=["no_decay", "strong", "to_zero"])
def test_decays_far_from_one(ops, ref, rule, shift):
    """The quotients of decay products: near one, below what a half may lose (pairs formed one by one), and zero."""
    both(ops, ref, rule, [70, 16], 2, 2, 96, 32, shift=shift)


@pytest.mark.parametrize("rule", ["head", "scalar"])
def test_runs_of_chunks(ops, ref, rule):
    """More chunks than the scratch holds at once: the state passes from run to run. Checked against the same rows in
    steps of 480, whose chunks fit."""
    H, G, D, V, T = 96, 1, 128, 128, 960
    qkv, gate = rnd(T, 2 * G * D + H * V, dtype=BF, seed=1), rnd(T, H * V, dtype=BF, seed=2)
    a, beta, a_log, bias = rnd(T, H, dtype=BF, seed=3), rnd(T, H, dtype=BF, seed=4), rnd(H, seed=5) - 1.0, rnd(H, seed=6) - 2.0
    ones, got = torch.ones(H * V, device=DEV), []
    for cut in (T, T // 2):
        state, outs = torch.zeros(1, H, V, D, device=DEV), []
        for at in range(0, T, cut):
            step, rows = state_step([cut], [0]), slice(at, at + cut)
            out = torch.empty(cut, H * V, dtype=BF, device=DEV)
            if rule == "head":
                ops.delta_rule_head(qkv[rows], beta[rows], a[rows], gate[rows], a_log, bias, ones[:V], 1e-5, state, step, out, H, G, D, V)
            else:
                ops.scalar_rule(qkv[rows], a[rows], a_log, bias, ones[:H], gate[rows], ones, 1, 1e-5, state, step, out, H, G, D, V)
            outs.append(out)
        got.append((torch.cat(outs), state))
    assert ops.lib.ra_recurrence_scratch((__import__("ctypes").c_int * 1)(T), 1, H, D, V, 3) < 30 * H * 17600
    torch.testing.assert_close(got[0][0], got[1][0], atol=0, rtol=0)        # the cut falls on a chunk's border
    torch.testing.assert_close(got[0][1], got[1][1], atol=0, rtol=0)


# ------------------------------------------------------------------ read-outs and states as they come, before the norm
NUMBER = {"channel": 0, "outer": 1, "scalar": 2, "head": 3}


def drawn(rule, q_lens, H, G, D, V, seed):
    """A layer's inputs as the designs have them: rows behind a SiLU, decays by the package's own laws (near one)."""
    T, law = sum(q_lens), torch.Generator(device=DEV).manual_seed(seed)
    uniform = lambda n, lo, hi: lo + (hi - lo) * torch.rand(n, generator=law, device=DEV)
    per = H * D if rule in ("channel", "outer") else H
    qkv = rnd(T, 2 * G * D + H * V, seed=seed)
    return dict(qkv=(qkv if rule == "outer" else torch.nn.functional.silu(qkv)).to(BF), b=rnd(T, H, dtype=BF, seed=seed + 1, scale=0.5),
                a=rnd(T, per + (H * V if rule == "channel" else 0), dtype=BF, seed=seed + 2, scale=0.5), a_log=uniform(H, 0.02, 1).log(),
                bias=uniform(per, 2, 5) if rule == "outer" else uniform(per, -4, -1), rate=1 / 16)


def recur(ops, rule, x, state, q_lens, H, G, D, V, chunks):
    """Read-outs [T, H V] of the step, by chunks of rows or row by row; the state moves on."""
    T, n, number = sum(q_lens), len(q_lens), NUMBER[rule]
    step = state_step(q_lens, list(range(n)))
    o, out = torch.empty(T, H * V, device=DEV), torch.empty(T, H * V, dtype=BF, device=DEV)
    rows = (ctypes.c_int * n)(*q_lens) if chunks else None
    floats = ops.lib.ra_recurrence_scratch(rows, n, H, D, V, number) if chunks else 0
    assert not chunks or floats > 0
    ws = torch.empty(floats, device=DEV) if chunks else None
    ones, gate = torch.ones(H * V, device=DEV), torch.zeros(T, H * V, dtype=BF, device=DEV)
    end = (_ptr(state), _ptr(step.cu_q), _ptr(step.slot_ids), _ptr(o), _ptr(out), n, T, max(q_lens), rows, _ptr(ws), floats, H)
    qkv, a, lib, last = (_ptr(x["qkv"]), x["qkv"].stride(0)), (_ptr(x["a"]), x["a"].stride(0)), ops.lib, (D, V, 1, ops._stream())
    b, g, law = (_ptr(x["b"]), H), (_ptr(gate), H * V), (_ptr(x["a_log"]), _ptr(x["bias"]))
    if rule == "channel":
        code = lib.ra_delta_rule(*qkv, *b, *a, *law, _ptr(ones), 1e-5, *end, G, *last)
    elif rule == "head":
        code = lib.ra_delta_rule_head(*qkv, *b, *a, *g, *law, _ptr(ones), 1e-5, *end, G, *last)
    elif rule == "outer":
        code = lib.ra_outer_rule(*qkv, *a, *g, law[1], x["rate"], _ptr(ones), 1e-5, *end, *last)
    else:
        code = lib.ra_scalar_rule(*qkv, *a, *g, *law, _ptr(ones), _ptr(ones), 1, 1e-5, *end, G, *last)
    ops._check(code, rule)
    return o


def recur64(rule, x, state, q_lens, H, G, D, V):
    """The same in 64 bits, row by row."""
    f = {k: v.double() if torch.is_tensor(v) else v for k, v in x.items()}
    T, per = sum(q_lens), D if rule in ("channel", "outer") else 1
    q, k, v = (t.view(T, -1, w) for t, w in zip(f["qkv"].split([G * D, G * D, H * V], 1), (D, D, V)))
    if rule in ("channel", "head"):
        q, k = (t * torch.rsqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
    q, k = (t.repeat_interleave(H // G, 1) for t in (q * (1.0 if rule == "scalar" else D ** -0.5), k))
    a = (f["a"][:, :H * per] + f["bias"]).view(T, H, per)
    step = torch.logaddexp(a, torch.zeros_like(a))
    decay = torch.sigmoid(a) ** f["rate"] if rule == "outer" else torch.exp(-f["a_log"].exp()[:, None] * step)
    k = k * step if rule == "scalar" else k
    beta, S, out, at = torch.sigmoid(f["b"]), state.double(), torch.empty(T, H, V, dtype=torch.float64, device=DEV), 0
    for s, n in enumerate(q_lens):
        for t in range(at, at + n):
            M = S[s] * decay[t][:, None]
            u = v[t]
            if rule in ("channel", "head"):
                u = beta[t][:, None] * (u - (M @ k[t][:, :, None])[..., 0])
            S[s] = M + u[:, :, None] * k[t][:, None]
            out[t] = (S[s] @ q[t][:, :, None])[..., 0]
        at += n
    return out.view(T, H * V), S


@pytest.mark.parametrize("rule,H,G,D,V", [("channel", 16, 4, 128, 128), ("head", 16, 4, 128, 128), ("outer", 16, 16, 128, 128),
                                          ("scalar", 32, 8, 128, 64)])
@pytest.mark.parametrize("q_lens", [[24] * 4, [33] * 3, [48] * 3, [250] * 2, [700]], ids=str)
def test_no_further_from_64_bits_than_the_walk(ops, rule, H, G, D, V, q_lens):
    """Over the designs' decays the chunks' read-outs and states are at most as far from the 64-bit recurrence as those of the
    kernels that go row by row (three draws together, 2 % for their scatter)."""
    far = {True: [0.0, 0.0], False: [0.0, 0.0]}
    for seed in (1, 101, 201):
        x = drawn(rule, q_lens, H, G, D, V, seed)
        start = torch.zeros(len(q_lens), H, V, D, device=DEV)
        want = recur64(rule, x, start, q_lens, H, G, D, V)
        for chunks in (True, False):
            state = start.clone()
            got = recur(ops, rule, x, state, q_lens, H, G, D, V, chunks), state
            for i in (0, 1):
                far[chunks][i] += float((got[i].double() - want[i]).norm() / want[i].norm()) / 3
    assert far[True][0] <= 1.02 * far[False][0] and far[True][1] <= 1.02 * far[False][1], far


def strange(x, what, rule, row, value, H, G, D, V):
    """The inputs with one number of one row replaced."""
    x = dict(x)
    name, column = {"q": ("qkv", 7), "k": ("qkv", G * D + 7), "v": ("qkv", 2 * G * D + 3), "decay": ("a", 7 if rule in ("channel", "outer") else 1),
                    "beta": ("b", 1)}[what]
    x[name] = x[name].clone()
    x[name][row, column] = value
    return x


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("what", ["q", "k", "v", "decay", "beta"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 1e30], ids=str)
def test_rows_before_one_that_is_no_number(ops, rule, what, value):
    """An infinity, NaN or very large number in one row: what the walk gives as a number is one by chunks too, rows before it
    and the other request among it (there the same: 32-bit sums of at most 90 rows of a unit's size in another order); what the
    walk does not, neither do the chunks."""
    H = G = 2
    q_lens = [90, 40]
    for D, V in ((64, 32), (128, 40)):
        base = drawn(rule, q_lens, H, G, D, V, 5)
        for row in (0, 3, 15, 16, 30, 31, 33, 50, 89):
            x = strange(base, what, rule, row, value, H, G, D, V)
            start = rnd(2, H, V, D, seed=8, scale=0.3)
            both = []
            for chunks in (True, False):
                state = start.clone()
                both.append((recur(ops, rule, x, state, q_lens, H, G, D, V, chunks), state))
            for got, want in zip(*both):
                assert torch.equal(want.isfinite(), got.isfinite()), row
            (o, state), (o_walk, state_walk) = both
            clear = torch.tensor([i < row or i >= q_lens[0] for i in range(sum(q_lens))], device=DEV)
            assert bool(o[clear].isfinite().all()), row
            torch.testing.assert_close(o[clear], o_walk[clear], atol=1e-4, rtol=1e-4)
            torch.testing.assert_close(state[1], state_walk[1], atol=1e-4, rtol=1e-4)
