"""The recurrences by chunks of rows on the matrix cores (bf16, requests of 16 rows and more) against the stand-ins that
walk the rows, at the edges of chunks and halves, of tiles of channels and columns, of runs of chunks and groups of requests,
with decays from one to zero, and with rows that begin at unaligned addresses."""
import pytest
import torch

from tests.test_kofipel_gpu import DEV, ops, ref, rnd, state_step  # noqa: F401

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
    (2, 1, 66, 34, [40], 2), (8, 2, 128, 64, [9, 40] * 35, 0)])
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
