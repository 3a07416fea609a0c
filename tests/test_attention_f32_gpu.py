"""float32 attention by the 32-bit matrix instructions (prompts) and with all loads of a pass in flight (single tokens)."""
import pytest
import torch

from tests.test_kernels_gpu import _step, ops, ref, rnd, tol  # noqa: F401

pytestmark = pytest.mark.gpu


F32_ATTN = [  # Hq, Hkv, D, P, [(q_len, q_start)], window, keep_first
    (4, 2, 64, 16, [(63, 0), (64, 0), (65, 0), (1, 15), (1, 16), (2, 63)], 0, 0),
    (4, 1, 128, 16, [(129, 0), (1, 127), (1, 128), (70, 190), (1, 0)], 0, 0),
    (3, 3, 128, 5, [(200, 31), (1, 400), (3, 0)], 70, 0),
    (2, 1, 64, 16, [(130, 300), (1, 2000), (1, 260)], 100, 33),
    (2, 2, 128, 64, [(5, 1000), (1, 1), (1, 3000)], 0, 0),
]


@pytest.mark.parametrize("Hq,Hkv,D,P,segs,window,keep", F32_ATTN)
@pytest.mark.parametrize("extras", [False, True])
def test_attention_f32(ops, ref, Hq, Hkv, D, P, segs, window, keep, extras):
    need = [-(-(a + b) // P) for a, b in segs]
    perm = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(5)).tolist()
    unseen = perm.pop()
    pages_of = [[perm.pop() for _ in range(k)] for k in need]
    step = _step([s[0] for s in segs], [s[1] for s in segs], P, pages_of)
    kp, vp = rnd(sum(need) + 1, Hkv, P, D, seed=51), rnd(sum(need) + 1, Hkv, P, D, seed=52)
    kp[unseen], vp[unseen] = float("nan"), float("nan")
    q = rnd(sum(s[0] for s in segs), Hq, D, seed=53)
    kw = dict(keep_first=keep)
    if extras:
        kw.update(head_scale=(1 + rnd(Hq, seed=54, scale=0.2)).abs(), softcap=20.0, sink_logit=rnd(Hq, seed=55), out_scale=0.5)
    a, b = torch.zeros_like(q), torch.zeros_like(q)
    ops.attention(q, a, kp, vp, step, 0, D ** -0.5, window, **kw)
    ref.attention(q, b, kp, vp, step, 0, D ** -0.5, window, **kw)
    torch.testing.assert_close(a, b, **tol(torch.float32))


@pytest.mark.parametrize("at", [0, 40, 64, 129])
def test_a_value_that_is_no_number_reaches_no_row_before_it(ops, ref, at):
    T, P, D = 130, 16, 64
    step = _step([T], [0], P, [list(range(9))])
    kp, vp, q = rnd(9, 1, P, D, seed=1), rnd(9, 1, P, D, seed=2), rnd(T, 2, D, seed=3)
    want = torch.zeros_like(q)
    ref.attention(q, want, kp, vp, step, 0, 0.125, 0)
    vp.view(-1, D)[at, 5] = float("nan")
    out = torch.zeros_like(q)
    ops.attention(q, out, kp, vp, step, 0, 0.125, 0)
    torch.testing.assert_close(out[:at], want[:at], **tol(torch.float32))
    assert bool(out[at:, :, 5].isnan().all())
    others = [i for i in range(D) if i != 5]
    torch.testing.assert_close(out[at:, :, others], want[at:, :, others], **tol(torch.float32))
