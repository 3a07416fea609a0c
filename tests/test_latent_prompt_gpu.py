"""Attention of whole prompts over latent rows with the heads' keys and values formed, against 64 bits, and where it is taken."""
import types

import pytest
import torch

from tests.test_kofipel_gpu import DEV, i32, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def prompt_step(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    tiles = sorted(((i, o) for i, n in enumerate(lens) for o in range(0, n, 128)), key=lambda t: -t[1])
    return types.SimpleNamespace(prefill_tiles={128: i32(tiles)}, n_tokens=cu[-1], n_decode=0, n_prefill_tokens=cu[-1],
                                 q_starts=[0] * len(lens), cu_q=i32(cu), cu_q_host=cu, max_q_len=max(lens))


@pytest.mark.parametrize("H,R", [(8, 64), (3, 64), (16, 0), (5, 0)])
@pytest.mark.parametrize("lens", [[2], [31, 2, 33], [64, 65, 127], [128, 129, 300]])
@pytest.mark.parametrize("extras", [False, True])
def test_whole_prompts_with_formed_keys(ops, H, R, lens, extras):
    """Results are bfloat16 (2^-9 of a value), the weights carry 16 bits and the scores 32-bit sums of bfloat16 products:
    bounded by one more rounding than the result's, 2^-8 of the largest value a row could have."""
    D = Dv = 128
    T, scale = sum(lens), 0.06
    q = rnd(T, H * (D + R) + 16, dtype=BF, seed=1)[:, 8:8 + H * (D + R)]
    kv = rnd(T, H * (D + Dv), dtype=BF, seed=2)
    pool = rnd(T // 16 + 3, 1, 16, R, dtype=BF, seed=3) if R else torch.empty(1, 1, 16, 0, dtype=BF, device=DEV)
    slots = torch.randperm((T // 16 + 3) * 16, generator=torch.Generator().manual_seed(4))[:T].int().to(DEV)
    angles = rnd(max(lens), 32, seed=5, scale=3.0)
    cos, sin = (angles.cos().contiguous(), angles.sin().contiguous()) if R and extras else (None, None)
    sink = rnd(H, seed=6, scale=4.0) if extras else None
    gate = rnd(T, H + 8, dtype=BF, seed=7)[:, 8:] if extras else None
    step = prompt_step(lens)
    out = torch.full((T, H * Dv), float("nan"), dtype=BF, device=DEV)
    ops.attention_latent_prompt(q, kv, D, R, Dv, pool, slots, cos, sin, step, scale, sink, gate, out)
    for a, b in zip(step.cu_q_host, step.cu_q_host[1:]):
        n = b - a
        qq = q[a:b].double().view(n, H, D + R).transpose(0, 1).clone()
        if cos is not None:
            c, s, x, y = cos[:n].double(), sin[:n].double(), qq[..., D:D + 32].clone(), qq[..., D + 32:].clone()
            qq[..., D:D + 32], qq[..., D + 32:] = (x * c - y * s).to(BF).double(), (y * c + x * s).to(BF).double()
        k, v = (kv[a:b, i * H * D:(i + 1) * H * D].double().view(n, H, D).transpose(0, 1) for i in (0, 1))
        if R:
            k = torch.cat([k, pool.view(-1, R)[slots[a:b].long()].double().expand(H, n, R)], -1)
        s = (qq @ k.transpose(1, 2) * scale).masked_fill(torch.ones(n, n, device=DEV, dtype=torch.bool).triu(1), -float("inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(H, n, 1)], -1)
        want = (s.softmax(-1)[..., :n] @ v).transpose(0, 1)
        if gate is not None:
            want = want * torch.sigmoid(gate[a:b].double())[..., None]
        got = out[a:b].double().view(n, H, Dv)
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs().amax(-1, keepdim=True) + 1e-6).all())


@pytest.mark.parametrize("direct,gate,window", [(False, True, None), (True, False, None), (False, False, 60)])
def test_the_mixer_gives_the_same_either_way(ops, direct, gate, window):
    """A step of whole prompts by formed keys and by the latents themselves: the same up to the roundings of bfloat16 keys,
    queries and values (2^-8 of the result's size each); portions and prompts beyond a window go by the latents."""
    from return_amd.parts.attention import LatentAttention
    from return_amd.parts.runtime import Runtime
    W, H, D, R, Dv, Q, C = 256, 8, 128, 0, 128, 96, 128
    params = {"hidden_size": W, "num_heads": H, "head_dim": D, "rot_dim": R, "value_dim": Dv, "q_rank": Q, "kv_rank": C,
              "scale": D ** -0.5, "eps": 1e-6, "position": None, "sink": True, "gate": gate, "window": window, "direct_q": direct}
    tensors = {}
    for i, (name, shape) in enumerate(LatentAttention.tensor_shapes(params).items()):
        tensors[name] = (torch.ones(shape) if name.endswith("norm") else rnd(*shape, seed=i, scale=shape[-1] ** -0.5).cpu())
    mixer = LatentAttention(params, tensors, Runtime(DEV, "bfloat16"))
    assert mixer.w_ukv is not None and 128 in mixer.step_needs()["prefill_tile_rows"]
    lens = [50, 2, 37]
    step = prompt_step(lens)
    T, n = sum(lens), len(lens)
    pages = [-(-q // 16) for q in lens]
    cu_pages = [0]
    for p in pages:
        cu_pages.append(cu_pages[-1] + p)
    slots = [(cu_pages[i] + j // 16) * 16 + j % 16 for i, q in enumerate(lens) for j in range(q)]
    rows = ops.latent_prefill_tile_rows(H, C, R, BF)[0]
    step.prefill_tiles[rows] = i32([(i, o) for i, q in enumerate(lens) for o in range(0, q, rows)])
    step.groups = [types.SimpleNamespace(slot_mapping=i32(slots), page_table=i32(list(range(cu_pages[-1]))), cu_pages=i32(cu_pages),
                                         kv_start=i32([0] * n))]
    step.positions, step.q_start, step.n_seqs = i32([j for q in lens for j in range(q)]), i32([0] * n), n
    step.q_lens, step.all_decode = lens, False
    cache = types.SimpleNamespace(group=0, k_pool=torch.empty(cu_pages[-1], 1, 16, R, dtype=BF, device=DEV),
                                  v_pool=torch.zeros(cu_pages[-1], 1, 16, C, dtype=BF, device=DEV))
    x = rnd(T, W, dtype=BF, seed=40)
    a = mixer.forward(x, step, cache).float()
    mixer.w_ukv = None
    b = mixer.forward(x, step, cache).float()
    assert float((a - b).norm() / b.norm()) < 2e-2 and not torch.equal(a, b)
    mixer.w_ukv = torch.zeros(1, device=DEV)
    assert mixer._whole_prompts(step)
    step.q_starts = [0, 16, 0]
    assert not mixer._whole_prompts(step)
    step.q_starts, step.n_decode = [0] * n, 1
    assert not mixer._whole_prompts(step)
    step.n_decode, mixer.window = 0, 49
    assert not mixer._whole_prompts(step)
