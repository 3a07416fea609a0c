"""The experts' products on the matrix cores (bf16) against a 64-bit product of the same bfloat16 operands: tiles of up to 256
rows in LDS (twelve pairs an expert and more) at every count of groups of 16 rows, few k-steps, experts without rows, widths
that are no multiple of a tile; tiles of 16 rows with W read in whole runs (fewer pairs) at one to eight waves, columns shared
out unevenly, more tiles than workgroups; both activations, factors on what an expert reads. The same of matrices in panels: tiles of
up to 320 rows at every count of groups, steps of K that are no multiple of four, W that ends inside a tile; few rows at one to eight steps a
wave."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from return_amd.kernels.hip_ops import HipOps
    return HipOps(DEV)


def check(ops, rows, E, H, I, ids, kind, panels=False):
    """One expert a token, so that the counts are exact. A result is two bf16 roundings (2^-9 each of the halves and of the
    activation) away from the 64-bit one, grown by the product with them: 2^-6 of the largest."""
    g = torch.Generator().manual_seed(len(ids) + H)
    x = torch.randn(len(ids), H, generator=g).bfloat16()
    w_up = (torch.randn(E, 2 * I, H, generator=g) * H ** -0.5).bfloat16()
    w_down = (torch.randn(E, H, I, generator=g) * I ** -0.5).bfloat16()
    factor = 0.5 + torch.rand(len(ids), 1, generator=g)
    kw = {"clamped": dict(activation="clamped", limit=1.0), "input": dict(weigh="input"), "silu": {}}[kind]
    # (the kernel that this is about)
    assert (ops.lib.ra_moe_panel_rows(len(ids), E) if panels else ops.lib.ra_moe_tile_rows(len(ids), E, 2 * I, H, 1)) == rows
    a, b = w_up.to(DEV), w_down.to(DEV)
    if panels:
        a, b = (ops.expert_panels(lambda e: w[e], E, H, I, gated, torch.bfloat16) for w, gated in ((a, True), (b, False)))
    got = ops.moe_experts(x.to(DEV), ids.int()[:, None].to(DEV), factor.to(DEV), a, b, **kw)
    want = torch.zeros(len(ids), H, dtype=torch.float64)
    for e in ids.unique().tolist():
        t = (ids == e).nonzero()[:, 0]
        h = (x[t].double() * (factor[t].double() if kind == "input" else 1.0)) @ w_up[e].double().T
        a, b = h[:, :I], h[:, I:]
        if kind == "clamped":
            a, b = a.clamp(max=1.0), b.clamp(-1.0, 1.0) + 1.0
            mid = a * torch.sigmoid(1.702 * a) * b
        else:
            mid = a * torch.sigmoid(a) * b
        want[t] = (mid @ w_down[e].double().T) * (1.0 if kind == "input" else factor[t].double())
    err = (got.cpu().double() - want).abs().max() / want.abs().max()
    assert err < 2.0 ** -6, float(err)


def shuffled(counts):
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])
    return ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(len(ids)))]


KINDS = ["silu", "clamped", "input"]


@pytest.mark.parametrize("E,H,I,counts", [
    (4, 32, 32, [8, 9, 31, 33]), (3, 64, 96, [16, 20, 0]), (2, 224, 40, [64, 65]), (5, 256, 160, [128, 129, 144, 145, 0]),
    (3, 96, 300, [160, 192, 193]), (4, 160, 128, [224, 225, 256, 257]), (2, 1024, 224, [272, 700]), (1, 128, 64, [12]),
    (6, 192, 2, [0, 0, 48, 0, 0, 500]), (2, 352, 288, [15, 300]), (3, 416, 32, [64, 97, 513])])
@pytest.mark.parametrize("kind", KINDS)
def test_products_of_many_rows(ops, E, H, I, counts, kind):
    check(ops, 256, E, H, I, shuffled(counts), kind)


@pytest.mark.parametrize("E,H,I,counts", [
    (4, 8, 8, [1, 0, 2, 0]), (3, 520, 24, [5, 16, 7]), (2, 1032, 40, [1, 20]), (8, 2048, 136, [1, 0, 0, 3, 17, 0, 33, 9]),
    (3, 4096, 56, [15, 1, 0]), (2, 2568, 1000, [1, 1]), (1, 3080, 16, [11]), (700, 64, 24, [1] * 650 + [0] * 50), (5, 512, 7, [0, 4, 0, 1, 0])])
@pytest.mark.parametrize("kind", KINDS)
def test_products_of_few_rows(ops, E, H, I, counts, kind):
    check(ops, 16, E, H, I, shuffled(counts), kind)


@pytest.mark.parametrize("E,H,I,counts", [
    (4, 64, 64, [1, 16, 17, 33]), (3, 128, 192, [48, 20, 0]), (2, 320, 64, [64, 65]), (5, 256, 192, [80, 96, 97, 112, 0]),
    (3, 64, 448, [128, 144, 160]), (4, 192, 128, [176, 192, 208, 209]), (2, 1024, 576, [256, 700]), (1, 128, 64, [2]),
    (6, 192, 64, [0, 0, 48, 0, 0, 500]), (2, 4096, 320, [15, 300]), (9, 448, 64, [64, 97, 0, 2, 5, 1, 1, 30, 1100]),
    (40, 64, 128, [7] * 20 + [330] * 3 + [0] * 17), (2, 64, 64, [320, 321]), (3, 64, 320, [225, 241, 289])])
@pytest.mark.parametrize("kind", KINDS)
def test_panels_many_rows(ops, E, H, I, counts, kind):
    check(ops, 320, E, H, I, shuffled(counts), kind, panels=True)


@pytest.mark.parametrize("E,H,I,counts", [
    (4, 64, 64, [1, 0, 2, 0]), (20, 576, 128, [5, 16, 7] + [0] * 17), (20, 1088, 192, [1, 20] + [0] * 18),
    (40, 2048, 128, [1, 0, 0, 3, 17, 0, 33, 9] + [0] * 32), (16, 4096, 64, [15, 1] + [0] * 14), (4, 2624, 4096, [1, 1, 0, 0]), (8, 3136, 64, [11] + [0] * 7),
    (700, 64, 64, [1] * 650 + [0] * 50), (5, 512, 1536, [0, 4, 0, 1, 0])])
@pytest.mark.parametrize("kind", KINDS)
def test_panels_few_rows(ops, E, H, I, counts, kind):
    check(ops, 16, E, H, I, shuffled(counts), kind, panels=True)


@pytest.mark.parametrize("rows", [16, 80, 160, 320])
@pytest.mark.parametrize("E,H,I,counts", [
    (4, 64, 64, [1, 16, 17, 33]), (2, 320, 64, [80, 81]), (3, 192, 448, [159, 160, 161]), (4, 448, 128, [176, 0, 320, 321]), (1, 1024, 192, [1700]),
    (2, 128, 320, [3300, 15]), (130, 128, 64, [1] * 60 + [700, 0, 161] + [17] * 67)])
@pytest.mark.parametrize("kind", KINDS)
def test_panels_by_tiles_of_every_height(ops, rows, E, H, I, counts, kind):
    """At the edges of the heights, with more than four tiles of an expert, whatever the rule would take for these sizes."""
    ops.panel_tile_rows = rows
    try:
        check(ops, ops.lib.ra_moe_panel_rows(sum(counts), E), E, H, I, shuffled(counts), kind, panels=True)
    finally:
        ops.panel_tile_rows = 0


@pytest.mark.parametrize("E,counts", [
    (3, [3649, 40, 0]), (1, [6081]), (2, [321, 320]), (4, [1700, 3300, 1281, 640]), (130, [1] * 60 + [700, 0, 1601] + [17] * 67),
    (200, [330, 0, 2, 16] * 50), (1024, [0] * 1000 + [400] * 24)])
@pytest.mark.parametrize("most_rows", [320, 160, 80])
def test_plan_of_tiles_of_panels(ops, E, counts, most_rows):
    """Every pair stands once, with its expert's; an expert's tiles are as few as their height allows, even within a group of 16 rows, so
    that of several of 320 rows none has fewer than ten groups; the largest tiles, by groups, come first; runs of up to four of an expert's tiles are numbered."""
    ids = shuffled(counts)
    order, tiles, meta, most, _ = ops._moe_plan(ids.int().to(DEV), E, most_rows)
    n = int(meta)
    order, tiles = order.cpu(), tiles[:n].cpu().tolist()
    assert n == sum(-(-c // most_rows) for c in counts) <= most and order.sort().values.tolist() == list(range(len(ids)))
    at, first_of = 0, []
    while tiles:
        e = tiles[0][0]
        of_e = [t for t in tiles if t[0] == e]
        assert tiles[:len(of_e)] == of_e and len(of_e) == -(-counts[e] // most_rows)
        first_of.append(((of_e[0][2] & 0xffff) + 15) // 16)
        groups = []
        for j, (_, start, packed) in enumerate(of_e):
            rows = packed & 0xffff
            assert start == at and packed >> 16 == min(len(of_e) - (j & ~3), 4) * 16 + (j & 3)
            assert (ids[order[at:at + rows].long()] == e).all()
            at += rows
            groups.append(-(-rows // 16))
        assert at - of_e[0][1] == counts[e] and 16 * max(groups) <= most_rows
        assert max(groups) - min(groups) <= 1 and (len(of_e) == 1 or 32 * min(groups) >= most_rows), (counts[e], groups)
        tiles = tiles[len(of_e):]
    assert at == len(ids) and first_of == sorted(first_of, reverse=True)


@pytest.mark.parametrize("weigh", ["input", "output"])
@pytest.mark.parametrize("tokens", [1, 7, 8, 9, 61, 64])
def test_panels_of_steps_in_parts_and_of_rows_at_odd_places(ops, tokens, weigh):
    """A step whose rows are beyond what an offset of 32 bits reaches goes in parts of its tokens (eight of them here), and rows that are not
    16-byte aligned are copied: the same bits. Tiles of one height, whose sums have one order whatever the step's size."""
    E, H, I, top = 5, 128, 192, 3
    g = torch.Generator().manual_seed(tokens)
    w_up, w_down = (torch.randn(*s, generator=g).bfloat16().to(DEV) * 0.1 for s in ((E, 2 * I, H), (E, H, I)))
    a, b = ops.expert_panels(lambda e: w_up[e], E, H, I, True, torch.bfloat16), ops.expert_panels(lambda e: w_down[e], E, H, I, False, torch.bfloat16)
    x = torch.randn(tokens, H, generator=g).bfloat16().to(DEV)
    ids = torch.rand(tokens, E, generator=g).argsort(1)[:, :top].int().to(DEV)
    weights = torch.rand(tokens, top, generator=g).to(DEV)
    ops.panel_tile_rows = 320
    try:
        want = ops.moe_experts(x, ids, weights, a, b, weigh=weigh)
        odd = torch.empty(tokens * H + 1, dtype=torch.bfloat16, device=DEV)[1:].view(tokens, H).copy_(x)
        assert odd.data_ptr() % 16 and torch.equal(ops.moe_experts(odd, ids, weights, a, b, weigh=weigh), want)
        ops.PANEL_STEP_BYTES = 9 * 2 * top * I
        assert torch.equal(ops.moe_experts(x, ids, weights, a, b, weigh=weigh), want)
    finally:
        ops.panel_tile_rows = 0
        ops.__dict__.pop("PANEL_STEP_BYTES", None)
