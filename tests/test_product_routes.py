"""Which way calls take, decided on the host: no kernel is launched here."""
import types

import pytest
import torch

BF = torch.bfloat16


def kernel_set(device, **lib):
    """The kernels' host side with entries that note their calls."""
    from return_amd.kernels.hip_ops import HipOps
    ops = object.__new__(HipOps)
    ops.device, ops.launched = torch.device(device), []
    ops._stream = lambda: 0
    ops.lib = types.SimpleNamespace(ra_gemm_heads_fits=lambda *a: 1, **lib)
    ops.lib.ra_gemm_heads_bf16 = lambda *a: ops.launched.append(a) or 0
    return ops


def test_batched_product_of_operands_on_another_device():
    """Addresses of host memory never reach the kernel; what the library takes is what it gives."""
    ops = kernel_set("cuda:0")
    a, b = torch.randn(3, 2, 64).to(BF), torch.randn(3, 64, 16).to(BF)
    assert torch.equal(ops.batched_product(a, b), torch.bmm(a, b)) and not ops.launched
    for x, y, out in [(a.to("meta"), b, None), (a, b.to("meta"), None), (a, b, torch.empty(3, 2, 16, dtype=BF, device="meta"))]:
        ops = kernel_set("cpu")
        try:
            ops.batched_product(x, y, out=out)
        except RuntimeError:
            pass
        assert not ops.launched
    out = torch.empty(3, 2, 16, dtype=BF)
    assert ops.batched_product(a, b, out=out) is out and len(ops.launched) == 1


@pytest.mark.parametrize("M,most", [(4097, 4096), (4096, 4096), (128, 4096), (8191, 4096), (12289, 4096), (700, 256), (41000, 1024)])
def test_float32_products_by_parts_come_in_even_pieces(M, most):
    """No piece is short: a remainder of a few rows would cost a pass over W that use_split would not give it."""
    sizes = []
    ops = kernel_set("cpu", ra_gemm_split_scratch=lambda m, N, K: 6 * m * K,
                     ra_gemm_split_f32=lambda x, w, y, m, N, K, scratch, room, stream: sizes.append((x, y, m)) or 0)
    ops.SPLIT_ROWS = most
    x, w = torch.empty(M, 32), torch.empty(4, 32)
    y = ops._linear_by_parts(x, w)
    assert sum(m for _, _, m in sizes) == M and len(sizes) == -(-M // most)
    assert all(M / len(sizes) - 128 < m <= most for _, _, m in sizes)
    at = 0
    for from_x, to_y, m in sizes:
        assert (from_x, to_y) == (x.data_ptr() + 128 * at, y.data_ptr() + 16 * at) and (at == 0 or at % 128 == 0)
        at += m


def test_float32_products_by_parts_leave_no_tile_half_empty():
    """129 to 192 rows (and 257 to 320 of middling widths) go by tiles of 64 rows: seen by the rows that the parts have room for."""
    from return_amd.kernels.hip_ops import load_library
    lib = load_library()
    for M, N, rows in [(128, 151936, 128), (129, 151936, 192), (160, 151936, 192), (192, 151936, 192), (193, 151936, 256),
                       (320, 32768, 320), (320, 151936, 384), (321, 32768, 384)]:
        assert lib.ra_gemm_split_scratch(M, N, 64) == rows * 64 * 6, (M, N)


def test_batched_products_that_the_library_forms_faster_are_its():
    """(rows, heads, K, N) on either side of the rule's lines."""
    ops = kernel_set("cpu")
    own = [(1, 32, 512, 128), (4, 32, 512, 128), (4, 64, 512, 128), (2, 32, 512, 64), (4, 16, 512, 256), (1, 32, 1024, 128),
           (2, 128, 512, 128), (2, 32, 512, 64), (1, 64, 512, 64)]
    library = [(5, 32, 512, 128), (8, 16, 512, 128), (4, 128, 512, 128), (3, 32, 512, 64), (1, 128, 512, 64), (2, 64, 512, 64),
               (4, 64, 512, 256), (2, 32, 1024, 128), (1, 64, 1024, 128), (1, 32, 1024, 512), (1, 32, 128, 512), (1, 32, 128, 128)]
    assert all(ops.use_heads(B, M, N, K) for M, B, K, N in own)
    assert not any(ops.use_heads(B, M, N, K) for M, B, K, N in library)
    a, b = torch.randn(16, 8, 512).to(BF), torch.randn(16, 512, 128).to(BF)
    ops.batched_product(a, b)
    assert not ops.launched


def test_token_input_goes_by_its_fastest_form():
    """(rows, columns, side channels) on either side of the rule's lines: 0 the loop over runs of columns, 1 a row a workgroup with its
    reads asked for ahead, 2 four rows a workgroup."""
    from return_amd.kernels.hip_ops import load_library
    form = load_library().ra_token_side_form
    for T, H, S, want in [(1, 4096, 32, 1), (64, 2048, 32, 1), (64, 2048, 24, 1), (1, 3072, 32, 0), (64, 4096, 24, 0), (1, 1024, 32, 0),
                          (64, 2048, 16, 0), (1, 4096, 8, 0), (65, 3072, 32, 1), (512, 1024, 8, 1), (128, 512, 8, 0), (513, 1024, 8, 0),
                          (640, 2560, 8, 0), (767, 768, 16, 1), (768, 4096, 16, 2), (2048, 2048, 8, 0), (2048, 1024, 16, 2),
                          (4096, 2048, 16, 0), (4096, 1024, 32, 2), (4096, 4096, 16, 2), (4096, 512, 32, 0)]:
        assert form(T, H, S) == want, (T, H, S)


def test_convolutions_go_by_their_faster_form():
    """(requests, longest, rows, channels, SiLU) on either side of the rule's lines: 1 eight channels a thread, 0 one."""
    from return_amd.kernels.hip_ops import load_library
    form = load_library().ra_causal_conv_form
    for n, longest, T, C, silu, want in [(1, 2048, 2048, 4096, 0, 1), (1, 64, 64, 4096, 0, 0), (64, 8, 512, 4096, 0, 1), (64, 7, 448, 4096, 0, 0),
                                         (1, 300, 300, 4096, 1, 0), (1, 2048, 2048, 4096, 1, 0), (1, 2048, 2048, 6144, 1, 1), (4, 701, 2804, 6144, 1, 1),
                                         (64, 64, 127, 6144, 1, 0), (64, 512, 575, 4096, 1, 1), (64, 512, 575, 1024, 1, 1), (64, 256, 319, 6144, 1, 1)]:
        assert form(T, n, longest, C, 2 * silu) == want, (n, longest, T, C, silu)


@pytest.mark.parametrize("tiles,shift,want", [({64: torch.zeros(1, 2, dtype=torch.int32)}, 0, "ra_attention_prefill_f32"),
                                              ({64: torch.zeros(1, 2, dtype=torch.int32)}, 1, "ra_attention_plain"),
                                              ({}, 0, "ra_attention_plain"), (None, 0, "ra_attention_plain")])
def test_float32_attention_of_steps_without_tile_lists_and_of_pools_at_odd_places(tiles, shift, want):
    """The kernels of 16-byte reads need the list of tiles and whole pieces; the plain kernel takes the rest, as it did."""
    names, i = [], torch.zeros(3, dtype=torch.int32)
    lib = {n: (lambda *a, n=n: names.append(n) or 0) for n in ("ra_attention_prefill_f32", "ra_attention_decode_f32", "ra_attention_plain")}
    ops = kernel_set("cpu", ra_attention_f32_fits=lambda D: 1, **lib)
    pools = [torch.zeros(16 * 64 + shift)[shift:].view(1, 1, 16, 64) for _ in range(2)]
    step = types.SimpleNamespace(n_tokens=5, n_decode=0, n_prefill_tokens=5, prefill_tiles=tiles, n_seqs=1, cu_q=i, q_start=i, prefill_toks=None,
                                 decode_segs=None, groups=[types.SimpleNamespace(page_table=i, cu_pages=i, kv_start=i)])
    q = torch.zeros(5, 2, 64)
    ops.attention(q, torch.zeros_like(q), *pools, step, 0, 0.125)
    assert names == [want]


def test_products_of_17_to_64_rows_that_the_library_forms_faster_are_its():
    """(result columns, gated) on either side of the rule's lines at 256 CUs."""
    ops = kernel_set("cpu", ra_gemm_rows_fits=lambda M, N, K: 1)
    ops.cu_count, ops.own_gemm = 256, False
    for N, gated, want in [(12288, True, True), (8192, True, True), (16384, True, True), (25600, True, False), (27648, True, False), (6144, True, False),
                           (16384, False, True), (151936, False, True), (6144, False, False)]:
        assert ops.use_rows(64, N, 5120, gated) == want, (N, gated)
    for N, K, want in [(16385, 1024, True), (28672, 512, True), (16385, 1032, False), (28672, 1280, False), (16384, 4096, True), (8191, 1024, False)]:
        assert ops.use_rows(17, N, K, True) == want, (N, K)


def test_many_very_short_prompts_go_over_the_latents():
    """(heads, prompts, tokens of each): tiles of 128 rows that hold a few tokens each, and many of them."""
    from return_amd.parts.attention import LatentAttention
    mixer = object.__new__(LatentAttention)
    mixer.w_ukv, mixer.window, mixer.rt = torch.zeros(1), None, types.SimpleNamespace(ops=types.SimpleNamespace(LATENT_PROMPT_ROWS=128))
    for H, n, q, want in [(32, 1, 2, True), (32, 64, 2, True), (32, 65, 2, False), (32, 128, 5, False), (32, 128, 8, True), (16, 128, 2, True),
                          (16, 256, 4, False), (16, 256, 8, True)]:
        mixer.H = H
        step = types.SimpleNamespace(n_decode=0, n_prefill_tokens=n * q, n_tokens=n * q, n_seqs=n, q_starts=[0] * n, max_q_len=q, prefill_tiles={128: None})
        assert mixer._whole_prompts(step) == want, (H, n, q)


def test_experts_in_panels_go_by_the_sweep_while_their_tiles_are_too_few():
    """(pairs, experts, hidden, inner) on either side of the rule's lines at 256 CUs: the sweep's 16 rows, or tiles of up to 320, 160 or 80."""
    ops = kernel_set("cpu", ra_moe_panel_rows=lambda n, E: 320 if n >= 2 * E else 16)
    ops.cu_count, ops.panel_tile_rows = 256, 0
    for n, E, H, I, want in [(128, 8, 2048, 1024, 16), (255, 8, 2048, 1024, 16), (256, 8, 2048, 1024, 320), (8 * 80, 8, 2048, 1024, 320), (8 * 81, 8, 2048, 1024, 80), (8 * 161, 8, 2048, 1024, 80), (8 * 240, 8, 2048, 1024, 80),
                             (8 * 320, 8, 2048, 1024, 80), (8 * 321, 8, 2048, 1024, 160), (383, 32, 1024, 512, 16), (384, 32, 1024, 512, 320), (32 * 80, 32, 1024, 512, 320), (32 * 81, 32, 1024, 512, 80),
                             (32 * 160, 32, 1024, 512, 80), (32 * 161, 32, 1024, 512, 160), (32 * 321, 32, 1024, 512, 320), (127, 64, 2048, 512, 16),
                             (128, 64, 2048, 512, 320), (64, 32, 4096, 3072, 320), (63, 32, 4096, 3072, 16), (383, 4, 1024, 1024, 16), (384, 4, 1024, 1024, 80), (4 * 700, 4, 1024, 1024, 160),
                             (40 * 128, 40, 1536, 512, 320), (16 * 12, 16, 1024, 1408, 320), (16, 8, 4096, 4096, 320), (15, 8, 4096, 4096, 16)]:
        assert ops.use_panel_rows(n, E, H, I) == want, (n, E, H, I)
        tiles = min(n, n // want + E)                          # (the plan's places; a tile's number has 15 bits)
        assert tiles <= 0x7fff
    ops.panel_tile_rows = 160
    assert ops.use_panel_rows(16, 8, 2048, 1024) == 160


def test_products_of_up_to_16_rows_that_the_sweep_forms_more_slowly_are_not_its():
    """(rows, result columns, K) on either side of the rule's lines at 256 CUs: beyond 256 result columns a CU narrow W leaves most of
    its waves without columns of K."""
    from return_amd.kernels.hip_ops import load_library
    lib = load_library()
    ops = kernel_set("cpu", ra_gemm_sweep_fits=lib.ra_gemm_sweep_fits)
    ops.cu_count = 256
    for M, N, K, want in [(1, 65536, 1024, True), (1, 65537, 1024, False), (8, 151936, 512, False), (8, 151936, 1528, False), (8, 151936, 1536, True),
                          (9, 151936, 760, False), (9, 151936, 768, True), (16, 151936, 4096, True), (16, 151936, 5120, True), (16, 151936, 8192, True),
                          (16, 151936, 9728, False), (8, 151936, 9728, True), (16, 65536, 12288, True), (1, 1024, 4096, True), (1, 1023, 4096, False),
                          (4, 3072, 512, False), (16, 2048, 8192, True), (16, 2047, 8192, False), (1, 4096, 4104, False), (16, 4351, 5112, False),
                          (8, 4352, 4104, True), (8, 2048, 5120, True), (8, 2047, 5120, False)]:
        assert ops.use_sweep(M, N, K, False) == want, (M, N, K)


def test_products_of_long_rows_that_the_library_forms_faster_are_its():
    """(rows, result columns, K) on either side of the rule's lines at 256 CUs; only bfloat16 results are the library's."""
    from return_amd.kernels.hip_ops import load_library
    lib = load_library()
    ops = kernel_set("cpu", ra_gemm_sweep_fits=lib.ra_gemm_sweep_fits)
    ops.cu_count, ops.product_plan, ops.own_gemm = 256, {}, False
    for M, N, K, want in [(5, 5120, 8704, "library"), (4, 5120, 8704, "sweep"), (8, 4096, 8704, "sweep"), (8, 4097, 8704, "library"), (9, 4096, 8704, "library"),
                          (8, 8191, 9728, "library"), (8, 8192, 9728, "sweep"), (8, 5120, 10240, "sweep"), (16, 5120, 10240, "library"),
                          (16, 5120, 12288, "sweep"), (16, 5120, 8448, "sweep"), (16, 6144, 8192, "sweep"), (16, 3072, 10240, "sweep")]:
        assert ops.route_linear(M, N, K, BF) == want, (M, N, K)
        assert ops.route_linear(M, N, K, torch.float32) == "sweep", (M, N, K)


def product_routes():
    """The rules and candidates of products, on the host."""
    from return_amd.kernels.hip_ops import load_library
    ops = kernel_set("cpu")
    ops.lib, ops.cu_count, ops.own_gemm, ops.product_plan = load_library(), 256, False, {}
    ops._library_fp32_out = ops._library_bmm_fp32 = True
    ops.gated_skinny_rows, ops._times = 8, {}
    return ops


@pytest.mark.parametrize("batches", [True, False])
def test_the_rule_for_a_residual_product_is_among_what_is_measured(batches):
    """Else nothing is measured, and the rule's choice stays whatever the other ways take."""
    ops = product_routes()
    ops._library_bmm_fp32 = batches                              # (whether the library has a batch with 32-bit results)
    for N, K in [(4096, 12288), (4096, 4096), (2560, 9728), (2560, 4096), (5120, 25600), (5120, 5120), (5120, 8192), (2048, 2048), (2048, 8192),
                 (1024, 3072), (512, 1536), (4096, 4160), (2048, 6152)]:
        for rows in ops.ROW_STEPS + ops.ROW_STEPS_RESIDUAL:
            ways = ops._candidates(rows, N, K, False, "residual")
            assert ops.route_linear(rows, N, K, "residual") in ways and len(ways) == len(set(ways)), (rows, N, K, ways)
            if rows > 64:
                assert "library" in ways and ("block" in ways) == (K % 64 == 0), (rows, N, K, ways)
    ops.own_gemm = True
    assert not any(w == "block" for w in ops._candidates(512, 4096, 4096, False, "residual"))
    # what a measurement has said is what is done, the one tiled product too
    ops.own_gemm = False
    for how in ("block", "library", "split8"):
        ops.product_plan = {(512, 4096, 4096, False, "residual"): how}
        assert ops.route_linear(400, 4096, 4096, "residual") == how
    assert ops.route_linear(513, 4096, 4096, "residual") != "split8"


def test_ways_of_many_rows_are_measured_beside_the_rule():
    """Which ways _measure times, and that it follows them: here the tiled product in one piece takes half as long as all others."""
    ops = product_routes()
    seen = []

    def fake(runs, weights, launches):
        seen.append(sorted(runs))
        return {how: 1.0 if how == "block" else 2.0 for how in runs}
    ops._time_ways = fake
    key = (512, 2048, 8192, False, "residual")
    assert ops.route_linear(512, 2048, 8192, "residual").startswith("split")
    assert ops._measure(key, [torch.zeros(2048, 8192, dtype=BF)], 1, 0.93) == "block"
    assert seen == [["block", "library", "split2", "split4", "split8"]]


@pytest.mark.parametrize("batches", [True, False])
@pytest.mark.parametrize("M,K", [(300, 1024), (100, 2048), (65, 8192)])
def test_residual_products_of_operands_at_odd_places_are_the_librarys_one_product(batches, M, K):
    """Sizes that the rule cuts into pieces of K, x 2 bytes off: also on a library without batches of 32-bit results."""
    ops = product_routes()
    ops._library_bmm_fp32 = batches
    w = torch.randn(2048, K).to(BF)
    x = torch.empty(M * K + 1, dtype=BF)[1:].view(M, K).copy_(torch.randn(M, K))
    assert ops.route_linear(M, 2048, K, "residual").startswith("split") and x.data_ptr() % 16
    y = ops.linear_residual(x, w)
    assert torch.equal(y, x @ w.t())
    ops.lib = types.SimpleNamespace(ra_gemm_block_bf16=lambda *a: ops.launched.append(a) or 0)
    shares = ops._split_product(x[:, :].clone(), w, 2)           # (operands in place: by tiles)
    assert len(ops.launched) == 1 and tuple(shares.tensor.shape) == (2, M, 2048)


class Noted:
    """The library with entries that note their calls in place of launching."""

    def __init__(self, *entries):
        from return_amd.kernels.hip_ops import load_library
        self.lib, self.entries, self.calls = load_library(), entries, []

    def __getattr__(self, name):
        if name in self.entries:
            return lambda *a: self.calls.append(name) or 0
        return getattr(self.lib, name)


def test_products_with_a_row_kernel_behind_go_by_the_tiles_where_the_two_kernels_take_longer():
    """(rows, columns, K) on either side of the line; the figures stand at the rule."""
    ops = product_routes()
    for M, N, K, one in [(1500, 12288, 4096, True), (3072, 12288, 4096, True), (2304, 12288, 4096, False), (256, 8192, 2048, True), (2048, 8192, 2048, True),
                         (512, 4096, 12288, False), (256, 12288, 4096, False)]:
        ops.lib = Noted("ra_gemm_block_bf16")
        x, w = torch.empty(M, K, dtype=BF), torch.empty(N, K, dtype=BF)
        assert (ops._act_by(x, w, False, 2, 0.0, 0.0, None) is not None) == one == (ops.lib.calls == ["ra_gemm_block_bf16"]), (M, N, K)


def test_a_measured_way_is_left_only_where_the_row_kernel_makes_up_for_it():
    """Gated products of few rows with a bias or a clamp behind: the plain product as it was measured, its times in microseconds."""
    key, x, w = (8, 24576, 4096, False, BF), torch.empty(6, 4096, dtype=BF), torch.empty(24576, 4096, dtype=BF)
    for plan, times, one in [({}, {}, True), ({key: "sweep"}, {}, True), ({key: "library"}, {"sweep": 40.0, "library": 30.0}, False),
                             ({key: "library"}, {"sweep": 40.0, "library": 36.5}, True), ({key: "library"}, {"library": 30.0}, False),
                             ({key: "library"}, {}, False)]:
        ops = product_routes()
        ops.lib, ops.product_plan, ops._times = Noted("ra_gemm_sweep_act_bf16"), plan, {key: {how: t * 1e-6 for how, t in times.items()}}
        for act, bias in ((1, None), (0, torch.empty(24576))):
            assert (ops._act_by(x, w, True, act, 7.0, 1.702, bias) is not None) == one, (plan, times)


def test_a_norm_derived_from_the_rms_norm_forms_its_own_rows_before_a_convolution():
    """The one kernel for a norm and the convolution behind it stands for these two parts, not for parts derived from them."""
    from return_amd.parts.block import ConvSideBlock
    from return_amd.parts.conv import ResidualCausalConv
    from return_amd.parts.norm import RMSNorm
    both = torch.zeros(2, 8)
    rt = types.SimpleNamespace(vector32=lambda t: t, ops=types.SimpleNamespace(norm_conv=lambda *a: both))

    class Doubled(RMSNorm):
        def forward(self, h, delta=None, out_rows=None):
            return 2 * h

    class Shifted(ResidualCausalConv):
        def forward(self, x, step, tail):
            return x + 1

    h, params = torch.randn(2, 8), {"size": 8, "eps": 1e-6, "taps": 4}
    part = {cls: cls(params, {"weight": torch.ones(8, 4) if issubclass(cls, ResidualCausalConv) else torch.ones(8)}, rt)
            for cls in (RMSNorm, Doubled, ResidualCausalConv, Shifted)}

    def formed(norm, conv):
        return ConvSideBlock._normed(part[norm], part[conv] if conv else None, h, None, None, {"tail": None}, "tail")
    assert formed(RMSNorm, ResidualCausalConv) is both
    assert torch.equal(formed(Doubled, Shifted), 2 * h + 1) and torch.equal(formed(Doubled, None), 2 * h)
    part[ResidualCausalConv].forward = lambda x, step, tail: x - 1
    assert torch.equal(formed(Doubled, ResidualCausalConv), 2 * h - 1)
