"""The tiled product of more than 64 rows: every tile at its edges, pieces of K, gated results, and which calls go to it."""
import os
import shutil

import pytest
import torch

from tests.test_kernels_gpu import ops, rnd  # noqa: F401
from tests.test_lds_stages import _compiled, _kernels, unfinished_reads
from tests.test_product_routes import kernel_set

BF = torch.bfloat16
TILES = [(256, 256), (224, 256), (192, 256), (160, 256), (128, 256), (96, 256), (256, 128), (192, 128), (160, 128), (128, 128), (96, 128),
         (64, 128)]


def bound(K, want):
    """A bfloat16 result: half a last place (2^-9) of it, and 32-bit sums of K products of about unit size (2^-24 each, twice over)."""
    return want.abs() * 2.0 ** -8 + 2.0 ** -22 * K


@pytest.mark.gpu
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("K", [64, 128, 448])
def test_every_tile_at_its_edges(ops, tile, K):
    """One row or 8 columns more than whole tiles, a row less, and K of one step, of fewer steps than there are stages, and of more."""
    bm, bn = TILES[tile]
    for M, N in [(bm, bn), (bm + 1, bn + 8), (2 * bm - 1, 2 * bn - 8), (65, 8)]:
        x, w = rnd(M, K, dtype=BF, seed=M), rnd(N, K, dtype=BF, seed=N, scale=0.3)
        want = x.double() @ w.double().t()
        y = ops._block_product(x, w, False, tile + 16, BF)
        assert bool(((y.double() - want).abs() <= bound(K, want)).all()), (M, N)
        for pieces in (1, 2) if K > 64 and K % 128 == 0 else (1,):
            y = torch.full((pieces, M, N), float("nan"), device=x.device)
            ops._check(ops.lib.ra_gemm_block_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, 0, tile + 16 * pieces, 0, 0, 0.0, 0.0, None,
                                                   ops._stream()), "")
            torch.testing.assert_close(y.double().sum(0), want, atol=2.0 ** -22 * K, rtol=1e-6)
    for M, I in [(bm + 1, bn // 2 + 8), (65, 8)]:
        x, w = rnd(M, K, dtype=BF, seed=M), rnd(2 * I, K, dtype=BF, seed=I, scale=0.2)
        gu = (x.double() @ w.double().t()).float().to(BF).double()
        want = gu[:, :I] * torch.sigmoid(gu[:, :I]) * gu[:, I:]
        y = ops._block_product(x, w, True, tile + 16, BF)
        # (a half that is rounded the other way, 2^-8 of it, moves silu by up to 1.1 times as much, and the result is rounded once more)
        lax = (gu[:, :I].abs() * 1.1 * gu[:, I:].abs() + want.abs()) * 2.0 ** -8 + want.abs() * 2.0 ** -8 + 2.0 ** -20 * K
        assert bool(((y.double() - want).abs() <= lax).all()), (M, I)


@pytest.mark.gpu
@pytest.mark.parametrize("tile,M,N", [(11, 64 * 13 - 5, 128 * 5 + 8), (11, 64 * 9, 128 * 3), (10, 96 * 11 - 1, 128 * 4 - 8), (6, 256 * 9 - 7, 128 * 2 + 16),
                                      (5, 96 * 14 - 90, 256 + 8), (0, 256 * 10 - 255, 256 * 2), (11, 64 * 8, 128 * 3 + 8)])
def test_every_tile_of_many_is_formed_once(ops, tile, M, N):
    """Up to eight tiles of rows, and more, which go by fours with a shorter last run; the workgroups no whole number an XCD; one, three and five
    pieces of K of several steps each, fewer and more than the stages. Results are written over what is no number."""
    K = 64 * 3 * 5
    x, w = rnd(M, K, dtype=BF, seed=M), rnd(N, K, dtype=BF, seed=N, scale=0.3)
    want = x.double() @ w.double().t()

    def run(gated, pieces, dtype):
        y = torch.full((M, N // 2) if gated else (M, N) if dtype == 1 else (pieces, M, N), float("nan"), dtype=BF if dtype == 1 else torch.float32, device=x.device)
        ops._check(ops.lib.ra_gemm_block_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, gated, tile + 16 * pieces, dtype, 0, 0.0, 0.0, None,
                                              ops._stream()), "")
        return y.double()
    assert bool(((run(0, 1, 1) - want).abs() <= bound(K, want)).all())
    for pieces in (1, 3, 5):
        y, step = run(0, pieces, 0), K // pieces
        for i in range(pieces):
            part = x[:, i * step:(i + 1) * step].double() @ w[:, i * step:(i + 1) * step].double().t()
            torch.testing.assert_close(y[i], part, atol=2.0 ** -22 * step, rtol=1e-6)
    if N % 16 == 0:
        gu = want.float().to(BF).double()
        g, u = gu[:, :N // 2], gu[:, N // 2:]
        silu = g * torch.sigmoid(g)
        lax = (g.abs() * 1.1 * u.abs() + (silu * u).abs()) * 2.0 ** -8 + (silu * u).abs() * 2.0 ** -8 + 2.0 ** -20 * K
        assert bool(((run(1, 1, 1) - silu * u).abs() <= lax).all())


@pytest.mark.gpu
def test_products_go_by_the_tiles_and_stay_the_products(ops):
    """The public entries at sizes that the rules give to the tiled product; operands at odd places go to the library as before."""
    from return_amd.parts.runtime import Slabs
    x, w = rnd(600, 1024, dtype=BF, seed=1), rnd(4096, 1024, dtype=BF, seed=2, scale=0.1)
    want = x.double() @ w.double().t()
    assert ops.route_linear(600, 4096, 1024, BF) == "block" and ops.route_gated(600, 2048, 1024) == "block"
    assert bool(((ops.linear(x, w).double() - want).abs() <= bound(1024, want)).all())
    odd = torch.empty(600 * 1024 + 1, dtype=BF, device=x.device)[1:].view(600, 1024).copy_(x)
    assert bool(((ops.linear(odd, w).double() - want).abs() <= bound(1024, want)).all())
    torch.testing.assert_close(ops.linear_silu_mul(odd, w).float(), ops.linear_silu_mul(x, w).float(), atol=2e-2, rtol=2e-2)
    x, w = rnd(300, 8192, dtype=BF, seed=3), rnd(2048, 8192, dtype=BF, seed=4, scale=0.1)
    want, how = x.double() @ w.double().t(), ops.route_linear(300, 2048, 8192, "residual")
    y = ops.linear_residual(x, w)
    assert how == f"split{y.tensor.shape[0]}" and isinstance(y, Slabs)
    torch.testing.assert_close(y.tensor.double().sum(0), want, atol=2.0 ** -22 * 8192, rtol=1e-6)


@pytest.mark.gpu
def test_values_that_are_no_numbers_reach_their_own_row_and_column(ops):
    x, w = rnd(130, 192, dtype=BF, seed=5), rnd(264, 192, dtype=BF, seed=6)
    x[129, 100], w[263, 3] = float("nan"), float("inf")
    y = ops._block_product(x, w, False, 9 + 16, BF)
    assert bool(torch.isnan(y[129]).all()) and not bool(torch.isfinite(y[:, 263]).any())
    assert bool(torch.isfinite(y[:129, :263]).all())


def test_which_products_go_by_the_tiles():
    """(rows, result columns, K) on either side of the rules' lines at 256 CUs, and sizes that the kernel does not take."""
    ops = kernel_set("cpu")
    ops.cu_count, ops.own_gemm = 256, False
    # (what was measured on either side stands at the rule)
    for M, N, K, want in [(64, 8192, 2048, False), (256, 8192, 2048, True), (256, 6144, 4096, False), (300, 6144, 4096, True),
                          (536, 6144, 2560, True), (1280, 6144, 2560, False), (536, 6144, 4096, True), (1999, 6144, 4096, False), (2048, 6144, 4096, False),
                          (2804, 6144, 4096, True), (384, 4096, 4096, False), (448, 4096, 4096, True), (800, 4096, 4096, True), (1100, 4096, 4096, True),
                          (1280, 8192, 2048, False), (1999, 8192, 2048, False), (3072, 8192, 2048, False), (1280, 12288, 2048, False), (2804, 12288, 2048, False),
                          (1280, 12288, 4096, False), (2048, 12288, 4096, False), (3072, 12288, 4096, False), (1280, 24576, 1024, False),
                          (2804, 8256, 2048, True), (1024, 8256, 256, True), (2048, 8256, 128, True), (2048, 8192, 128, False), (4096, 16384, 64, False),
                          (256, 10304, 4096, True), (1999, 10304, 4096, True), (1999, 10240, 4096, False), (1536, 2048, 12288, False), (1536, 2048, 8184, False),
                          (536, 6144, 2568, False), (536, 6140, 2560, False), (536, 32, 4096, False)]:
        assert ops.use_block(M, N, K) == want, (M, N, K)
    for M, I, K, want in [(64, 12288, 4096, False), (65, 1536, 512, True), (300, 12288, 4096, True), (1024, 12288, 4096, True), (1400, 12288, 4096, True),
                          (2048, 12288, 4096, False), (4096, 12288, 4096, False), (2804, 12288, 4096, True), (536, 9728, 2560, True), (2804, 9728, 2560, True),
                          (300, 8192, 2048, True), (2804, 8192, 2048, True), (128, 3072, 4096, False), (536, 3072, 4096, True), (1000, 1024, 4096, True),
                          (300, 256, 512, True), (300, 256, 1024, True), (300, 104, 4096, False), (300, 512, 12288, False), (300, 1024, 4096, False),
                          (300, 768, 8192, False), (2048, 3072, 12288, False), (300, 104, 512, True), (300, 100, 512, False), (300, 104, 520, False)]:
        assert ops.use_block_gated(M, I, K) == want, (M, I, K)
    for M, N, K, want in [(64, 2560, 9728, 0), (536, 2560, 9728, 4), (2048, 4096, 4096, 1), (536, 2047, 4096, 0), (536, 2048, 4100, 0),
                          (2048, 4096, 12288, 1), (4096, 4096, 4096, 0), (2048, 8192, 8192, 0), (4096, 8192, 8192, 0), (2048, 5120, 25600, 0)]:
        assert ops.use_block_residual(M, N, K) == want, (M, N, K)
    ops.own_gemm = True
    assert not ops.use_block(536, 6144, 2560) and not ops.use_block_gated(536, 9728, 2560) and not ops.use_block_residual(536, 2560, 9728)


def test_pieces_are_those_that_the_norm_has_forms_for():
    """By the plan alone 4,096 x 12,288 took three pieces at 288 row counts, 5,120 x 25,600 five at 544."""
    from return_amd.kernels.hip_ops import load_library
    lib = load_library()
    for N, K in [(4096, 12288), (2048, 6144), (5120, 25600), (5120, 5120), (4096, 6656)]:
        pieces = {lib.ra_gemm_block_plan(M, N, K, 0, 8, 256, None, None) >> 4 for M in range(65, 2100)}
        assert pieces <= {1, 2, 4, 8} and len(pieces) > 1, (N, K, pieces)
    assert lib.ra_gemm_block_plan(800, 4096, 12288, 0, -3, 256, None, None) < 0


def test_plans_and_calls_that_are_refused():
    """No tile beyond the list, no pieces that K does not have, no operand of 2 GiB: refused before anything is launched."""
    from return_amd.kernels.hip_ops import load_library
    lib = load_library()
    for M, N, K, gated in [(0, 64, 64, 0), (64, 64, 0, 0), (64, 64, 96, 0), (64, 60, 64, 0), (64, 24, 64, 1), (1 << 20, 64, 1024, 0), (64, 1 << 20, 1024, 0)]:
        assert lib.ra_gemm_block_plan(M, N, K, gated, 1, 256, None, None) < 0, (M, N, K, gated)
    assert lib.ra_gemm_block_plan(300, 2048, 8192, 0, -4, 256, None, None) >> 4 == 4 and lib.ra_gemm_block_plan(300, 2048, 192, 0, -2, 256, None, None) < 0
    assert lib.ra_gemm_block_plan(300, 2048, 8192, 0, 9, 256, None, None) < 0 and lib.ra_gemm_block_plan(300, 2048, 8192, 0, 0, 256, None, None) < 0
    for plan, M, N, K, gated, dtype, at in [(-1, 64, 64, 64, 0, 1, 0), (12 + 16, 64, 64, 64, 0, 1, 0), (0, 64, 64, 64, 0, 1, 0), (9 + 32, 64, 64, 64, 0, 0, 0),
                                            (9 + 32, 64, 64, 128, 0, 1, 0), (9 + 16, 64, 64, 64, 1, 0, 0), (9 + 16, 64, 60, 64, 0, 1, 0),
                                            (9 + 16, 64, 64, 64, 0, 1, 8), (9 + 16 * 9, 64, 64, 576, 0, 0, 0)]:
        assert lib.ra_gemm_block_bf16(16 + at, 16, 16, M, N, K, gated, plan, dtype, 0, 0.0, 0.0, None, None) != 0, plan


@pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")), reason="no hipcc")
def test_no_stage_of_a_tile_is_refilled_before_it_is_read(tmp_path):
    kernels = {n: b for n, b in _kernels(_compiled("gemm_block.hip", tmp_path)).items() if any(" lds" in i for _, c in b for i in c)}
    assert len(kernels) == 3 * len(TILES)
    for name, blocks in kernels.items():
        copies, bad = unfinished_reads(blocks, behind_same=True)
        assert copies > 0 and not bad, (name, bad[:4], len(bad))
