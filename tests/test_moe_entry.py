"""What the experts' products refuse before anything is launched (host code: no GPU)."""
import pytest

from return_amd.kernels.hip_ops import load_library

BF16, REFUSED = 1, 1


@pytest.mark.parametrize("n_pairs,N,K,gated", [
    (64, 70000, 16384, 0), (64, 35000, 16384, 1),             # an expert's matrix of 2 GiB and more
    (70000, 64, 16384, 0), (70000, 64, 16384, 1),             # rows of x as many
    (64, 64, 40, 0), (64, 64, 8, 1)])                         # K no multiple of 32
def test_tiles_in_lds_are_refused_beyond_their_range(n_pairs, N, K, gated):
    lib = load_library()
    pointers = [None] * 6
    assert lib.ra_moe_tile_rows(n_pairs, 4, N * (1 + gated), K, BF16) != 256
    assert lib.ra_moe_product(*pointers, n_pairs, 4, 256, N, K, 1, gated, BF16, None) == REFUSED
    assert lib.ra_moe_product_act(*pointers, n_pairs, 4, 256, N, K, 1, gated, 0, 0.0, 0.0, None, BF16, None) == REFUSED
