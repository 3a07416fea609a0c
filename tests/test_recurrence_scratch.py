"""The scratch that the recurrences' kernels by chunks of rows ask for (host code: no GPU)."""
import ctypes

import pytest

from return_amd.kernels.hip_ops import load_library

LIMIT = 48 << 20          # floats


@pytest.mark.parametrize("H,D,V,rule", [(64, 128, 128, 0), (32, 128, 128, 3), (128, 64, 64, 2), (16, 128, 4096, 1), (340, 128, 4096, 1), (1, 1, 1, 0)])
@pytest.mark.parametrize("q_lens", [[16], [24] * 64, [100] * 64, [33, 5000] * 40, [1, 3, 4096], [23] * 7, [40] * 300], ids=lambda q: f"{len(q)} of {q[-1]}")
def test_at_most_its_limit(H, D, V, rule, q_lens):
    """Never more than the limit, unless one chunk of one request alone takes more; something wherever a request is long
    enough, nothing where none is."""
    need = load_library().ra_recurrence_scratch((ctypes.c_int * len(q_lens))(*q_lens), len(q_lens), H, D, V, rule)
    one = load_library().ra_recurrence_scratch((ctypes.c_int * 1)(32), 1, H, D, V, rule)
    assert need <= max(LIMIT, one)
    assert (need > 0) == (max(q_lens) >= (24 if rule == 2 else 16))
    assert need == 0 or need >= one
