"""When a mixed step's two attention kernels go to two streams: by the keys that its decoded tokens read (no GPU)."""
import types

import pytest

from return_amd.kernels.hip_ops import HipOps

KI = 1024


def beside(lens, window=0, keep_first=0, portion=(512, 2048), calls=1):
    """The rule for a step of decoded tokens in requests of these lengths and a portion (rows, rows before it)."""
    step = types.SimpleNamespace(n_decode=len(lens), max_decode_seq_len=max(lens, default=0), q_lens=[1] * len(lens) + [portion[0]],
                                 q_starts=[n - 1 for n in lens] + [portion[1]])
    ops = types.SimpleNamespace(overlap_attention=None)
    got = {HipOps._side_by_side(ops, step, window, keep_first) for _ in range(calls)}
    assert len(got) == 1
    return got.pop()


@pytest.mark.parametrize("lens, window, keep_first, want", [
    ([8 * KI] * 64, 0, 0, True), ([8 * KI] * 63 + [8 * KI - 1], 0, 0, False),
    ([450] * 23 + [32 * KI], 0, 0, False),                  # 786 Ki if every one were as long as the longest
    ([64 + i * 36 for i in range(128)], 0, 0, False), ([64 + i * 64 for i in range(128)], 0, 0, True),
    ([512 * KI], 0, 0, True), ([512 * KI, 5], 0, 0, True), ([512 * KI - 1], 0, 0, False), ([], 0, 0, False),
    ([9 * KI] * 64, 8 * KI, 0, True), ([9 * KI] * 63 + [100], 8 * KI, 0, False), ([9 * KI] * 64, 8 * KI - 64, 0, False),
    ([9 * KI] * 64, 8 * KI - 64, 64, True), ([8 * KI - 60] * 64, 8 * KI - 64, 64, False), ([9 * KI] * 64, 100, 0, False)])
def test_keys_that_are_read_decide(lens, window, keep_first, want):
    assert beside(lens, window, keep_first, calls=3) is want
    assert beside(lens, window, keep_first, portion=(700, 40000)) is want
