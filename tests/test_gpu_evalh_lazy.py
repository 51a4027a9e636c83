"""The lazily reduced constraint folds at the ends of their operands' range:
every column, challenge and selector takes the stored values 0, 1, r - 1,
r - 2, the field's one and 2^253 in turn (all combinations of neighbours), and
constant columns of r - 1; 16 permutation columns; bit for bit."""
import numpy as np
import pytest
import test_gpu_evalh as base

pytestmark = pytest.mark.gpu

R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001
ENDS = [0, 1, R - 1, R - 2, (1 << 256) % R, 1 << 253]


class _Ends:
    def __init__(self, zo, top):
        self._zo, self._values = zo, [R - 1] if top else ENDS
        self._n = 0

    def __getattr__(self, name):
        return getattr(self._zo, name)

    def rand_fr(self, n, seed):
        # column number k steps its value every 6^(k mod 4) rows
        v = np.array([[(x >> (64 * i)) & (2**64 - 1) for i in range(4)] for x in self._values], dtype=np.uint64)
        step = 6 ** (self._n % 4)
        self._n += 1
        return v[(np.arange(n) // step + seed) % len(v)]


@pytest.mark.parametrize("top", [False, True])
@pytest.mark.parametrize("which", ["permutation", "logup", "shuffle", "shuffle_v2", "set"])
def test_folds_at_range_ends(gpu, zo, which, top):
    z = _Ends(zo, top)
    if which == "permutation":
        base.test_permutation_kernels(gpu, z, 12)
    elif which == "logup":
        base.test_logup_kernels(gpu, z, 12)
    elif which == "shuffle":
        base.test_shuffle_kernels(gpu, z, 12)
    elif which == "shuffle_v2":
        base.test_shuffle_v2_group_counts(gpu, z, 16, 4)
    else:
        base.test_permutation_eval_h_set(gpu, z, 16, 4)
