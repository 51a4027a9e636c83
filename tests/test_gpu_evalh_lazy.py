"""The lazily reduced constraint folds at the ends of their operands' range:
every column, challenge and selector takes the stored values 0, 1, r - 1,
r - 2, the field's one and 2^253 in turn (all combinations of neighbours), and
constant columns of r - 1; 16 permutation columns; bit for bit.  A product's
size also depends on its Montgomery quotient, which these values do not choose:
the last two tests take rows from the top and the bottom of the range at random
(and one known row), as test_host_folds does for every fold on the CPU."""
import numpy as np
import pytest
import test_gpu_evalh as base
from test_host_folds import SET_CHALLENGES, SET_RESULT, SET_ROW, limbs, ranged

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


def _permutation_set(h, z, x, la, vs, ss, y, beta, gamma, bd, rot):
    dv, call, A = base._env()
    th = dv.to_dev(h)
    call("zk_permutation_eval_h_set", A.hold(th), A.put(z), A.put_all(vs), A.put_all(ss), len(vs), A.put(beta),
         A.put(gamma), A.put(bd), A.put(x), A.put(la), A.put(y), rot, len(h), dv.stream_handle())
    return dv.from_dev(th)


def test_permutation_set_known_row(gpu):
    row, c = limbs(SET_ROW), limbs(SET_CHALLENGES)
    h, zn, z, x, la, v0, s0, v1, s1 = [np.repeat(row[k:k + 1], 2, axis=0) for k in range(9)]
    zz = np.concatenate([z[:1], zn[:1]])  # row 0 reads z(wX) from row 1
    got = _permutation_set(h, zz, x, la, [v0, v1], [s0, s1], c[0:1], c[1:2], c[2:3], c[3:5], 1)
    assert (got[0] == limbs([SET_RESULT])[0]).all()


@pytest.mark.parametrize("nc", [1, 4])
def test_permutation_set_canonical(gpu, zo, nc):
    n, rot = 1 << 17, 4
    rng = np.random.default_rng(nc)
    h, z, x, la = [ranged(n, rng) for _ in range(4)]
    vs, ss = [ranged(n, rng) for _ in range(nc)], [ranged(n, rng) for _ in range(nc)]
    y, (beta, gamma), bd = limbs([R * 95 // 100]), ranged(2, rng).reshape(2, 1, 4), ranged(nc, rng)
    lhs, rhs = zo.field_op(z, rot, None, None, 0, None, n, 2), z
    for c in range(nc):
        vg = zo.field_op(vs[c], 0, None, None, 0, gamma, n, 0)
        lhs = zo.field_op(lhs, 0, None, zo.field_op(ss[c], 0, beta, vg, 0, None, n, 0), 0, None, n, 1)
        rhs = zo.field_op(rhs, 0, None, zo.field_op(x, 0, bd[c:c + 1], vg, 0, None, n, 0), 0, None, n, 1)
    t = zo.field_op(zo.field_op(lhs, 0, None, rhs, 0, None, n, 3), 0, None, la, 0, None, n, 1)
    exp = zo.field_op(h, 0, y, t, 0, None, n, 0)
    got = _permutation_set(h, z, x, la, vs, ss, y, beta, gamma, bd, rot)
    assert int((got != exp).any(axis=1).sum()) == 0
