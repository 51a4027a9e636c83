"""GPU parity of the batch inversion, logup and grand-product tiles at their
borders: elements per thread 2 / 4 / 8 (2^17 and 2^20 elements), partial
last tiles, one row, tiles of 1024 product rows, several tiles per thread of
the top workgroup (above 2^18 rows), zero denominators and zero numerators at
the edges of tiles.  Compared with the CPU oracle to the byte.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

R = 21888242871839275222246405745257275088548364400416034343698204186575808495617


def _dv():
    from zkprover import device as dv
    from zkprover._lib import call
    return dv, call


@pytest.mark.parametrize("n", [1, 2, 511, 513, 1 << 17, (1 << 17) + 1, 1 << 20, (1 << 20) + 1])
def test_inversion_and_logup_tiles(gpu, zo, n):
    from zkprover.device import Arena
    dv, call = _dv()
    A = Arena()
    st = dv.stream_handle()
    x = zo.rand_fr(n, 7 + n)
    beta = zo.rand_fr(1, 8)
    minus_beta = zo.fr_sub(zo.fr_zeros(1), beta)[0]
    for i in {0, n // 2, n - 1} if n > 2 else set():
        x[i] = minus_beta  # x + beta = 0: inverse 0
    tmp, s, z = dv.empty(n), dv.empty(n), dv.empty(n)
    exp = zo.fr_zeros(n)
    for it in range(2):
        call("logup_sum_input_inv", dv.ptr(s), A.put(x), dv.ptr(tmp), A.put(beta), it, n, st)
        exp = zo.logup_sum_input_inv(exp, x, beta, it)
    assert (dv.from_dev(s) == exp).all()
    m = zo.rand_fr(n, 9 + n)
    last = dv.to_dev(zo.rand_fr(1, 10))
    li = n // 3
    exp_z, exp_last = zo.eval_logup_z_compose(exp, x, m, beta, zo.rand_fr(1, 10), li)
    call("eval_logup_z_compose", dv.ptr(z), dv.ptr(s), A.put(x), A.put(m), A.put(beta), dv.ptr(last), li, n, st)
    assert (dv.from_dev(z) == exp_z).all()
    assert (dv.from_dev(last) == exp_last).all()


def _shuffle(zo, inputs, shuffles, beta):
    from zkprover.device import Arena
    dv, call = _dv()
    A = Arena()
    n, g = len(inputs[0]), len(inputs)
    betas = np.concatenate([zo.fr_pow(beta, j + 1) for j in range(g)])
    z, tmp = dv.empty(n), dv.empty(n)
    call("zk_shuffle_z", dv.ptr(z), A.put_all(inputs), A.put_all(shuffles), g, A.put(betas), dv.ptr(tmp), n,
         dv.stream_handle())
    return dv.from_dev(z)


# 600000 rows: 586 tiles, three per thread of the top workgroup; 1100000: five, read twice
@pytest.mark.parametrize("n,rows", [(1, []), (3, [1]), (1023, []), (1025, [1023]), (5000, [0]), (5000, [1024, 1025]),
                                    (5000, [2047, 4999]), (600000, [299999]),
                                    (1100000, [7, 1099999])])
def test_shuffle_zero_denominators(gpu, zo, n, rows):
    beta = zo.rand_fr(1, 3)
    inputs, shuffles = [zo.rand_fr(n, 4), zo.rand_fr(n, 5)], [zo.rand_fr(n, 6), zo.rand_fr(n, 7)]
    minus_beta = zo.fr_sub(zo.fr_zeros(1), beta)[0]
    for r in rows:
        shuffles[0][r] = minus_beta
    assert (_shuffle(zo, inputs, shuffles, beta) == zo.shuffle_z(inputs, shuffles, beta)).all()
    # zero numerators at the same rows
    for r in rows:
        inputs[0][r] = minus_beta
    assert (_shuffle(zo, inputs, shuffles, beta) == zo.shuffle_z(inputs, shuffles, beta)).all()
    if rows:
        shuffles[0] = zo.rand_fr(n, 6)
        assert (_shuffle(zo, inputs, shuffles, beta) == zo.shuffle_z(inputs, shuffles, beta)).all()


@pytest.mark.parametrize("n,ncols", [(1, 1), (2, 2), (1023, 1), (1024, 2), (1025, 3), (300007, 2)])
def test_permutation_ragged_rows(gpu, zo, n, ncols):
    from zkprover.device import Arena
    dv, call = _dv()
    A = Arena()
    beta, gamma = zo.rand_fr(1, 1), zo.rand_fr(1, 2)
    delta, omega = zo.to_mont([pow(7, 1 << 28, R)]), zo.root_of_unity(max(1, (n - 1).bit_length()))
    vals, sig = [zo.rand_fr(n, 20 + j) for j in range(ncols)], [zo.rand_fr(n, 30 + j) for j in range(ncols)]
    if n > 10:  # a zero denominator: v = -(beta sigma + gamma)
        r = n // 2
        t = zo.fr_add(zo.fr_mul(beta, sig[0][r:r + 1]), gamma)
        vals[0][r] = zo.fr_sub(zo.fr_zeros(1), t)[0]
    dstart = zo.fr_pow(delta, 2)
    z, tmp = dv.empty(n), dv.empty(n)
    call("zk_permutation_z_set", dv.ptr(z), A.put_all(vals), A.put_all(sig), ncols, A.put(beta), A.put(gamma),
         A.put(dstart), A.put(delta), A.put(omega), dv.ptr(tmp), n, dv.stream_handle())
    assert (dv.from_dev(z) == zo.permutation_z_set(vals, sig, beta, gamma, dstart, delta, omega)).all()
