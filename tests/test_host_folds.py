"""CPU: the lazily reduced row arithmetic of the eval_h folds
(zkwasm-prover_amd/csrc/evalh_rows.h) against full-width products reduced after
every step, with operands drawn from the whole range, from its top and from its
bottom, so that the sums under one reduction come near their bounds; stored
values must be canonical."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001
FOLDS = ["perm_p1", "perm_p2", "logup", "logup_extra", "shuffle", "perm_set", "gates"]

# stored words of one row of a two-column permutation set whose product and
# Montgomery quotient are both large: y, beta, gamma, bd_0, bd_1 / h, z(wX), z,
# X, l_active, v_0, sigma_0, v_1, sigma_1
SET_CHALLENGES = [
    0x22ED3D0638B0B0645448BDB50C989039B7AE094EEB65FBF4A10B14096EDACD60,
    0x0BA6B2A0B44E16295D2C084493734D19381177E96784CDD1FA42B1EA516C1EF1,
    0x06D5799B21ABA714D670A3B0CF7DF86E2664004B075D4B92B10618D54DACD172,
    0x21C0B44431847982BBD9B21692D156AED0E940ABCAFFE9796858D5839CA71830,
    0x102B0035E1B27D7523D2C7ECDC08A88AAA658A7E180884044C7155EE4E830393]
SET_ROW = [
    0x28E2DD1BEDEFCC97AECA5613C9E0FD0184CD9A055E8A6F565EF5D4D38DC58F75,
    0x1749E76E45F305608AE8E3B249042098AB7434DFDB4ED82981317B8CD22A1518,
    0x1E58477C792AA28513508BA0EFF5BEAA877D14B8EB3A53AC9859AF056982D1BA,
    0x2804CF69F365E56EE057779BB085B3411A06F04EF24401DF08C6D8D03C2F96AE,
    0x2F7B8B46007A144167E606893A707B70734A88F42F49D601956274F2D320CD95,
    0x0969D8AC009B9E6FF4C18468F8D2EC41D9345A0315EB5D26BC4B462E6A090457,
    0x283AEE3229ECBE7578AD14F924F02B68A1A560F72905662E4509B5B40F1FE0C3,
    0x0B63E2FBE4D0046978B6CFB4E770C6857F15878B15A34ACD97686B230415CE01,
    0x10B5183A029DA99B79648CF727043668503ECBC0AAAF3C5A915EEEE60B853262]
SET_RESULT = 0x005A9BB916047611848640A9FA67093C439AA17D4DBD810DA15477D14EF587CA


def limbs(values):
    return np.array([[(x >> (64 * i)) & (2**64 - 1) for i in range(4)] for x in values], dtype=np.uint64)


def ranged(n, rng):
    """n stored values: a quarter uniform, half from the top 2 %, an eighth
    each from the bottom 2 % and of the ends 0, 1, r - 1 and one"""
    top = R >> 192
    v = rng.integers(0, 2**64, (n, 4), dtype=np.uint64)
    kind = rng.integers(0, 8, n)
    v[:, 3] = np.where(kind < 2, rng.integers(0, top, n), np.where(
        kind < 6, rng.integers(top * 98 // 100, top, n), rng.integers(0, top // 50, n))).astype(np.uint64)
    ends = limbs([0, 1, R - 1, (1 << 256) % R])
    v[kind == 7] = ends[rng.integers(0, 4, int((kind == 7).sum()))]
    return v


@pytest.fixture(scope="module")
def folds(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("folds") / "libfolds.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-w", "-I", os.path.join(HERE, "host_folds"), "-I",
                    os.path.join(ROOT, "zkwasm-prover_amd", "csrc"),
                    os.path.join(HERE, "host_folds", "check.cpp"), "-o", out], check=True)
    L = ctypes.CDLL(out)
    L.folds_run.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_int,
                            ctypes.c_void_p, ctypes.c_void_p]

    def run(which, rows, challenges, cols):
        n, width = rows.shape[:2]
        out, exp = np.zeros((n, 4), dtype=np.uint64), np.zeros((n, 4), dtype=np.uint64)
        L.folds_run(FOLDS.index(which), rows.ctypes.data, n, width, challenges.ctypes.data, cols, out.ctypes.data,
                    exp.ctypes.data)
        return out, exp
    return run


def test_permutation_set_known_row(folds):
    out, exp = folds("perm_set", limbs(SET_ROW).reshape(1, 9, 4), limbs(SET_CHALLENGES), 2)
    assert (exp == limbs([SET_RESULT])).all()
    assert (out == exp).all()


@pytest.mark.parametrize("y", [R - 1, R * 95 // 100, R // 2], ids=["top", "95", "half"])
@pytest.mark.parametrize("which,width,cols", [("perm_p1", 5, 0), ("perm_p2", 8, 3), ("logup", 11, 0),
                                              ("logup_extra", 6, 0), ("shuffle", 8, 1), ("shuffle", 12, 3),
                                              ("perm_set", 7, 1), ("perm_set", 13, 4), ("gates", 5, 0),
                                              ("gates", 11, 3)])
def test_fold_rows_canonical(folds, which, width, cols, y):
    n = 100000
    rng = np.random.default_rng(width + cols)
    rows = ranged(n * width, rng).reshape(n, width, 4)
    challenges = np.concatenate([limbs([y]), ranged(8, rng)])
    out, exp = folds(which, rows, challenges, cols)
    assert int((out != exp).any(axis=1).sum()) == 0
