"""NTT passes on the matrix cores (degrees 6 to 8, launches of at least 2^19
elements) against the CPU oracle, bit for bit: the degrees in first,
middle and last passes (degree 8: first only), batches just below and at the threshold (which counts
the transforms of one launch, at most 48, of 2^15 elements or more), workgroups
with a part of their tiles, extreme inputs (the byte columns' bounds), iNTT scaling, coset extensions and capture."""
import ctypes

import numpy as np
import pytest
from test_gpu_field_ntt import _CosetItem, _gpu_ntt, _ntt_batch, _omegas_dev

pytestmark = pytest.mark.gpu

R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001
TOP = np.array([[(R - 1) >> (64 * i) & (2**64 - 1) for i in range(4)]], dtype=np.uint64)


def _pattern(zo, kind, n, seed):
    if kind == "random":
        return zo.rand_fr(n, seed)
    x = np.zeros((n, 4), dtype=np.uint64)
    if kind == "top":
        x[:] = TOP
    elif kind == "top_odd":
        x[1::2] = TOP
    elif kind == "top_half":
        x[n // 2:] = TOP
    else:  # one element, the last
        x[-1:] = TOP
    return x


# plans: 2^19 = 7 6 6, 2^20 = 7 7 6, 2^21 = 7 7 7, 2^22 = 8 7 7
@pytest.mark.parametrize("log_n,kind,inverse", [(19, "top", False), (19, "top_odd", True), (20, "top_half", False),
                                                (21, "random", True), (21, "last", False), (22, "top_odd", True)])
def test_single_transform(gpu, zo, log_n, kind, inverse):
    n = 1 << log_n
    x = _pattern(zo, kind, n, 40 + log_n)
    w, n_inv = zo.root_of_unity(log_n), None
    if inverse:
        w, n_inv = zo.fr_inv(w), zo.fr_inv(zo.fr_from_u64(n))
        exp = zo.ntt(x, log_n, w, n_inv)
    else:
        exp = zo.ntt(x, log_n, w)
    assert (_gpu_ntt(zo, x, log_n, w, n_inv) == exp).all()


# 2^16 = 8 8 at the threshold, one transform short of it, and with others
# beside it; 2^15 = 8 7, in one launch and with one transform in a second, which
# stays below the threshold; 2^12 = 6 6, radix-2 passes in several launches;
# transforms whose tiles don't divide evenly among their workgroups
@pytest.mark.parametrize("logs", [[16] * 8, [16] * 7 + [12, 14], [16] * 8 + [15, 12, 3], [15] * 16, [12] * 128,
                                  [18, 17, 18, 13], [15] * 49, [18] * 3, [17, 15, 19, 16, 15, 15]])
def test_batch(gpu, zo, logs):
    specs, exps = [], []
    for m, k in enumerate(logs):
        x, w = _pattern(zo, "top" if m % 5 == 4 else "random", 1 << k, 700 + m), zo.root_of_unity(k)
        if m % 3 == 2:
            w, n_inv = zo.fr_inv(w), zo.fr_inv(zo.fr_from_u64(1 << k))
            specs.append((x, k, w, n_inv))
            exps.append(zo.ntt(x, k, w, n_inv))
        else:
            specs.append((x, k, w, None))
            exps.append(zo.ntt(x, k, w))
    got = _ntt_batch(zo, specs)
    assert [m for m in range(len(logs)) if not (got[m] == exps[m]).all()] == []


@pytest.mark.parametrize("shapes", [[(18, 1)], [(17, 2), (16, 3)], [(12, 4)] * 8, [(19, 3)],
                                    [(16, 2)] * 3])
def test_coset_extension(gpu, zo, shapes):
    from zkprover import device as dv
    from zkprover._lib import lib
    f = lib().zk_coset_extend_batch
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    f.restype = ctypes.c_int
    zeta = zo.to_mont([pow(7, (R - 1) // 3, R)])
    cp = np.concatenate([zeta, zo.fr_mul(zeta, zeta)])
    keep, items, exps = [], (_CosetItem * len(shapes))(), []
    for m, (log_n, ext) in enumerate(shapes):
        n, N = 1 << log_n, 1 << (log_n + ext)
        coeffs = _pattern(zo, "top" if m % 2 else "random", n, 60 + m)
        w = zo.root_of_unity(log_n + ext)
        host = np.zeros((N, 4), dtype=np.uint64)
        host[:n] = coeffs
        exps.append(zo.ntt(zo.extended_prepare(host, cp, n, N, 0), log_n + ext, w))
        om, src, buf, tmp = _omegas_dev(zo, log_n + ext, w), dv.to_dev(coeffs), dv.empty(N), dv.empty(N)
        keep.append((om, src, buf, tmp))
        items[m] = _CosetItem(src.data_ptr(), buf.data_ptr(), tmp.data_ptr(), om.data_ptr(), log_n, ext)
    dcp = dv.to_dev(cp)
    sw = (ctypes.c_ubyte * len(shapes))()
    assert f(ctypes.addressof(items), len(shapes), dcp.data_ptr(), 3, sw, dv.stream_handle()) == 0
    for m, (_, _, buf, tmp) in enumerate(keep):
        assert (dv.from_dev(tmp if sw[m] else buf) == exps[m]).all(), shapes[m]


def test_captured_batch_replays(gpu, zo):
    """a captured batch replays to the oracle's bytes, with its buffers cleared
    and other eager work between the replays"""
    import torch
    from test_gpu_graph import _NttItem
    from zkprover import device as dv
    from zkprover._lib import call
    stream = torch.cuda.Stream()
    sh = stream.cuda_stream
    logs = [18, 18, 16]
    xs = [zo.rand_fr(1 << k, 90 + m) for m, k in enumerate(logs)]
    ws = [zo.root_of_unity(k) for k in logs]
    oms = [_omegas_dev(zo, k, w) for k, w in zip(logs, ws)]
    orig = [dv.to_dev(x) for x in xs]
    bufs, tmps = [dv.empty(1 << k) for k in logs], [dv.empty(1 << k) for k in logs]
    items = (_NttItem * len(logs))(*[_NttItem(bufs[m].data_ptr(), tmps[m].data_ptr(), oms[m].data_ptr(), None, k, 0)
                                     for m, k in enumerate(logs)])
    swapped, exec_ = (ctypes.c_ubyte * len(logs))(), ctypes.c_void_p()
    torch.cuda.synchronize()
    call("zk_graph_begin", sh)
    for m, k in enumerate(logs):
        call("zk_copy", bufs[m].data_ptr(), orig[m].data_ptr(), (1 << k) * 32, sh)
    call("zk_ntt_batch", ctypes.addressof(items), len(logs), ctypes.addressof(swapped), sh)
    call("zk_graph_end", sh, ctypes.byref(exec_))
    exps = [zo.ntt(x, k, w) for x, k, w in zip(xs, logs, ws)]
    try:
        for rep in range(3):
            for b in bufs + tmps:
                b.zero_()
            torch.cuda.synchronize()
            call("zk_graph_launch", exec_, sh)
            torch.cuda.synchronize()
            for m in range(len(logs)):
                assert (dv.from_dev(tmps[m] if swapped[m] else bufs[m]) == exps[m]).all(), (rep, m)
    finally:
        call("zk_graph_destroy", exec_)


def _to_int(v):
    return sum(int(v[i]) << (64 * i) for i in range(4))


@pytest.mark.parametrize("inverse", [False, True])
def test_2e24_known_values(gpu, zo, inverse):
    """2^24 (four passes of degree 6) on five nonzero inputs: out[k] = s sum a_j
    w^(j k), s = 1 / n in the inverse, at 3000 outputs"""
    k, n = 24, 1 << 24
    rng = np.random.default_rng(24 + inverse)
    where = np.concatenate([[1, n - 1, n // 3], rng.integers(0, n, 2)])
    x = np.zeros((n, 4), dtype=np.uint64)
    x[where] = zo.rand_fr(5, 24)
    w, n_inv, scale = zo.root_of_unity(k), None, 1
    if inverse:
        w, n_inv, scale = zo.fr_inv(w), zo.fr_inv(zo.fr_from_u64(n)), pow(n, -1, R)
    got = _gpu_ntt(zo, x, k, w, n_inv)
    root = zo.from_mont(w)[0]
    vals = [_to_int(x[j]) * scale % R for j in where]
    for o in np.concatenate([[0, 1, n - 1, n // 2, 4096, 4095], rng.integers(0, n, 3000)]):
        exp = sum(v * pow(root, int(j) * int(o) % n, R) for j, v in zip(where, vals)) % R
        assert _to_int(got[o]) == exp, o
