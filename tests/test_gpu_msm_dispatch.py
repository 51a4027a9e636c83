"""GPU parity of the MSM at the borders of its dispatch: the one-workgroup
window sort and the two-level sort, small and large sort tiles, windows with
fewer than 16 buckets, the bucket reductions by quads of lanes (with and
without a merge of parts) and by segments, chunk partials summed by a quad and
by a workgroup, and the exceptional additions (equal and opposite points).
Every result is compared with the CPU oracle's MSM as an affine point.
"""
import numpy as np
import pytest

from test_gpu_msm import _zk_msm, _zk_msm_batch

pytestmark = pytest.mark.gpu

R = 21888242871839275222246405745257275088548364400416034343698204186575808495617


def _check(zo, pts, sc, c=0):
    got = _zk_msm(pts, sc, c)
    assert (zo.g1_to_affine(got) == zo.g1_to_affine(zo.msm(pts, sc))).all()


# kWindowSortMax = 24576 scalars, windows of at most 1024 buckets (c <= 11);
# 1024-scalar tiles; B < 16 below c = 5; a part merge above 4096 buckets (c >= 14)
@pytest.mark.parametrize("n,c", [(1, 2), (17, 3), (1023, 4), (1025, 5), (4097, 6), (24575, 9), (24576, 11),
                                 (24577, 11), (24576, 12), (300, 14), (5000, 15), (3000, 17)])
def test_msm_dispatch_borders(gpu, zo, n, c):
    _check(zo, zo.gen_bases_random(n, 300 + n), zo.rand_fr(n, 301 + c), c)


def test_msm_batch_dispatch_borders(gpu, zo):
    """one item above the window sort's limit moves the whole batch; 33 items
    cross the bucket count of the two reductions"""
    for ns in ([24576, 1, 777], [24577, 1, 777], [900 + m for m in range(33)]):
        pts = zo.gen_bases_random(max(ns), 5)
        sets = [zo.rand_fr(n, 40 + n) for n in ns]
        out = _zk_msm_batch([pts[:n] for n in ns], sets, 9)
        for n, s, got in zip(ns, sets, out):
            assert (zo.g1_to_affine(got.reshape(1, 12)) == zo.g1_to_affine(zo.msm(pts[:n], s))).all(), n


def _negated(pts):
    p = 21888242871839275222246405745257275088696311157297823662689037894645226208583
    out = pts.reshape(-1, 8).copy()
    for k in range(len(out)):
        y = sum(int(out[k, 4 + i]) << (64 * i) for i in range(4))
        y = (p - y) % p
        out[k, 4:] = [(y >> (64 * i)) & 0xFFFFFFFFFFFFFFFF for i in range(4)]
    return out.reshape(pts.shape)


@pytest.mark.parametrize("n", [2, 40, 100, 1000, 5000])
def test_msm_equal_partials(gpu, zo, n):
    """one point throughout: every chunk of a bucket has the same partial sum,
    and neighbouring buckets the same total (doublings in every merge)"""
    one = zo.gen_bases_random(1, 9).reshape(1, -1)
    pts = np.repeat(one, n, axis=0).reshape(n, -1)
    _check(zo, pts, np.repeat(zo.fr_from_u64(1), n, axis=0), 7)
    _check(zo, pts, np.concatenate([zo.fr_from_u64(1 + k % 4) for k in range(n)]), 7)


def test_msm_opposite_buckets(gpu, zo):
    """neighbouring buckets (and equal ones) hold opposite points: identities
    in the merges and in the masked sums"""
    n = 64
    half = zo.gen_bases_random(n // 2, 10)
    neg = _negated(half)
    pts = np.empty((n, half.reshape(n // 2, -1).shape[1]), dtype=np.uint64)
    pts[0::2], pts[1::2] = half.reshape(n // 2, -1), neg.reshape(n // 2, -1)
    for vals in ([1] * n, [1 + k % 2 for k in range(n)], [1 + k // 2 for k in range(n)]):
        _check(zo, pts, np.concatenate([zo.fr_from_u64(v) for v in vals]), 8)


# one to a few heavy buckets: up to 1024 heads after the first chunk go to one
# workgroup, more to one for each 512 (chunks of 8 here: 8200 entries are a tail
# and 1024 heads when the run starts a chunk)
@pytest.mark.parametrize("n", [2048, 8192, 8200, 8201, 8209, 12297, 12305, 30000, 70001])
def test_msm_heavy_buckets(gpu, zo, n):
    pts = zo.gen_bases_random(n, 77)
    one = zo.fr_from_u64(1)
    _check(zo, pts, np.repeat(one, n, axis=0), 8)
    rm1 = zo.to_mont([R - 1])
    sc = np.repeat(rm1, n, axis=0)
    sc[:: 3] = zo.fr_from_u64(200)
    sc[1:: 101] = zo.rand_fr(len(sc[1:: 101]), 78)
    _check(zo, pts, sc, 0)


def test_msm_heavy_bucket_equal_points(gpu, zo):
    """equal parts of one bucket (doublings when the parts are added) and parts
    that cancel"""
    n = 8 * 512 * 4
    pts = np.repeat(zo.gen_bases_random(1, 9).reshape(1, -1), n, axis=0)
    sc = np.repeat(zo.fr_from_u64(1), n, axis=0)
    _check(zo, pts, sc, 9)
    pts[n // 2:] = _negated(pts[n // 2:].reshape(n // 2, -1)).reshape(n // 2, -1)
    _check(zo, pts, sc, 9)
