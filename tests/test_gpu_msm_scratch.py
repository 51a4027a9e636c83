"""GPU: MSMs in scratch of sizes that callers have kept (what
zk_msm_scratch_bytes and zk_msm_batch_scratch_bytes asked for when the bucket
reduction had two points per eight buckets as its own arrays), among them the
narrowest windows: accepted, with the oracle's result."""
import ctypes

import numpy as np
import pytest

from test_gpu_msm_table import OUT_BYTES, _decl, _Item, _table

pytestmark = pytest.mark.gpu


def _run(pts, sets, c, table_c, nbytes):
    import torch
    from zkprover import device as dv
    from zkprover._lib import call
    L = _decl()
    L.zk_msm.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_size_t,
                                                 ctypes.c_void_p]
    keep, items = [], (_Item * len(sets))()
    for m, s in enumerate(sets):
        dp, ds = dv.to_dev(pts[:len(s)].reshape(-1, 4)), dv.to_dev(s)
        src = _table(dp, len(s), table_c) if table_c else dp
        keep += [dp, ds, src]
        items[m] = _Item(src.data_ptr(), ds.data_ptr(), len(s), table_c)
    scratch = torch.empty(nbytes, dtype=torch.uint8, device=dv.device())
    out = torch.zeros(len(sets) * OUT_BYTES, dtype=torch.uint8, device=dv.device())
    if len(sets) == 1 and not table_c:
        call("zk_msm", out.data_ptr(), keep[0].data_ptr(), keep[1].data_ptr(), len(sets[0]), c, scratch.data_ptr(),
             nbytes, dv.stream_handle())
    else:
        call("zk_msm_batch", out.data_ptr(), ctypes.addressof(items), len(sets), c, scratch.data_ptr(), nbytes,
             dv.stream_handle())
    return out.view(len(sets), OUT_BYTES)[:, :96].cpu().numpy().copy().view(np.uint64)


@pytest.mark.parametrize("ns,c,table_c,nbytes", [
    ([1], 2, 0, 84992), ([5], 4, 0, 115200), ([347], 13, 0, 15409408), ([3, 14, 9], 2, 0, 382464),
    ([33, 20, 5], 8, 0, 2396160), ([31], 0, 15, 3113472), ([14], 0, 16, 6108416)])
def test_msm_in_kept_scratch(gpu, zo, ns, c, table_c, nbytes):
    pts = zo.gen_bases_random(max(ns), 60 + max(ns))
    sets = [zo.rand_fr(n, 70 + m) for m, n in enumerate(ns)]
    got = _run(pts, sets, c, table_c, nbytes)
    for n, s, g in zip(ns, sets, got):
        assert (zo.g1_to_affine(g.reshape(1, 12)) == zo.g1_to_affine(zo.msm(pts[:n], s))).all(), n
