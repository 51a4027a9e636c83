"""CPU: the window msm() takes in buffers of the reference driver's layout
(src/cuda/msm.rs:269-311), at sizes between the powers of two whose buffers hold
the default window's arrays with the large sort tiles' histogram only."""
import ctypes

import pytest

from zkprover._lib import lib


@pytest.mark.parametrize("count,n", [(1, 241001), (1, 246001), (2, 283001), (4, 340001), (8, 430001), (2, 530001),
                                     (4, 640001), (8, 800001), (2, 1050001), (4, 1200001), (8, 1600001)])
def test_default_window_between_powers_of_two(count, n):
    L = lib()
    wb, w, k = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    L.zkp_msm_policy.restype = None
    L.zkp_msm_policy(count, n, ctypes.byref(wb), ctypes.byref(w), ctypes.byref(k))
    assert L.zk_msm_plan_window(n, w.value, wb.value, k.value) == L.zk_msm_default_window(n)
