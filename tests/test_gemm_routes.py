"""Which kernel takes a Q4_K product: the shapes of the GEMM tests reach every
kernel and K split they are there for (the choice is by time models, so a refit
could move a shape to another kernel unseen)."""
from __future__ import annotations

import ctypes

import pytest

Q4K = 1
KERNELS = ("eight-wave", "half-block", "ping-pong")


def route(rt, m, n, k):
    """(kernel, K splits) of a Q4_K product m x n x k."""
    def fn(name, args, res):
        f = rt.lib()[name]
        f.argtypes, f.restype = args, res
        return f
    i, b = ctypes.c_int, ctypes.c_bool
    if fn("_ZN2rt12rows_gemm_okEiiii", [i] * 4, b)(Q4K, m, n, k):
        return "few-row", None
    if fn("_ZN2rt14q4k_gemm_widenEiii", [i] * 3, b)(m, n, k):
        return "widened", None
    v = fn("_ZN2rt15q4k_gemm_kernelEiiib", [i, i, i, b], i)(m, (n + 255) // 256, k, False)
    return KERNELS[v & 15], v >> 4


# of test_gpu_gemm.py and test_gemm_tiles.py
@pytest.mark.parametrize("m,n,k,kernel,splits", [
    (2, 256, 256, "few-row", None), (17, 300, 512, "few-row", None), (130, 260, 768, "few-row", None),
    (64, 2048, 2560, "few-row", None), (512, 10240, 2560, "eight-wave", 1), (512, 2560, 10240, "eight-wave", 6),
    (1100, 1024, 2560, "widened", None), (2100, 2560, 10240, "ping-pong", 2), (1024, 2560, 2048, "widened", None),
    (1025, 2560, 2048, "widened", None), (1000, 16384, 512, "half-block", 1),
    (4608, 9216, 3072, "ping-pong", 1), (4608, 12288, 3072, "ping-pong", 1), (4608, 3072, 12288, "ping-pong", 1),
    (4096, 2560, 10240, "ping-pong", 1), (4096, 2560, 2048, "ping-pong", 1), (1500, 5632, 8192, "ping-pong", 1),
    (1300, 9000, 2560, "ping-pong", 1),
    (1300, 6001, 1024, "ping-pong", 1), (1537, 5120, 256, "widened", None), (2305, 3000, 512, "half-block", 1),
    (1100, 1500, 10240, "half-block", 4), (1400, 259, 3584, "widened", None), (600, 10241, 768, "eight-wave", 1),
    (1847, 2146, 3840, "widened", None), (601, 4378, 5632, "ping-pong", 3),
])
def test_q4k_gemm_route(rt, m, n, k, kernel, splits):
    assert route(rt, m, n, k) == (kernel, splits)
