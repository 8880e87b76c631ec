"""Child process of test_alloc_fault_gpu.py: k-means steps on a point set (qvh_points_*, include/qvh.h)
with the device allocation numbered QVH_FAULT_ALLOC failing. A set_centroids that fails leaves no
centroids, so that a step is refused; a nearest that fails leaves the steps of the installed
centroids as they were. Prints the calls that met the failure, then "state ok"."""

import ctypes as C
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "tests"))

from qvh_ctypes import LIB  # noqa: E402

vp = C.c_void_p
L = C.CDLL(LIB)
L.qvh_last_error.restype = C.c_char_p
L.qvh_points_create.argtypes = [vp, C.c_uint64, C.c_uint32, C.POINTER(vp)]
L.qvh_points_destroy.argtypes = [vp]
L.qvh_points_nearest.argtypes = [vp, vp, C.c_uint32, C.c_int, vp]
L.qvh_points_set_centroids.argtypes = [vp, vp, C.c_uint32, C.c_uint32]
L.qvh_points_step.argtypes = [vp, vp]


def ptr(a):
    return a.ctypes.data_as(vp)


def counts_of(x, cent):
    d = ((x[:, None, :].astype(np.float64) - cent[None]) ** 2).sum(2)
    return np.bincount(d.argmin(1), minlength=cent.shape[0])


def injected(status):
    if status == 0:
        return False
    assert b"injected allocation failure" in L.qvh_last_error(), L.qvh_last_error()
    return True


def main():
    rng = np.random.default_rng(0)
    x = rng.standard_normal((1_000, 6)).astype(np.float32)
    few, many = x[:3].copy(), np.ascontiguousarray(np.tile(x, (5, 1)))
    h = vp()
    if injected(L.qvh_points_create(ptr(x), x.shape[0], 6, C.byref(h))):
        print("fault at create")
        print("state ok")
        return
    counts = np.zeros(many.shape[0], np.uint32)

    def install_and_step(cent):
        if injected(L.qvh_points_set_centroids(h, ptr(cent), cent.shape[0], 1)):
            print("fault at set_centroids", cent.shape[0], flush=True)
            assert L.qvh_points_step(h, ptr(counts)) == -22 and b"no centroids" in L.qvh_last_error()
            assert L.qvh_points_set_centroids(h, ptr(cent), cent.shape[0], 1) == 0  # the failure comes once
        if injected(L.qvh_points_step(h, ptr(counts))):
            print("fault at step", flush=True)
            assert L.qvh_points_step(h, ptr(counts)) == 0
        assert np.array_equal(counts[: cent.shape[0]].astype(np.int64), counts_of(x, cent))

    install_and_step(few)
    install_and_step(many)
    install_and_step(few)
    huge = np.ascontiguousarray(np.tile(many, (3, 1)))
    assign = np.zeros(x.shape[0], np.uint32)
    if injected(L.qvh_points_nearest(h, ptr(huge), huge.shape[0], 0, ptr(assign))):
        print("fault at nearest", flush=True)
    L.qvh_points_step(h, ptr(counts))  # of the means that the step before left
    assert int(counts[:3].sum()) == x.shape[0] and (counts[:3] > 0).all()
    L.qvh_points_destroy(h)
    print("state ok", flush=True)


if __name__ == "__main__":
    main()
