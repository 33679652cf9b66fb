"""Run by test_host_io.py in a process of its own, with the stand-in runtime
loaded before the library: host_io_check.py RUNTIME CHECK."""
import ctypes
import sys

import numpy as np

import fake_hip

E_HIP, E_Y32_OVF, E_RANGE = -5, -4, -7
PRO_RMSNORM_DYNQ8, EPI_Y32 = 2, 0
N_, K = 40, 256

rt, lib = fake_hip.load(sys.argv[1])
P = ctypes.c_void_p
ctx, w = P(), P()
assert lib.w4a8_ctx_create(0, ctypes.byref(ctx)) == 0
img = np.zeros((N_, 192), np.uint8)
assert lib.w4a8_weights_upload(ctx, P(img.ctypes.data), ctypes.c_int64(N_), K, 4,
                               ctypes.byref(w)) == 0

x, nw = np.zeros(K, np.int16), np.zeros(K, np.int16)
out, x8, xn = np.zeros(N_, np.int32), np.zeros(K, np.int8), np.zeros(K, np.int16)
e_x = np.zeros(1, np.int32)
OUTS = (out, x8, e_x, xn)


def ptr(a):
    return P(a.ctypes.data)


def call(in_f=7):
    """Status of one RMSNorm matvec, and whether each output was written."""
    for a in OUTS:
        a.fill(0x77)
    rc = lib.w4a8_matvec_fused(ctx, w, PRO_RMSNORM_DYNQ8, ptr(x), ptr(nw), in_f, 1, EPI_Y32, 0,
                               ptr(out), ptr(x8), ptr(e_x), ptr(xn))
    return rc, [bool((a != 0x77).all()) for a in OUTS], [bool((a == 0x77).all()) for a in OUTS]


def failed_copies():
    assert call()[:2] == (0, [True] * 4)
    # the launch that brings the results back, the stream's wait, the flag
    for how in ((3, 0, 0, 0), (0, 1, 1, 0), (0, 0, 1, 0)):
        rt.fake_set(*how)
        rc, _, kept = call()
        assert rc == E_HIP and kept == [True] * 4, (how, rc, kept)
        rt.fake_set(0, 0, 0, 0)
        assert call()[:2] == (0, [True] * 4)
    # an overflow is reported with the results, and cleared
    rt.fake_set(0, 0, 0, 1)
    assert call()[:2] == (E_Y32_OVF, [True] * 4)
    rt.fake_set(0, 0, 0, 0)
    assert call()[:2] == (0, [True] * 4)


def refused_calls():
    call()
    before = rt.fake_launches()
    rc, _, kept = call(in_f=41)
    assert rc == E_RANGE and kept == [True] * 4
    assert rt.fake_launches() == before, "a refused call left work on the stream"


{"failed_copies": failed_copies, "refused_calls": refused_calls}[sys.argv[2]]()
print("ok")
