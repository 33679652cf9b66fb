"""Run by test_matmul_forms.py in a process of its own, with the stand-in
runtime: matmul_forms_check.py RUNTIME, cases (rows, K, B, plan) as JSON on
stdin; prints for each the matmul_kernel instance it launches, [NW, TM, CT,
KS, half8, plan], and its workgroups."""
import ctypes
import json
import re
import sys

import fake_hip

rt, lib = fake_hip.load(sys.argv[1])
P = ctypes.c_void_p
ctx = P()
assert lib.w4a8_ctx_create(0, ctypes.byref(ctx)) == 0
img = (ctypes.c_char * 64)()
at = P((ctypes.addressof(img) + 15) & ~15)   # never read: kernels do nothing


def weights(rows, K):
    w = P()
    assert lib.w4a8_weights_upload_async(ctx, at, ctypes.c_int64(rows), K, 4,
                                         ctypes.byref(w)) == 0
    return w


out = []
for rows, K, B, plan in json.load(sys.stdin):
    Ks = K if isinstance(K, list) else [K] * len(rows)
    ws = [weights(n, k) for n, k in zip(rows, Ks)]
    if plan:
        p = P()
        assert lib.w4a8_mplan_create(ctx, B, ctypes.byref(p)) == 0
        assert all(lib.w4a8_mplan_add(p, w, at, at) == 0 for w in ws)
        assert lib.w4a8_mplan_run(p) == 0
        lib.w4a8_mplan_destroy(p)
    else:
        many = P * len(ws)
        assert lib.w4a8_matmul_y32_multi_async(ctx, len(ws), many(*ws), many(*[at] * len(ws)), B,
                                               many(*[at] * len(ws))) == 0
    grid = ctypes.c_uint()
    name = rt.fake_last_kernel(ctypes.byref(grid)).decode()
    form = re.search(r"matmul_kernelI((?:L[ib]\d+E)+)E", name)
    out.append([[int(v) for v in re.findall(r"L[ib](\d+)E", form[1])], grid.value])
    for w in ws:
        lib.w4a8_weights_free(w)
print(json.dumps(out))
