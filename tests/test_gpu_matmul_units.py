"""The batched kernel's unit shapes at their edges: split and shared units,
one and two tiles a wavefront, every count of token tiles, partial quads of
groups, ragged rows, and more units than workgroups, as one launch and as a
matmul plan.  Whole numbers, compared bit for bit with the C oracle per
token."""
import numpy as np
import pytest

from helpers import rand_image
from oracle import cfast, law

pytestmark = pytest.mark.gpu

GUARD = 0x5A5A5A5A


# The forms on 256 CUs: wavefronts, tiles a wavefront, wavefronts a tile is
# split over (test_matmul_forms.py checks that each case takes its own, and
# that every instance of the kernel has one).
CASES = {
    # split: the wavefronts take quads of groups (NG 1, 9, 17, 27, 33, 96)
    (4, 1, 4): [
        ([16], 128, 1), ([40, 17], 1152, 8), ([100], 3456, 9), ([33], 4224, 16),
        ([300], 12288, 17), ([50], 4224, 32), ([33], 640, 48), ([70, 16], 2176, 64),
        ([9600], 2176, 8), ([8300, 40], 6272, 16)],     # 600 and 522 units on 512 workgroups
    # shared: one tile a wavefront (the last unit holds one tile)
    (4, 1, 1): [
        ([12290], 2176, 8), ([6150], 256, 33), ([6200], 896, 16), ([6145, 5], 3456, 64),
        ([6150], 640, 24), ([12290], 2176, 20)],
    # ... on eight wavefronts, beyond a unit of four tiles per CU
    (8, 1, 1): [
        ([16400], 128, 5), ([16385, 17], 1152, 64), ([16384, 100], 2176, 20), ([16500], 640, 48)],
    # shared: two tiles a wavefront, beyond 8 tiles per CU
    (4, 2, 1): [
        ([65700], 128, 3),                              # 514 units on 512 workgroups
        ([32770, 20], 256, 24), ([40000], 128, 40), ([32770], 128, 64)],
}


@pytest.mark.parametrize("plan", [False, True])
@pytest.mark.parametrize("rows,K,B", sum(CASES.values(), []))
def test_matmul_units(engine, rows, K, B, plan):
    import torch

    from fable5_llm_amd.engine import MatmulPlan
    rng = np.random.default_rng(sum(rows) + K + B)
    sh = law.sh_for_k(K)
    imgs = [rand_image(rng, n, K)[0] for n in rows]
    x = rng.integers(-128, 128, (B, K)).astype(np.int8)
    dev = torch.device("cuda", 0)
    xd = torch.from_numpy(x).to(dev)
    pad = 64
    out = torch.full((sum(B * n + pad for n in rows),), GUARD, dtype=torch.int32, device=dev)
    ys, at = [], 0
    for n in rows:
        ys.append(out[at:at + B * n].view(B, n))
        at += B * n + pad
    ws = [engine.upload(i, n, K, sh) for i, n in zip(imgs, rows)]
    p = MatmulPlan(engine, B) if plan else None
    try:
        torch.cuda.synchronize()
        if plan:
            for w, y in zip(ws, ys):
                p.add(w, xd, y)
            p.run()
        else:
            engine.matmul_multi_async(ws, [xd] * len(ws), ys)
        engine.sync()
        at = 0
        for i, n, y in zip(imgs, rows, ys):
            got = y.cpu().numpy()
            for b in range(B):
                assert np.array_equal(got[b], cfast.matvec_y32_img(i, n, K, sh, x[b])), b
            at += B * n
            assert (out[at:at + pad].cpu().numpy() == GUARD).all(), "written past the output"
            at += pad
    finally:
        if p is not None:
            p.close()
        for w in ws:
            w.free()


# split plans whose workgroups go on from a tile of one K to a tile of
# another: 513 to 768 tiles, the longest first
MIXED = [([3000, 4096, 4100, 9], [384, 4224, 1152, 128], 1),
         ([3000, 4096, 4100, 9], [384, 4224, 1152, 128], 8),
         ([1500, 9000, 9], [12288, 6272, 128], 16)]


@pytest.mark.parametrize("rows,K,B", MIXED)
def test_split_plan_of_several_k(engine, rows, K, B):
    import torch

    from fable5_llm_amd.engine import MatmulPlan
    rng = np.random.default_rng(B)
    dev = torch.device("cuda", 0)
    imgs = [rand_image(rng, n, k)[0] for n, k in zip(rows, K)]
    xs = [rng.integers(-128, 128, (B, k)).astype(np.int8) for k in K]
    xd = [torch.from_numpy(x).to(dev) for x in xs]
    ys = [torch.full((B, n), GUARD, dtype=torch.int32, device=dev) for n in rows]
    ws = [engine.upload(i, n, k, law.sh_for_k(k)) for i, n, k in zip(imgs, rows, K)]
    p = MatmulPlan(engine, B)
    try:
        torch.cuda.synchronize()
        for w, x, y in zip(ws, xd, ys):
            p.add(w, x, y)
        for _ in range(2):
            for y in ys:
                y.fill_(GUARD)
            torch.cuda.synchronize()
            p.run()
            engine.sync()
            for i, n, k, x, y in zip(imgs, rows, K, xs, ys):
                got = y.cpu().numpy()
                for b in range(B):
                    assert np.array_equal(
                        got[b], cfast.matvec_y32_img(i, n, k, law.sh_for_k(k), x[b])), (n, k, b)
    finally:
        p.close()
        for w in ws:
            w.free()


@pytest.mark.parametrize("rows,B", [(48, 2), (48, 40), (16400, 2)])
def test_matmul_overflow_reported(engine, rows, B):
    # the last row of the last token overflows y32 (sh 0, the largest scale
    # and codes); every other row is small
    rng = np.random.default_rng(rows + B)
    K = 4096
    m = np.ones((rows, K // 128), dtype=np.uint16)
    m[-1] = 65535
    img, _ = rand_image(rng, rows, K, m)
    im = img.reshape(rows, -1)
    im[-1, :K // 2] = 0x88
    x = rng.integers(-4, 5, (B, K)).astype(np.int8)
    x[-1] = -128
    w = engine.upload(img, rows, K, 0)
    try:
        with pytest.raises(AssertionError, match="y32 overflow"):
            engine.matmul_y32(w, x)
        x[-1] = 0
        got = engine.matmul_y32(w, x)
        for b in range(B):
            assert np.array_equal(got[b], cfast.matvec_y32_img(img, rows, K, 0, x[b]))
    finally:
        w.free()
