"""The batched kernel's unit shapes at their edges: split and shared units,
one and two tiles a wavefront, every count of token tiles, partial quads of
groups, ragged rows, and more units than workgroups.  Whole numbers, compared
bit for bit with the C oracle per token."""
import numpy as np
import pytest

from helpers import rand_image
from oracle import cfast, law

pytestmark = pytest.mark.gpu

GUARD = 0x5A5A5A5A


@pytest.mark.parametrize("rows,K,B", [
    # split: the wavefronts take quads of groups (NG 1, 9, 17, 27, 33, 96)
    ([16], 128, 1), ([40, 17], 1152, 8), ([100], 3456, 9), ([33], 4224, 16),
    ([300], 12288, 17), ([50], 4224, 32), ([33], 640, 48), ([70, 16], 2176, 64),
    ([9600], 2176, 8),          # 600 units on 512 workgroups
    # shared: one tile a wavefront (the last unit holds one tile)
    ([12290], 2176, 8), ([6150], 256, 33), ([6200], 896, 16), ([6145, 5], 3456, 64),
    # shared: two tiles a wavefront
    ([16400], 128, 5), ([16385, 17], 1152, 64), ([16384, 100], 2176, 20), ([16500], 640, 48),
    ([65700], 128, 3),          # 514 units on 512 workgroups
])
def test_matmul_units(engine, rows, K, B):
    import torch
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
    try:
        torch.cuda.synchronize()
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
