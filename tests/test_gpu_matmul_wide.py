"""The batched kernel's units of eight wavefronts at their edges: one tile each
(beyond a unit of four tiles per CU, up to 8 tiles per CU) and two (beyond,
where the rounds are nearly full), with every count of token tiles, quads of
groups that end early, ragged rows and last units of one tile; and the
four-wavefront units on the other side of each line.  Whole numbers, compared bit for bit with the C oracle per token."""
import numpy as np
import pytest

from helpers import rand_image
from oracle import cfast, law

pytestmark = pytest.mark.gpu

GUARD = 0x5A5A5A5A


# The forms on 256 CUs, as in test_gpu_matmul_units.py
CASES = {
    # four wavefronts of one tile: 1024 tiles, a unit on every CU
    (4, 1, 1): [([16369], 128, 1)],
    # eight of one tile: up to 2048 tiles
    (8, 1, 1): [([16400, 20], 1152, 9), ([16600], 640, 33), ([32768], 256, 64)],
    # four of two tiles: past 2048 tiles, rounds not full; and up to 8 tokens
    (4, 2, 1): [([32770], 128, 17), ([60001], 128, 8)],
    # eight of two tiles: 233 to 253 units on as many workgroups, 510 on 256
    (8, 2, 1): [([60001], 128, 9), ([64497, 5], 384, 17), ([59500], 640, 48), ([130400], 128, 64)],
}


@pytest.mark.parametrize("plan", [False, True])
@pytest.mark.parametrize("rows,K,B", sum(CASES.values(), []))
def test_matmul_wide_units(engine, rows, K, B, plan):
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
