"""Host-buffer calls through the context's pinned block: results on both
sides of the block's size, calls of different sizes one after another, and
the error word, which matvec reports and clears and the elementwise calls
leave alone."""
import numpy as np
import pytest

from fable5_llm_amd import _native as N
from helpers import activation_x16, rand_image
from oracle import cfast, law

pytestmark = pytest.mark.gpu


def test_sizes_around_the_block(engine):
    K = 128
    rng = np.random.default_rng(5)
    sh = law.sh_for_k(K)
    # int32 results plus x8 and e_x: 40832 rows are the most that fit
    ws, imgs = {}, {}
    for n in (40832, 16, 40833, 50000):
        imgs[n] = rand_image(rng, n, K)[0]
        ws[n] = engine.upload(imgs[n], n, K, sh)
    try:
        for n in (40832, 16, 40833, 40832, 50000, 16):
            x = activation_x16(rng, K)
            got, x8, e, _ = engine.matvec_fused(ws[n], x, prologue=N.PRO_DYNQ8)
            wx8, we = law.dyn_quant_i8(x)
            assert e == we and np.array_equal(x8, wx8)
            assert np.array_equal(got, cfast.matvec_y32_img(imgs[n], n, K, sh, wx8)), n
    finally:
        for w in ws.values():
            w.free()


def test_pending_overflow_is_matvecs_to_report(engine):
    import torch
    K, n = 4096, 48
    rng = np.random.default_rng(6)
    img, _ = rand_image(rng, n, K, np.full((n, K // 128), 65535, np.uint16))
    img.reshape(n, -1)[:, :K // 2] = 0x88
    w = engine.upload(img, n, K, 0)
    good_img, _ = rand_image(rng, n, K)
    good = engine.upload(good_img, n, K, law.sh_for_k(K))
    dev = torch.device("cuda", 0)
    x = torch.full((K,), -128, dtype=torch.int8, device=dev)
    y = torch.zeros(n, dtype=torch.int32, device=dev)
    x8 = rng.integers(-128, 128, K).astype(np.int8)
    x16 = activation_x16(rng, 4096)
    try:
        torch.cuda.synchronize()
        engine.site_async([w], [N.EPI_Y32], [0], [y], x, prologue=N.PRO_X8)
        wx8, we = law.dyn_quant_i8(x16)
        got, e = engine.dynq8(x16)
        assert e == we and np.array_equal(got, wx8)
        with pytest.raises(AssertionError, match="y32 overflow"):
            engine.matvec_y32(good, x8)
        assert np.array_equal(engine.matvec_y32(good, x8),
                              cfast.matvec_y32_img(good_img, n, K, law.sh_for_k(K), x8))
        engine.sync()
    finally:
        w.free()
        good.free()


def test_epilogue_and_p0_arguments(engine):
    import torch
    dev = torch.device("cuda", 0)
    img, _ = rand_image(np.random.default_rng(7), 16, 128)
    w = engine.upload(img, 16, 128, 4)
    x = torch.zeros(128, dtype=torch.int8, device=dev)
    y = torch.zeros(16, dtype=torch.int32, device=dev)
    try:
        for eps, p0s in (([0], [0]), ((0,), (0,)), (np.array([0]), np.array([0]))):
            engine.site_async([w], eps, p0s, [y], x, prologue=N.PRO_X8)
        with pytest.raises(OverflowError):
            engine.site_async([w], [0], [1 << 31], [y], x, prologue=N.PRO_X8)
        with pytest.raises(ValueError, match="device tensor"):
            engine.site_async([w], [0], [0], [y], x.cpu(), prologue=N.PRO_X8)
        with pytest.raises(ValueError, match="contiguous"):
            engine.site_async([w], [0], [0], [torch.zeros(32, dtype=torch.int32, device=dev)[::2]],
                              x, prologue=N.PRO_X8)
        with pytest.raises(ValueError, match="bytes"):
            engine.site_async([w], [0], [0], [y[:15]], x, prologue=N.PRO_X8)
        engine.sync()
    finally:
        w.free()
