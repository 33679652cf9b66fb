"""gemv_kernel's ways to share tiles: teams of four wavefronts, one team of
twelve (no second tile per workgroup, more than four blocks a tile), and in
step (more than two tiles a team), at the edges of each, for every prologue
and for the widths where its pieces end.  Whole numbers, compared bit for bit
with the oracle."""
import numpy as np
import pytest

from fable5_llm_amd import _native as N
from helpers import activation_x16, norm_weight_q14, rand_image
from oracle import cfast, law

pytestmark = pytest.mark.gpu


def _expect(img, n, K, sh, pro, x, nw):
    if pro == N.PRO_RMSNORM_DYNQ8:
        x = np.asarray(law.rmsnorm_fx(x, nw, 7, True), dtype=np.int16)
    x8, e = (x, 0) if pro == N.PRO_X8 else cfast.dyn_quant_i8(x)
    return cfast.matvec_y32_img(img, n, K, sh, x8), x8, e


@pytest.mark.parametrize("pro", [N.PRO_X8, N.PRO_DYNQ8, N.PRO_RMSNORM_DYNQ8])
@pytest.mark.parametrize("rows,K", [
    (16, 128), (100, 640), (272, 1024),           # one block or none per wavefront
    (4096, 4096), (4097, 4096), (4113, 1024),     # 256 tiles, one more, two more
    (33, 4224), (4096, 12288), (4096, 8192), (300, 5248),   # one team of twelve
    (4100, 8192),                                 # ... and a tile too many for it
    (8200, 2048), (12289, 4096), (12304, 8192),   # up to three and four tiles a workgroup
    (24576, 1024), (24570, 4224), (24576, 128),   # two a team
    (24592, 1024), (24592, 4224), (24590, 128),   # two a team and one more: in step from here
    (40000, 512), (37000, 3200),
])
def test_gemv_teams(engine, pro, rows, K):
    if pro == N.PRO_RMSNORM_DYNQ8 and (K & (K - 1) or K > 8192):
        pytest.skip("RMSNorm takes powers of two up to 8192")
    rng = np.random.default_rng(rows + K + pro)
    img, _ = rand_image(rng, rows, K)
    sh = law.sh_for_k(K)
    if pro == N.PRO_X8:
        x = rng.integers(-128, 128, K).astype(np.int8)
    else:
        x = activation_x16(rng, K)
    nw = (norm_weight_q14(rng, K) - (1 << 14)).astype(np.int16)
    want, x8, e = _expect(img, rows, K, sh, pro, x, nw)
    w = engine.upload(img, rows, K, sh)
    try:
        for _ in range(2):
            got, gx8, ge, _ = engine.matvec_fused(w, x, prologue=pro, epilogue=N.EPI_Y32,
                                                  norm_w=nw, in_f=7, one_plus=True)
            assert np.array_equal(gx8, x8) and ge == e
            assert np.array_equal(got, want)
    finally:
        w.free()


@pytest.mark.parametrize("fill", [0, 1, 127, 128, 255, 32767, -32768, "mixed"])
@pytest.mark.parametrize("K", [128, 4096, 8192])
def test_prologue_extremes(engine, fill, K):
    # DYNQ8 and RMSNorm at the int16 rails, zero and the exponent's edges
    rng = np.random.default_rng(K)
    x = rng.choice(np.array([-32768, 32767, 0, 1, -1, 255, -129], np.int16), K) \
        if fill == "mixed" else np.full(K, fill, np.int16)
    nw = rng.choice(np.array([-32768, 32767, 0, -16384, -16385, 100], np.int16), K)
    img, _ = rand_image(rng, 40, K)
    sh = law.sh_for_k(K)
    w = engine.upload(img, 40, K, sh)
    try:
        got, x8, e, _ = engine.matvec_fused(w, x, prologue=N.PRO_DYNQ8)
        wx8, we = law.dyn_quant_i8(x)
        assert np.array_equal(x8, wx8) and e == we
        assert np.array_equal(got, cfast.matvec_y32_img(img, 40, K, sh, wx8))
        for in_f in (0, 7, 40):
            for one in (False, True):
                xn = np.asarray(law.rmsnorm_fx(x, nw, in_f, one), dtype=np.int16)
                got, x8, e, gxn = engine.matvec_fused(
                    w, x, prologue=N.PRO_RMSNORM_DYNQ8, norm_w=nw, in_f=in_f, one_plus=one)
                assert np.array_equal(gxn, xn)
                assert np.array_equal(engine.rmsnorm(x, nw, in_f, one), xn)
                wx8, we = law.dyn_quant_i8(xn)
                assert np.array_equal(x8, wx8) and e == we
    finally:
        w.free()


@pytest.mark.parametrize("K", [128, 1152, 2176, 4096])   # 1, 2, 3 and 4 blocks a tile
def test_argmax_in_step(engine, K):
    # a long head: the winner, and a tie after it, in a tile that each of a
    # team's four wavefronts finishes, those without blocks of it too
    G = engine.grid
    rows = (9 * G + 200) * 16 - 7            # four tile iterations for team 0
    rng = np.random.default_rng(K)
    img, _ = rand_image(rng, rows, K)
    x16 = activation_x16(rng, K)
    x8, _ = law.dyn_quant_i8(x16)
    sh = law.sh_for_k(K)
    best, _ = law.pack_ddr_rows(np.where(x8 >= 0, 7, -8).astype(np.int8)[None],
                                np.full((1, K // 128), 65535, np.uint16))
    best = np.frombuffer(best, np.uint8) if isinstance(best, bytes) else np.asarray(best).reshape(-1)
    for it in range(4):
        im = img.reshape(rows, -1).copy()
        win = (3 * G * it + 5) * 16 + 3      # tile 5 of team 0's iteration
        im[win] = best
        im[win + 16] = best                  # the next workgroup's tile
        w = engine.upload(im.reshape(-1), rows, K, sh)
        try:
            want = law.amax32(cfast.matvec_y32_img(im.reshape(-1), rows, K, sh, x8))
            assert want[0] == win
            assert tuple(engine.head_argmax(w, x16, prologue=N.PRO_DYNQ8)) == tuple(want), it
        finally:
            w.free()
