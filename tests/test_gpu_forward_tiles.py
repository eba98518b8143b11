"""The large-grid forward kernels at the edges of their token tiles, each forced by its knob, against the
oracle: token counts that leave the last 32-, 64- or 128-token tile nearly empty or full (tiles of tokens
past the last are not launched), ragged rows, one super-block and several.  Rows of equal activations put
every code at 127, so the Q4_K kernel's sums of 16 codes are at their largest (2032), against weights whose
minima are at theirs.  y is an f32 sum of K / 32 (K / 256) block terms; both sides round each once, so 2e-6
of the largest value holds for the K here."""
import os

import numpy as np
import pytest

import oracle as O
import rust_trainer_amd as rt

pytestmark = pytest.mark.gpu

KNOBS = {"mm128": {"RTQ_FWD_MM": "1", "RTQ_FWD_I8": "0"}, "mm64": {"RTQ_FWD_MM": "2", "RTQ_FWD_I8": "0"},
         "mm32": {"RTQ_FWD_MM": "3"}, "i8": {"RTQ_FWD_MM": "2", "RTQ_FWD_I8": "1"}, "mmk": {"RTQ_FWD_MMK": "1"}, "auto": {}}


@pytest.fixture(scope="module", params=list(KNOBS))
def ctx(request):
    knobs = KNOBS[request.param]
    old = {k: os.environ.get(k) for k in knobs}
    os.environ.update(knobs)
    try:
        c = rt.Context(0)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v
    c.formats = (O.Q4_K, O.Q6_K) if request.param == "mmk" else (O.Q4_0, O.Q8_0) if knobs else (O.Q4_0, O.Q8_0, O.Q4_K, O.Q6_K)
    yield c
    c.close()


@pytest.mark.parametrize("n,k,t", [(130, 256, 17), (64, 512, 32), (200, 768, 33), (130, 512, 64), (257, 256, 65), (128, 512, 128),
                                   (144, 256, 129)])
def test_forward_token_tiles(ctx, n, k, t):
    for wtype in ctx.formats:
        w = O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k)
        w[: n // 2, : k // 2] = -0.05 + 0.001 * w[: n // 2, : k // 2]  # nearly all minimum
        x = O.Rng(2).vec_normal(t * k, 1.0).reshape(t, k)
        x[::3] = 0.75  # every code 127
        a = O.Rng(3).vec_normal(5 * k, 0.05).reshape(5, k)
        b = O.Rng(4).vec_normal(n * 5, 0.05).reshape(n, 5)
        blocks = O.quantize(wtype, w)
        lin = rt.Linear("tiles", rt.HipFrozen(wtype, blocks, n, k, ctx=ctx))
        y = lin.forward(x, t).reshape(t, n)
        want = np.asarray(O.frozen_forward(wtype, blocks, n, k, x, nthreads=8), np.float64).reshape(t, n)
        assert np.abs(y - want).max() <= 2e-6 * np.abs(want).max(), wtype
        lin.lora = rt.Lora(5, 10.0, a, b)
        y = lin.forward(x, t).reshape(t, n)
        want = want + 2 * (x.astype(np.float64) @ a.T.astype(np.float64)) @ b.T.astype(np.float64)
        assert np.abs(y - want).max() <= 2e-6 * np.abs(want).max(), wtype


def test_forward_nan_rows(ctx):
    """A token with a NaN gives NaN for every output on every kernel of the Q8_0 activations, the int8 ones too (a
    NaN has no code there), and leaves the other tokens as they were.  (Q8_K's quantiser caps a code at 127, a NaN
    among them.)"""
    n, k, t = 130, 512, 70
    formats = set(ctx.formats) & {O.Q4_0, O.Q8_0}
    if not formats:
        pytest.skip("no Q8_0 activations on this kernel")
    for wtype in formats:
        blocks = O.quantize(wtype, O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k))
        w = rt.HipFrozen(wtype, blocks, n, k, ctx=ctx)
        x = O.Rng(2).vec_normal(t * k, 1.0).reshape(t, k)
        plain = w.forward(x, t).reshape(t, n)
        x[3, 100], x[66] = np.nan, np.nan
        y = w.forward(x, t).reshape(t, n)
        bad = np.isin(np.arange(t), (3, 66))
        assert np.isnan(y[bad]).all(), wtype
        assert np.array_equal(y[~bad], plain[~bad]), wtype


@pytest.mark.parametrize("wtype,n,k,t,r,kernel", [
    (O.Q4_0, 8192, 1024, 140, 0, "rtq_mm32_q4_0"), (O.Q8_0, 16384, 512, 20, 0, "rtq_mm32_q8_0"),
    (O.Q4_0, 2048, 4096, 64, 0, "rtq_fwd_q4_0_w8r1"), (O.Q8_0, 8190, 640, 200, 0, "rtq_mm32_q8_0"),
    (O.Q4_0, 8192, 512, 1024, 0, "rtq_mm_q4_0"), (O.Q4_0, 8199, 512, 900, 0, "rtq_mm_q4_0"),
    (O.Q4_0, 8192, 512, 700, 0, "rtq_mmi8_64_q4_0"), (O.Q8_0, 3072, 4096, 512, 0, "rtq_fwd_q8_0_w8"),
    (O.Q8_0, 3072, 4096, 512, 64, "rtq_mm32_q8_0"), (O.Q6_K, 8697, 256, 119, 0, "rtq_mmk32_q6_k"),
    (O.Q4_K, 16384, 512, 31, 0, "rtq_fwd_q4_k_w"), (O.Q4_K, 24576, 512, 31, 0, "rtq_mmk32_q4_k"),
    (O.Q4_K, 6144, 256, 256, 16, "rtq_mmk32_q4_k"), (O.Q4_K, 6144, 256, 256, 0, "rtq_mmk64_q4_k"),
    (O.Q6_K, 6144, 2048, 448, 0, "rtq_fwd_q6_k_w"), (O.Q6_K, 2489, 1024, 430, 16, "rtq_fwd_q6_k_w"),
    (O.Q6_K, 2489, 1024, 430, 64, "rtq_mmk32_q6_k"), (O.Q6_K, 6144, 1024, 520, 64, "rtq_mmk64_q6_k")])
def test_default_forward_kernels(wtype, n, k, t, r, kernel):
    """Which kernel the default context takes on both sides of its rules' lines, each against the oracle."""
    c = rt.Context(0)
    blocks = O.quantize(wtype, O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k))
    x = O.Rng(2).vec_normal(t * k, 1.0).reshape(t, k)
    lin = rt.Linear("default", rt.HipFrozen(wtype, blocks, n, k, ctx=c))
    want = np.asarray(O.frozen_forward(wtype, blocks, n, k, x, nthreads=8), np.float64).reshape(t, n)
    if r:
        a, b = O.Rng(3).vec_normal(r * k, 0.05).reshape(r, k), O.Rng(4).vec_normal(n * r, 0.05).reshape(n, r)
        lin.lora = rt.Lora(r, 2.0 * r, a, b)
        want += 2 * (x.astype(np.float64) @ a.T.astype(np.float64)) @ b.T.astype(np.float64)
    c.set_timing(True)
    y = lin.forward(x, t).reshape(t, n)
    ran = c.timing()
    c.close()
    assert kernel in ran, ran
    assert np.abs(y - want).max() <= 2e-6 * np.abs(want).max()
