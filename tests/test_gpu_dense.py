"""The split-bf16 products of the trainer-native weights (rtq_dense_*) against float64, at the edges of
their tiles: one token, 31 / 32 / 33 and 64 / 65 tokens, rows that leave a tile or a 32-row step ragged,
a row count that is no multiple of 4 (scalar dy loads), one 32-column block, enough tiles for the
64-token form either way, several row splits; each test asserts which kernels ran.  The strided f32 GEMM, which
takes the calls that do not fit these kernels, runs through the same cases (RTQ_DENSE_SPLIT=0).  An f32 dot of n terms is within (n / 2 + 2) 2^-24 of the sum of its
terms' magnitudes however it is ordered; the products here leave out terms below 2^-30 each, so the
bound below is (n / 16 + 4) 2^-24 of that sum (a rounding per 32-element step and of the split's parts)."""
import os

import numpy as np
import pytest

import oracle as O
import rust_trainer_amd as rt

pytestmark = pytest.mark.gpu

SHAPES = [(64, 32, 1), (37, 96, 31), (65, 64, 32), (200, 160, 33), (130, 256, 64), (257, 128, 65), (1030, 2048, 17),
          (4096, 1024, 600), (70, 4096, 520), (1030, 8192, 257)]


def _weight(ctx, kind, n, k):
    w = O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k)
    if kind == "f32":
        return rt.HipFrozen.f32(w, n, k, ctx=ctx), w.astype(np.float64)
    b = rt.pack_trainer_q8_0(w, n, k)
    nb = n * k // 32
    return (rt.HipFrozen(rt.TYPE_TQ8_0, b, n, k, ctx=ctx),
            (b[:4 * nb].view(np.float32).astype(np.float64)[:, None] * b[4 * nb:].view(np.int8).reshape(nb, 32)).reshape(n, k))


@pytest.fixture(scope="module")
def ctx():
    c = rt.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module", params=["split", "gemm"])
def either(request, ctx):
    if request.param == "split":
        yield "split", ctx
        return
    old = os.environ.get("RTQ_DENSE_SPLIT")
    os.environ["RTQ_DENSE_SPLIT"] = "0"
    try:
        c = rt.Context(0)
    finally:
        os.environ.pop("RTQ_DENSE_SPLIT") if old is None else os.environ.update(RTQ_DENSE_SPLIT=old)
    yield "gemm", c
    c.close()


def _kernels(kind, n, k, t):
    """The product kernels of a forward and a backward on 256 CUs."""
    tok = [64 if -(-out // 64) * -(-t // 64) >= 512 else 32 for out in (n, k)]
    q8 = "_q8" if kind == "tq8" else ""
    return {f"rtq_dense_fwd{tok[0]}{q8}", f"rtq_dense_bwd{tok[1]}{q8}"}


@pytest.mark.parametrize("kind", ["f32", "tq8"])
@pytest.mark.parametrize("n,k,t", SHAPES)
def test_dense_products(either, kind, n, k, t):
    path, ctx = either
    hw, w = _weight(ctx, kind, n, k)
    x = O.Rng(2).vec_normal(t * k, 1.0).reshape(t, k)
    dy = O.Rng(3).vec_normal(t * n, 1.0).reshape(t, n) * np.exp(O.Rng(4).vec_normal(t, 2.0))[:, None].astype(np.float32)
    a = O.Rng(5).vec_normal(7 * k, 0.05).reshape(7, k)
    b = O.Rng(6).vec_normal(n * 7, 0.05).reshape(n, 7)
    lin = rt.Linear("dense", hw, bias=O.Rng(7).vec_normal(n, 0.1))
    lin.lora = rt.Lora(7, 14.0, a, b)
    eps = 2.0 ** -24
    x64, dy64, a64, b64 = (v.astype(np.float64) for v in (x, dy, a, b))

    def close(got, want, size, terms):
        bound = terms / 16 + 4 if path == "split" else terms / 2 + 2
        assert (np.abs(np.asarray(got, np.float64).reshape(want.shape) - want) <= bound * eps * size).all()

    ctx.set_timing(True)
    ctx.reset_timing()
    y = lin.forward(x, t)
    h = x64 @ a64.T
    size = np.abs(x64) @ np.abs(w.T) + np.abs(lin.bias) + 2 * (np.abs(x64) @ np.abs(a64.T)) @ np.abs(b64.T)
    close(y, x64 @ w.T + lin.bias + 2 * h @ b64.T, 2 * size, k)
    dx = lin.backward(x, dy, t)
    size = np.abs(dy64) @ np.abs(w) + 2 * (np.abs(dy64) @ np.abs(b64)) @ np.abs(a64)
    close(dx, dy64 @ w + 2 * (dy64 @ b64) @ a64, 2 * size, n)
    close(lin.lora.ga, 2 * (dy64 @ b64).T @ x64, 2 * 2 * (np.abs(dy64) @ np.abs(b64)).T @ np.abs(x64), n + t)
    close(lin.lora.gb, 2 * dy64.T @ h, 2 * 2 * np.abs(dy64).T @ (np.abs(x64) @ np.abs(a64.T)), k + t)
    close(hw.forward(x, t), x64 @ w.T, np.abs(x64) @ np.abs(w.T), k)
    dx0 = O.Rng(8).vec_normal(t * k, 1.0)
    dx = dx0.copy()
    hw.backward_input(dy, t, dx)  # accumulates
    close(dx, dy64 @ w + dx0.reshape(t, k), np.abs(dy64) @ np.abs(w) + np.abs(dx0.reshape(t, k)), n)
    ran = {name for name in ctx.timing() if "dense" in name or "gemm" in name}
    ctx.set_timing(False)
    if path == "split":
        assert ran == _kernels(kind, n, k, t), ran
    else:
        assert ran and all(name.startswith("rtq_m_gemm") for name in ran - {"rtq_dense_bias"}), ran


@pytest.mark.parametrize("kind", ["f32", "tq8"])
def test_dense_products_keep_infinities(ctx, kind):
    """A product with an infinite operand is what f32 sums give, not the NaN of an infinity's split."""
    n, k, t = 70, 64, 40
    hw, w = _weight(ctx, kind, n, k)
    x = O.Rng(2).vec_normal(t * k, 1.0).reshape(t, k)
    dy = O.Rng(3).vec_normal(t * n, 1.0).reshape(t, n)
    x[3, 5], x[4, 6], x[5, 7], x[5, 8] = np.inf, np.nan, np.inf, -np.inf
    dy[7, 69], dy[8, 0] = -np.inf, np.nan
    y = hw.forward(x, t).reshape(t, n)
    dx = np.zeros(t * k, np.float32)
    hw.backward_input(dy, t, dx)
    with np.errstate(invalid="ignore"):
        for got, want in ((y, x.astype(np.float64) @ w.T), (dx.reshape(t, k), dy.astype(np.float64) @ w)):
            assert np.array_equal(np.isnan(got), np.isnan(want))
            inf = np.isinf(want)
            assert np.array_equal(got[inf], want[inf].astype(np.float32))
            assert np.isfinite(got[np.isfinite(want)]).all()


@pytest.mark.parametrize("kind", ["f32", "tq8"])
@pytest.mark.parametrize("n,k,t", [(65, 64, 33), (1030, 2048, 65)])
@pytest.mark.parametrize("unit", [0, -112, -118])
def test_dense_products_of_single_terms(ctx, kind, n, k, t, unit):
    """Rows with one non-zero element, as masked gradients have: each output is one product, so nothing averages
    out what the split leaves behind.  An f32 product is off by at most 2^-24; here the corrections' sum, up to
    2^-6 of the product, is rounded seven times more, which is 2^-24 (1 + 7 / 64).  TQ8_0's forward rounds the
    product with the code, then that with the scale, and the corrections twice.  Small values (2^unit), whose planes
    or products are denormal, keep that; an output below the least normal value may be zero."""
    hw, w = _weight(ctx, kind, n, k)
    r = np.random.RandomState(1)
    x, dy = np.zeros((t, k), np.float32), np.zeros((t, n), np.float32)
    xc, dc = r.randint(0, k, t), r.randint(0, n, t)
    x[np.arange(t), xc] = np.exp(r.randn(t)) * 2.0 ** unit
    dy[np.arange(t), dc] = -np.exp(3 * r.randn(t)) * 2.0 ** unit
    eps = 2.0 ** -24
    y = hw.forward(x, t).reshape(t, n)
    want = x[np.arange(t), xc].astype(np.float64)[:, None] * w[:, xc].T
    assert (np.abs(y - want) <= (2.125 if kind == "tq8" else 1.125) * eps * np.abs(want) + 2.0 ** -126).all()
    dx = np.zeros(t * k, np.float32)
    hw.backward_input(dy, t, dx)
    want = dy[np.arange(t), dc].astype(np.float64)[:, None] * w.astype(np.float32)[dc]  # codes decoded to f32
    assert (np.abs(dx.reshape(t, k) - want) <= 1.125 * eps * np.abs(want) + 2.0 ** -126).all()


@pytest.mark.parametrize("kind", ["f32", "tq8"])
def test_dense_products_of_nan_rows_take_their_time(ctx, kind):
    """A diverged run's NaN activations and gradients: their products are NaN, by the second sum that keeps
    infinities apart, at a small multiple of the ordinary time (the second sum runs on the f32 MFMA, a sixteenth
    of the bf16 one's rate, without the first one's staging)."""
    n, k, t = 1024, 1024, 512
    hw, _ = _weight(ctx, kind, n, k)

    def ms(x):
        ctx.set_timing(True)
        ctx.reset_timing()
        for _ in range(3):
            out = hw.forward(x, t)
            hw.backward_input(x, t, np.zeros(t * k, np.float32))
        ran = {name: v for name, v in ctx.timing().items() if name.startswith("rtq_dense")}
        ctx.set_timing(False)
        assert len(ran) == 2, ran
        return sum(v[1] for v in ran.values()), out

    x = O.Rng(2).vec_normal(t * k, 1.0)
    ms(x)
    plain, _ = ms(x)
    slow, out = ms(np.full(t * k, np.nan, np.float32))
    assert np.isnan(out).all()
    assert slow <= 20 * plain, (slow, plain)


@pytest.mark.parametrize("kind", ["f32", "tq8"])
def test_dense_products_of_large_values(ctx, kind):
    """Operands near the top of f32's range whose products with the weight are far from it: a block's sum with
    the codes (up to 127) overflows before its scale (here about 5e-4) brings it back."""
    n, k, t = 70, 64, 40
    hw, w = _weight(ctx, kind, n, k)
    x = O.Rng(2).vec_normal(t * k, 1e37).reshape(t, k)
    x[3, 5] = 3.4e38
    x[4] = np.where(w[0] < 0, -2e36, 2e36)  # no product with a code overflows, their sum does
    dy = O.Rng(3).vec_normal(t * n, 1e37).reshape(t, n)
    dx = np.zeros(t * k, np.float32)
    hw.backward_input(dy, t, dx)
    for got, a, b in ((hw.forward(x, t), x.astype(np.float64), w.T), (dx, dy.astype(np.float64), w)):
        want, size = a @ b, np.abs(a) @ np.abs(b)
        assert np.abs(want).max() < 1e38
        assert (np.abs(got.reshape(want.shape).astype(np.float64) - want) <= (b.shape[0] / 16 + 4) * 2.0 ** -24 * size).all()
