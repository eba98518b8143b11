"""dx = dy . W where the tiles do not fill whole rounds of the chip: the first rounds' tiles are summed by
one workgroup each, the rest split over several and added by the finish.  Ragged tokens, columns and rows
on the 64- and the 256-token kernel (RTQ_DX_WIDE), plain, accumulating and with an adapter.  Every row
within 2e-6 of its largest float64 value (three split f16 products per element leave about 2^-21 each;
the same bound as the other dx tests)."""
import os

import numpy as np
import pytest

import oracle as O
import rust_trainer_amd as rt

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["0", "1"], ids=["tok64", "tok256"])
def ctx(request):
    old = os.environ.get("RTQ_DX_WIDE")
    os.environ["RTQ_DX_WIDE"] = request.param
    try:
        c = rt.Context(0)
    finally:
        if old is None:
            del os.environ["RTQ_DX_WIDE"]
        else:
            os.environ["RTQ_DX_WIDE"] = old
    yield c
    c.close()


# (format, rows, columns, tokens): 64-token tiles of 64 columns chunks: 512 whole + 64 / 128 split;
# 256-token tiles: 256 whole + 64 split, and 64 tiles all split; a weight of one 32-row step pair
@pytest.mark.parametrize("wtype,n,k,t", [(O.Q4_0, 500, 8160, 1100), (O.Q6_K, 448, 8192, 570), (O.Q8_0, 64, 8192, 1030),
                                         (O.Q4_K, 1030, 8192, 250)])
def test_dx_split_tiles(ctx, wtype, n, k, t):
    w = O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k)
    blocks = O.quantize(wtype, w)
    dense = O.dequantize(wtype, blocks, k).reshape(n, k).astype(np.float64)
    dy = O.Rng(3).vec_normal(t * n, 1.0).reshape(t, n)
    hw = rt.HipFrozen(wtype, blocks, n, k, ctx=ctx)
    want = dy.astype(np.float64) @ dense
    scale = np.abs(want).max(axis=1, keepdims=True)
    dx0 = O.Rng(4).vec_normal(t * k, 1.0).reshape(t, k)
    dx = dx0.reshape(-1).copy()
    hw.backward_input(dy, t, dx)
    # the sum with dx0 is rounded once more (2^-24 of a value up to about 5 + scale)
    assert (np.abs(dx.reshape(t, k) - (want + dx0)) <= 2e-6 * scale + 2.0 ** -24 * (np.abs(dx0) + np.abs(want))).all()
    a = O.Rng(5).vec_normal(8 * k, 0.05).reshape(8, k)
    b = O.Rng(6).vec_normal(n * 8, 0.05).reshape(n, 8)
    lin = rt.Linear("dx", hw)
    lin.lora = rt.Lora(8, 16.0, a, b)
    x = O.Rng(7).vec_normal(t * k, 1.0).reshape(t, k)
    got = lin.backward(x, dy, t).reshape(t, k)
    full = want + 2 * (dy.astype(np.float64) @ b) @ a.astype(np.float64)
    assert (np.abs(got - full) / np.abs(full).max(axis=1, keepdims=True)).max() <= 2e-6


@pytest.fixture(scope="module", params=["0", "1"], ids=["tok64", "tok256"])
def whole(request):
    knobs = {"RTQ_DX_WIDE": request.param, "RTQ_DX_SPLITS": "1"}
    old = {k: os.environ.get(k) for k in knobs}
    os.environ.update(knobs)
    try:
        c = rt.Context(0)
    finally:
        for k, v in old.items():
            os.environ.pop(k) if v is None else os.environ.update({k: v})
    yield c
    c.close()


@pytest.mark.parametrize("wtype", [O.Q4_0, O.Q8_0, O.Q4_K, O.Q6_K])
@pytest.mark.parametrize("n,t", [(1500, 70), (1027, 300)])
def test_dx_of_rows_of_wide_range(whole, wtype, n, t):
    """Rows of dy with slices of 256 far below their largest, all summed by one workgroup: where the weight is
    zero against the large values, the small ones' products are the result, to the same 2e-6.  Large values in the
    first rows, the last, in between, next to zeros, everything tiny, and small slices alone.  (A range is shared by
    256 rows, or 480 on 256-token tiles: those of the large values hold nothing else here.)"""
    k = 512
    w = O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k)
    big = np.array([5, 600, n - 1])
    w[big, :64] = 0.0
    blocks = O.quantize(wtype, w)
    dense = O.dequantize(wtype, blocks, k).reshape(n, k).astype(np.float64)
    assert (dense[big, :64] == 0).all()
    dy = O.Rng(3).vec_normal(t * n, 1.0).reshape(t, n)
    first, middle, last = slice(0, 480), slice(480, 960), slice(960, n)
    dy[0::6, first] = 0.0
    dy[0::6, big[0]] = 2.0 ** 45
    dy[1::6, last] = 0.0
    dy[1::6, big[2]] = -2.0 ** 50
    dy[2::6, :960] = 0.0
    dy[2::6, big[1]] = 2.0 ** 30
    dy[3::6, first] = dy[3::6, last] = 0.0
    dy[3::6, big[0]], dy[3::6, big[2]] = 2.0 ** 40, -2.0 ** 20
    dy[4::6] *= 2.0 ** -100
    dy[4::6, middle] = 0.0
    dy[4::6, big[1]] = 2.0 ** -60
    dy[5::6, middle] *= 2.0 ** -30
    dx = np.zeros(t * k, np.float32)
    rt.HipFrozen(wtype, blocks, n, k, ctx=whole).backward_input(dy, t, dx)
    want = dy.astype(np.float64) @ dense
    for cols in (slice(0, 64), slice(64, k)):
        err = np.abs(dx.reshape(t, k) - want)[:, cols] / np.abs(want[:, cols]).max(axis=1, keepdims=True)
        assert err.max() <= 2e-6, (cols, np.unravel_index(err.argmax(), err.shape), err.max())


@pytest.fixture(scope="module", params=["0", "1"], ids=["default", "tok32"])
def any_dx(request):
    old = os.environ.get("RTQ_DX_32")
    os.environ["RTQ_DX_32"] = request.param
    try:
        c = rt.Context(0)
    finally:
        os.environ.pop("RTQ_DX_32") if old is None else os.environ.update(RTQ_DX_32=old)
    yield c
    c.close()


@pytest.mark.parametrize("wtype,n,k,t", [(O.Q6_K, 426, 256, 22), (O.Q4_0, 70, 96, 17), (O.Q8_0, 300, 544, 70)])
def test_dx_of_small_weights(any_dx, wtype, n, k, t):
    """Weights of a few 32-row steps, split down to one step a workgroup by the default plan."""
    blocks = O.quantize(wtype, O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k))
    dy = O.Rng(3).vec_normal(t * n, 1.0).reshape(t, n)
    dx = np.zeros(t * k, np.float32)
    rt.HipFrozen(wtype, blocks, n, k, ctx=any_dx).backward_input(dy, t, dx)
    want = dy.astype(np.float64) @ O.dequantize(wtype, blocks, k).reshape(n, k).astype(np.float64)
    assert (np.abs(dx.reshape(t, k) - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True)).all()


@pytest.mark.parametrize("t", [1, 8, 40])
def test_dx_of_tiny_rows(any_dx, t):
    """Rows whose largest value is below 2^-113, where 2^15 over it is no finite float."""
    n, k = 600, 256
    blocks = O.quantize(O.Q8_0, O.Rng(1).vec_normal(n * k, 0.02).reshape(n, k))
    dy = O.Rng(3).vec_normal(t * n, 2.0 ** -118).reshape(t, n)
    dx = np.zeros(t * k, np.float32)
    rt.HipFrozen(O.Q8_0, blocks, n, k, ctx=any_dx).backward_input(dy, t, dx)
    want = dy.astype(np.float64) @ O.dequantize(O.Q8_0, blocks, k).reshape(n, k).astype(np.float64)
    # 2e-6 of the largest, and what 2^-126 at the range's bottom leaves: results near 2^-121 keep 2^-149 steps
    assert (np.abs(dx.reshape(t, k) - want) <= 2e-6 * np.abs(want).max(axis=1, keepdims=True) + n * 2.0 ** -149).all()
