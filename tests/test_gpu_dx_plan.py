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
