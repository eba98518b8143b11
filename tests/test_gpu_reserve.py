"""Context.reserve: no call up to the reserved tokens, rows, columns and rank grows the workspace (which would
synchronise the device, and fail inside a caller's graph capture).  The dx plans are not monotonic: a narrower
weight or fewer tokens can need more partials than the widest call (the first case by 1.35 times, which had been
more than the reserve's quarter to spare)."""
import random

import numpy as np
import pytest
import torch

import rust_trainer_amd as rt

pytestmark = pytest.mark.gpu

TYPES = {rt.TYPE_Q4_0: (32, 18, (0,)), rt.TYPE_Q8_0: (32, 34, (0,)), rt.TYPE_Q4_K: (256, 144, (0, 2)), rt.TYPE_TQ8_0: (32, 36, ())}


def _weight(ctx, wtype, n, k):
    elems, size, scales = TYPES[wtype]
    b = np.zeros((n * k // elems, size), np.uint8)
    for o in scales:
        b[:, o:o + 2] = np.array([0.01], np.float16).view(np.uint8)
    return rt.HipFrozen(wtype, b.reshape(-1), n, k, ctx=ctx)


def _random_calls(seed, t, n, k):
    r = random.Random(seed)
    out = []
    for wtype in TYPES:
        unit = TYPES[wtype][0]
        for _ in range(4):
            cols = max(unit, unit * r.randint(1, k // unit))
            out.append((wtype, r.randint(max(1, n // 4), n), cols, [r.randint(1, t), r.randint(1, min(t, 16)), t]))
    return out


@pytest.mark.parametrize("t,n,k,calls", [
    (2048, 14336, 14336, [(rt.TYPE_Q8_0, 14336, 11520, [2048])]),
    (1055, 79699, 1024, [(rt.TYPE_Q8_0, 79699, 768, [1040])]),
    (700, 3000, 2560, _random_calls(1, 700, 3000, 2560)),
    (96, 20000, 1024, _random_calls(2, 96, 20000, 1024)),
    (16, 5000, 4096, _random_calls(3, 16, 5000, 4096)),
], ids=["wide", "tall", "mixed", "head", "short"])
def test_reserved_workspace_does_not_grow(t, n, k, calls):
    rank = 16
    c = rt.Context(0)
    try:
        weights = [(_weight(c, w, rows, cols), rows, cols, ts) for w, rows, cols, ts in calls]
        dy, x = torch.zeros(t * n, device="cuda"), torch.zeros(t * k, device="cuda")
        y, dx = torch.zeros(t * n, device="cuda"), torch.zeros(t * k, device="cuda")
        a, b = torch.zeros(rank * k, device="cuda"), torch.zeros(n * rank, device="cuda")
        ga, gb = torch.zeros(rank * k, device="cuda"), torch.zeros(n * rank, device="cuda")
        lib = rt._ffi.lib()
        c.reserve(t, n, k, rank)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        lora = rt._ffi.RtqLora(rank, 2.0 * rank, a.data_ptr(), b.data_ptr(), 1)
        for w, rows, cols, ts in weights:
            for tokens in ts:
                for ad in (None, rt._ffi.ctypes.byref(lora)):
                    rt._ffi.check(lib.rtq_linear_forward_d(c.handle, w.handle, None, ad, x.data_ptr(), tokens, y.data_ptr(), None), "fwd")
                    rt._ffi.check(lib.rtq_linear_backward_d(c.handle, w.handle, ad, x.data_ptr(), dy.data_ptr(), tokens, dx.data_ptr(),
                                                            ga.data_ptr() if ad else None, gb.data_ptr() if ad else None, None), "bwd")
                torch.cuda.synchronize()
                assert torch.cuda.mem_get_info()[0] >= free, (rows, cols, tokens)
    finally:
        c.close()
