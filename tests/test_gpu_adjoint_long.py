"""tp_adjoint on more points of a stream than it expands at a time (2^24)."""
import ctypes

import numpy as np
import pytest

import trois_photons as tp

pytestmark = pytest.mark.gpu

STEP = 1 << 24


@pytest.mark.parametrize("precision", [tp.PREC_F64, tp.PREC_F32])
def test_long_streams(valeurs, precision):
    import torch
    n, width = 3 * STEP + 77, 1001
    dtype = torch.float32 if precision == tp.PREC_F32 else torch.float64
    params = tp.params_from_config(tp.Configuration.load(valeurs))
    out = [torch.full((n + 1, k), 7.0, dtype=dtype, device="cuda:0") for k in (5, 60)]
    st = tp.rng_state(tp.RNG_XOSHIRO, 77)
    with tp.Engine(0) as engine:
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info(0)[0]
        print(f"adjoint n={n} precision={precision}", flush=True)
        engine._check(tp.lib.tp_adjoint(engine.h, ctypes.byref(params), tp.RNG_XOSHIRO, ctypes.byref(st), None, n, precision, 1,
                                        ctypes.c_void_p(out[0].data_ptr()), ctypes.c_void_p(out[1].data_ptr()), None), "tp_adjoint")
        assert free - torch.cuda.mem_get_info(0)[0] < 96 * STEP + (64 << 20)
        for x in out:
            assert bool((x[n] == 7).all())
        # the points around the edges, each from the stream's state there
        for first in (0, STEP - 500, 2 * STEP - 1, 3 * STEP - 1000, n - width):
            at = type(st).from_buffer_copy(st)
            tp.rng_skip(tp.RNG_XOSHIRO, at, 12 * first)
            ref = engine.adjoint(params, width, precision, st=at)
            for x, r in zip(out, ref):
                assert np.array_equal(x[first:first + width].cpu().numpy(), r.reshape(width, -1), equal_nan=True), first
