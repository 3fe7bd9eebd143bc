"""tp_adjoint at the edges of its launches: point counts around a workgroup's
and around the run lengths of the stream's expansion, outputs aligned to one
double only, absent outputs, and photons kept in the order they were drawn."""
import ctypes

import numpy as np
import pytest

import trois_photons as tp
from oracle_ffi import OracleGrad

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    print("creating engine on cuda:0", flush=True)
    with tp.Engine(0) as e:
        yield e


@pytest.mark.parametrize("precision", [tp.PREC_F64, tp.PREC_F32])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 4097, 131071, 131073, 262145])
def test_stream_points_equal_given_points(engine, oracle, valeurs, n, precision):
    """The stream's uniforms are exact, so the outputs are those of the same points given, bit for bit."""
    print(f"adjoint n={n} precision={precision}", flush=True)
    params = tp.params_from_config(tp.Configuration.load(valeurs))
    st = tp.rng_state(tp.RNG_XOSHIRO, 77)
    u = oracle.uniforms(oracle.rng("xoshiro", 77), 12 * n).reshape(n, 12)
    a = engine.adjoint(params, n, precision, st=st)
    b = engine.adjoint(params, n, precision, u=u)
    for x, y in zip(a, b):
        assert np.array_equal(x, y, equal_nan=True)


@pytest.mark.parametrize("sort,cut_plane", [(True, 0.0), (False, 0.0), (True, 0.3), (False, 0.3)])
def test_order_and_plane_cut(engine, oracle, valeurs, sort, cut_plane):
    """Against the oracle's gradient, with the bounds of the shipped configuration's test."""
    cfg = tp.Configuration.load(valeurs)
    params = tp.params_from_config(cfg)
    params.sort_photons, params.cut_plane = int(sort), cut_plane
    ocfg = oracle.config(valeurs)
    ocfg.cut_plane = cut_plane
    u = oracle.uniforms(oracle.rng("xoshiro", 5), 12 * 3001).reshape(-1, 12)
    F, gu, gp = engine.adjoint(params, len(u), tp.PREC_F64, u=u)
    oF, ogu, ogp = OracleGrad(oracle, ocfg, sort=sort).grad(u)
    keep = np.any(oF != 0, axis=1)
    assert np.array_equal(keep, np.any(F != 0, axis=1)) and 0 < keep.sum() < len(u)
    assert np.all(gu[~keep] == 0) and np.all(gp[~keep] == 0)
    for x, y in ((F[:, None], oF[:, None]), (gu, ogu), (gp, ogp)):
        r = np.abs(x[keep] - y[keep]) / np.abs(y[keep]).max(axis=-1, keepdims=True)
        assert np.percentile(r, 99) < 1e-10 and r.max() < 1e-6


@pytest.mark.parametrize("n", [64, 100])
@pytest.mark.parametrize("missing", [None, 0, 1, 2])
def test_unaligned_and_absent_outputs(engine, valeurs, n, missing):
    import torch
    params = tp.params_from_config(tp.Configuration.load(valeurs))
    st = tp.rng_state(tp.RNG_XOSHIRO, 3)
    ref = engine.adjoint(params, n, tp.PREC_F64, st=st)
    sizes = (5 * n, 60 * n, 60 * n)
    buf = [torch.full((s + 3,), 7.0, dtype=torch.float64, device="cuda:0") for s in sizes]
    ptr = [ctypes.c_void_p(0 if k == missing else b.data_ptr() + 8) for k, b in enumerate(buf)]
    torch.cuda.synchronize()
    engine._check(tp.lib.tp_adjoint(engine.h, ctypes.byref(params), tp.RNG_XOSHIRO, ctypes.byref(st), None, n,
                                    tp.PREC_F64, 1, *ptr), "tp_adjoint")
    for k, (b, s) in enumerate(zip(buf, sizes)):
        b = b.cpu().numpy()
        assert np.all(b[:1] == 7) and np.all(b[s + 1:] == 7)
        assert np.all(b == 7) if k == missing else np.array_equal(b[1:s + 1], ref[k].ravel())
