"""The closed-form helicity gradients of the f64 adjoint (tp_helicity.h, built
for the host) against the spinor amplitudes on dual numbers over long double,
and the spinor of a photon along -Z."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

HERE = os.path.dirname(os.path.abspath(__file__))
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def helgrad(tmp_path_factory):
    out = tmp_path_factory.mktemp("helgrad") / "libhelgrad.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I" + os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "helgrad_check.cpp"), "-o", str(out)], check=True)
    lib = C.CDLL(str(out))

    def call(name, e, g, p):
        p = np.ascontiguousarray(p, np.float64)
        m, d = np.zeros((len(p), 5)), np.zeros((len(p), 5, 3, 4))
        fn = getattr(lib, name)
        fn.argtypes = [C.c_double] * 4 + [C.c_long] + [C.c_void_p] * 3
        fn(e, *g, len(p), p.ctypes.data, m.ctypes.data, d.ctypes.data)
        return m, d
    return call


def run_constants(valeurs):
    import trois_photons as tp
    P = tp.params_from_config(tp.Configuration.load(valeurs))
    return P.e_total, (P.g_a, P.g_beta_p, P.g_beta_m)


@pytest.mark.parametrize("order", [(0, 1, 2), (2, 0, 1), (1, 2, 0), (2, 1, 0)])
def test_gradients_match_dual_numbers(helgrad, oracle, valeurs, order):
    """Some 60 roundings lie between the momenta and a derivative, each of them
    amplified by at most the condition 2 E / (E + Z) of a photon's spinor and that
    of the products of a near-collinear pair, 1 / (1 - cos)."""
    e, g = run_constants(valeurs)
    u = np.random.default_rng(12).random((6000, 12))
    p, keep, _, _, _ = oracle.events(oracle.config(valeurs), oracle.opts("xoshiro"), u)
    p = np.ascontiguousarray(p[keep.astype(bool)][:, 2:, :][:, list(order)])
    m, d = helgrad("tp_helgrad_closed", e, g, p)
    rm, rd = helgrad("tp_helgrad_spinors", e, g, p)
    # the interference on the scale of its amplitudes, a derivative on the scale of its photon's largest
    both = 2 * np.sqrt(rm[:, :1] * rm[:, 1:2])
    scale = np.concatenate([rm[:, :3], both, both], 1)
    size = np.abs(rd).max(axis=3, keepdims=True) + (scale[:, :, None] / p[:, None, :, 3])[..., None]
    cond = (2 * p[:, :, 3] / (p[:, :, 3] + p[:, :, 2])).max(axis=1)
    n = p[:, :, :3] / p[:, :, 3:]
    angle = np.min([1 - (n[:, i] * n[:, j]).sum(1) for i, j in ((0, 1), (0, 2), (1, 2))], axis=0)
    bound = 64 * EPS * cond / np.minimum(angle, 1)
    em, ed = (np.abs(m - rm) / scale).max(axis=1), (np.abs(d - rd) / size).max(axis=(1, 2, 3))
    print(f"{len(p)} events: sums within {np.max(em / bound):.3f}, derivatives within {np.max(ed / bound):.3f} of the bound; "
          f"derivatives' median {np.median(ed) / EPS:.1f} eps, p99 {np.percentile(ed, 99) / EPS:.0f} eps")
    assert np.all(em <= bound) and np.all(ed <= bound)


def test_photon_along_minus_z(helgrad, valeurs):
    """E + Z = 0: the spinor (0, sqrt(2E)) depends on E alone (spinor.rs:40-44); E + Z < 0 gives NaN."""
    e, g = run_constants(valeurs)
    h = e / 2
    p = np.array([[[0.5 * h, 0.3 * h, 0.4 * h, 0.], [-0.5 * h, -0.3 * h, 0.3 * h, 0.], [0., 0., -0.7 * h, 0.7 * h]]] * 3)
    p[:, :2, 3] = np.linalg.norm(p[:, :2, :3], axis=2)
    p = p[np.arange(3)[:, None], [[0, 1, 2], [2, 0, 1], [1, 2, 0]]]
    m, d = helgrad("tp_helgrad_closed", e, g, p)
    rm, rd = helgrad("tp_helgrad_spinors", e, g, p)
    assert np.all(np.abs(m - rm) <= 64 * EPS * np.abs(rm).max(axis=1, keepdims=True))
    along = p[:, :, 3] + p[:, :, 2] == 0
    assert np.all(d[np.broadcast_to(along[:, None], d.shape[:3])][:, :3] == 0)
    # the limit ez -> 0 is taken at ez = E 2^-120, a relative 2^-60 off
    assert np.all(np.abs(d - rd) <= 64 * EPS * np.abs(rd).max(axis=(2, 3), keepdims=True))
    p[0, 2, 2] *= 1.01
    m, d = helgrad("tp_helgrad_closed", e, g, p)
    assert np.all(np.isnan(m[0])) and np.all(np.isnan(d[0, :, 2, 3])) and np.all(d[0, :, 2, :3] == 0)
