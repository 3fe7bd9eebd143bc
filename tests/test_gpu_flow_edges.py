"""The proposal's kernels at the edges of their launches: samples around a
workgroup's, either side of the size where the forward and inverse kernels take
other tiles, and batches of few and of partly filled chunks in the gradients."""
import numpy as np
import pytest

import flow_ref as F
import trois_photons as tp
from test_gpu_flow import base_points

pytestmark = pytest.mark.gpu

BIG = 1 << 20


@pytest.fixture(scope="module")
def rflow():
    print("creating engine on cuda:0", flush=True)
    with tp.Engine(0) as e:
        f = tp.Flow(e)
        w = F.random_params(1)
        f.set_params(w)
        yield f, w
        f.close()


@pytest.mark.parametrize("n", [1, 15, 17, 255, 257, 383, 385, 70_001])
def test_a_sample_does_not_depend_on_the_batch(rflow, n):
    """Sample i of n is sample i of more than 2^20, bit for bit, forward and inverse."""
    f, _ = rflow
    print(f"flow sample and density n={n}", flush=True)
    u, z, lq = f.sample(n, key=5)
    U, Z, LQ = f.sample(BIG + 5, key=5)
    assert np.array_equal(u, U[:n]) and np.array_equal(z, Z[:n]) and np.array_equal(lq, LQ[:n])
    assert np.array_equal(f.density(u), f.density(U)[:n])


@pytest.mark.parametrize("n", [16, 32, 48, 64, 80, 240, 256, 272, 528, 4112])
def test_gradients_of_small_batches(rflow, n):
    """Activations and deltas are rounded to bf16 (2^-9 relative): the sums differ by that much of each term at most,
    times the few products a delta passes through."""
    f, w = rflow
    rng = np.random.default_rng(n)
    v = base_points(n, n)
    gz = np.zeros((n, 16), np.float32)
    gz[:, :12] = rng.normal(0, 1, (n, 12))
    print(f"flow backward n={n}", flush=True)
    g, gv = f.grad(v, gz)
    gr, gvr = F.grad(v, gz, w, emulate=True)
    for l in range(F.L):
        sl = slice(l * F.LP, (l + 1) * F.LP)
        assert np.linalg.norm(g[sl] - gr[sl]) <= 12 * 2**-9 * np.linalg.norm(gr[sl]), l
    assert np.median(np.abs(gv[:, :12] - gvr) / (np.abs(gvr).max(1, keepdims=True) + 1e-6)) < 1e-2
