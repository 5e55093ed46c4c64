"""Extents that have compile-time Fourier passes, in pairs that have no
compile-time pass over both axes: up to a volume they take the run-time pass
over a plane or a column, above it single axes.  Shapes on both sides of each
line against the oracle.

Tolerances as in test_gpu_fft_any.py (1e-13 of the largest value) and, for the
mixed solves, whose first 6 iterations run in FP32, test_gpu_large_ragged.py
(1e-4 on theta, 5e-4 on the links).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")


@pytest.mark.parametrize("dims", [(8, 8, 64, 64), (16, 16, 16, 96), (32, 32, 24, 24), (48, 96, 8, 8), (48, 96, 24, 24),
                                  (64, 64, 16, 8)])
def test_landau_transform(dims):
    print(f"[fft routes] {dims}", flush=True)
    rng = np.random.default_rng(8)
    V = int(np.prod(dims))
    F = rng.standard_normal((4, V)) + 1j * rng.standard_normal((4, V))
    ref = O.Lattice(dims, nth=8).fourier_accelerate(F)
    with gl.Gfix(dims, gl.LANDAU) as g:
        out = g.stage_fa(F)
    assert np.abs(out - ref).max() < 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("dims", [(8, 8, 16, 64), (8, 8, 64, 32), (16, 16, 16, 64), (16, 16, 24, 24), (32, 32, 24, 24),
                                  (32, 64, 16, 16)])
def test_mixed_iterations(dims):
    print(f"[fft routes] mixed {dims}", flush=True)
    L = O.Lattice(dims, nth=8)
    U = L.heatbath(6.0, 2, 1, seed=11)
    L.random_gtrans(U, seed=7, nth=8)
    W = U.copy()
    r = L.facg(W, max_iters=6, trace=16)
    with gl.Gfix(dims, precision=gl.MIXED) as g:
        g.set_links(U)
        it, _ = g.run(gl.CG, 0.08, 1e-14, 6)
        assert it == r["iters"]
        assert np.all(np.abs(g.trace()[:7, 0] / r["trace_theta"][:7] - 1) < 1e-4)
        assert np.abs(g.get_links() - W).max() < 5e-4
