"""The run-time Fourier pass (extents without a compile-time kernel) against
the oracle: planes, columns and single axes at the edges of what a tile
holds, odd and mixed-radix extents, the smallest and the longest axes.

Tolerance: 1e-13 of the largest value, as for the compile-time passes (a
transform of N points rounds at a few log2 N units of 1.1e-16, and p^2 and
the inverse add a few more).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")


@pytest.mark.parametrize("dims", [(2, 3, 5, 7), (3, 2, 2, 2), (20, 28, 10, 36), (9, 15, 21, 5), (12, 12, 12, 24),
                                  (28, 28, 4, 6), (2, 2, 2, 98), (64, 64, 2, 2), (50, 96, 3, 2), (72, 96, 2, 2),
                                  (2, 2, 70, 70), (2, 3, 96, 90), (2048, 2, 2, 3), (2, 2, 2, 2000), (7, 49, 5, 25),
                                  (18, 14, 30, 40)])
def test_landau_transform(dims):
    print(f"[fft_any] {dims}", flush=True)
    rng = np.random.default_rng(8)
    V = int(np.prod(dims))
    F = rng.standard_normal((4, V)) + 1j * rng.standard_normal((4, V))
    ref = O.Lattice(dims, nth=2).fourier_accelerate(F)
    with gl.Gfix(dims, gl.LANDAU) as g:
        out = g.stage_fa(F)
    assert np.abs(out - ref).max() < 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("dims", [(3, 5, 7, 2), (15, 14, 10, 4), (20, 20, 20, 3), (2, 98, 3, 2), (72, 96, 3, 2),
                                  (2, 3, 2000, 2), (28, 10, 36, 5)])
def test_slice_transform(dims):
    print(f"[fft_any] slices of {dims}", flush=True)
    rng = np.random.default_rng(9)
    V = int(np.prod(dims))
    F = rng.standard_normal((4, V)) + 1j * rng.standard_normal((4, V))
    L = O.Lattice(dims, nth=2)
    n = V // dims[3]
    psq = L.psq(3)
    ref = np.empty_like(F)
    for t in range(dims[3]):
        part = np.ascontiguousarray(F[:, t * n:(t + 1) * n])
        ref[:, t * n:(t + 1) * n] = O.fft(O.fft(part, dims, 3, -1) * psq, dims, 3, +1)
    with gl.Gfix(dims, gl.COULOMB) as g:
        out = g.stage_fa(F)
    assert np.abs(out - ref).max() < 1e-13 * np.abs(ref).max()
