"""The kernels of small lattices (up to 65536 sites: four wavefronts per 64
sites, beta and the step taken from the partial sums by the kernels that use
them) against the oracle: sizes at which the last 64 or 256 sites are not
whole, the largest lattice that takes them and the next one, which does not;
FP32 with probe tiles that divide the lattice and without.

Tolerances.  FP64: 1e-11 on the links after 6 iterations (rounding of 1e-15
a stage, which the parabola fit amplifies less than 10-fold over the first
iterations).  Mixed: the first 6 iterations run in FP32, where a link is off
by about 20 roundings of 6e-8; theta is a mean of squares of differences of
links of order one, so its relative error stays below 1e-5 in one iteration
and, amplified 10-fold, below 1e-4.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (3, 3, 3, 3), (4, 4, 4, 4), (5, 3, 7, 6), (8, 4, 4, 6), (9, 7, 5, 14),
                                  (16, 16, 16, 16), (16, 16, 16, 18)])
def test_small_lattice(dims):
    print(f"[small lattice] {dims}", flush=True)
    L = O.Lattice(dims, nth=4)
    U = L.heatbath(6.0, 4, 1, seed=11)
    L.random_gtrans(U, seed=7, nth=4)
    W = U.copy()
    r = L.facg(W, max_iters=6, trace=16)
    for precision in (gl.FP64, gl.MIXED):
        with gl.Gfix(dims, precision=precision) as g:
            g.set_links(U)
            it, _ = g.run(gl.CG, 0.08, 1e-14, 6)
            th = g.trace()[:7, 0]
            assert it == r["iters"]
            assert np.all(np.abs(th / r["trace_theta"][:7] - 1) < (1e-11 if precision == gl.FP64 else 1e-4))
            if precision == gl.FP64:
                assert np.abs(g.get_links() - W).max() < 1e-11
