"""Lattices above 65536 sites, which take the kernels of large ones, of extents
that the usual sizes do not have: a last block that is not whole, block counts
that the 8 XCDs do not divide, extents that the FP32 line search's tiles do not
divide, and x-y planes and z-t columns that need the larger LDS pools of the
run-time transforms, in both precisions -- against the oracle.

Tolerances.  FP64: 1e-11 on theta and the links after 6 iterations (rounding
of 1e-15 a stage, amplified less than 10-fold over the first iterations).
Mixed, whose first 6 iterations run in FP32: 1e-4 on theta, as in
test_gpu_small_lattice.py; on the links 5e-4: an accelerated field of size
10 off by 20 roundings of 6e-8 moves a transform by 0.3 * 1.2e-5 = 4e-6 a
step, 7 steps amplified 10-fold make 2.5e-4, and a link takes two transforms.
The probes are sums in another order than the oracle's: 1e-13 of their size,
or of the 4 sqrt(V) that traces of either sign add up to.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")


def _input(dims):
    L = O.Lattice(dims, nth=4)
    U = L.heatbath(6.0, 2, 1, seed=11)
    L.random_gtrans(U, seed=7, nth=4)
    return L, U


@pytest.mark.parametrize("dims", [(12, 10, 42, 40), (4, 4, 70, 60), (70, 60, 4, 5)])
def test_first_iterations(dims):
    print(f"[large ragged] {dims}", flush=True)
    L, U = _input(dims)
    W = U.copy()
    r = L.facg(W, max_iters=6, trace=16)
    for precision in (gl.FP64, gl.MIXED):
        with gl.Gfix(dims, precision=precision) as g:
            g.set_links(U)
            it, _ = g.run(gl.CG, 0.08, 1e-14, 6)
            th = np.abs(g.trace()[:7, 0] / r["trace_theta"][:7] - 1).max()
            off = np.abs(g.get_links() - W).max()
        print(f"[large ragged]   precision {precision}: theta {th:.1e} links {off:.1e}", flush=True)
        assert it == r["iters"]
        assert th < (1e-11 if precision == gl.FP64 else 1e-4)
        assert off < (1e-11 if precision == gl.FP64 else 5e-4)


@pytest.mark.parametrize("dims", [(12, 10, 42, 40), (16, 16, 16, 18)])
def test_line_search_stage(dims):
    print(f"[large ragged] line search {dims}", flush=True)
    L, U = _input(dims)
    _, F = L.fa_deriv(U)
    F = L.fourier_accelerate(F)
    red = np.zeros(3 + 8 * L.nth)
    W = U.copy()
    a_o = O.lib().or_line_search_landau(L.ref, O._dp(W), O._dp(F), O._dp(red))
    probes = np.array([sum(red[j + 8 * t] for t in range(L.nth)) for j in range(3)])
    with gl.Gfix(dims) as g:
        g.set_links(U)
        pr, a_g = g.stage_line_search(F)
    # the probe at 0 is a sum of 4 V traces of either sign
    assert np.all(np.abs(pr - probes) < 1e-13 * np.maximum(np.abs(probes), 4 * np.sqrt(L.V)))
    assert abs(a_g - a_o) < 1e-10 * abs(a_o)
