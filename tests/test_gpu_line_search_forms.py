"""The two forms of the FP32 line search on lattices its tiles divide: tiles,
and one site per thread, which the autotuner times beside them (in 32^3x64's
time slabs it is the faster one) and GLU_GFIX_LS_TILE=0 asks for.

Tolerance against the oracle: 1e-4 relative on theta over 6 FP32 iterations,
as in test_gpu_small_lattice.py (a link is off by about 20 roundings of 6e-8,
theta by 1e-5 in one iteration, amplified less than 10-fold).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")


@pytest.mark.parametrize("dims", [(8, 8, 8, 8), (16, 16, 16, 18)])
def test_both_forms_follow_the_oracle(dims, monkeypatch):
    print(f"[line search forms] {dims}", flush=True)
    L = O.Lattice(dims, nth=4)
    U = L.heatbath(6.0, 4, 1, seed=11)
    L.random_gtrans(U, seed=7, nth=4)
    W = U.copy()
    r = L.facg(W, max_iters=6, trace=16)
    rows = []
    for tile in ("1", "0"):
        monkeypatch.setenv("GLU_GFIX_LS_TILE", tile)
        with gl.Gfix(dims, precision=gl.MIXED) as g:
            g.set_links(U)
            it, _ = g.run(gl.CG, 0.08, 1e-14, 6)
            assert it == r["iters"]
            rows.append(g.trace()[:7])
        assert np.all(np.abs(rows[-1][:, 0] / r["trace_theta"][:7] - 1) < 1e-4)
    # another order of the probes' sums, so other last bits of the steps
    assert not np.array_equal(rows[0], rows[1])


def test_autotuner_times_both_forms():
    dims = (16, 16, 16, 36)
    print(f"[line search forms] tuner {dims}", flush=True)
    with gl.Gfix(dims, precision=gl.MIXED) as g:
        g.heatbath(6.0, 4, 1, seed=3)
        g.random_transform(seed=4)
        rep = g.autotune()
        assert "on tiles" in rep and "one site per thread" in rep, rep
        it, th = g.run(gl.CG, 0.08, 1e-14, 1000)
        assert th < 1e-14 and it < 1000


@pytest.mark.parametrize("dims,precision", [((8, 8, 8, 8), gl.FP64), ((8, 8, 8, 8), gl.MIXED), ((6, 6, 6, 10), gl.MIXED)])
def test_autotuner_times_what_a_small_lattice_runs(dims, precision):
    """Small lattices (up to 65536 sites) run stencil kernels of their own,
    without an order of the workgroups: the tuner times none."""
    print(f"[line search forms] small tuner {dims} {precision}", flush=True)
    with gl.Gfix(dims, precision=precision) as g:
        g.heatbath(6.0, 4, 1, seed=3)
        g.random_transform(seed=4)
        rep = g.autotune()
        assert "order plain" not in rep and "stencil order: none" in rep, rep
        assert ("site order" in rep) == (precision == gl.MIXED and dims[0] % 8 == 0), rep
        it, th = g.run(gl.CG, 0.08, 1e-14, 1000)
        assert th < 1e-14 and it < 1000
