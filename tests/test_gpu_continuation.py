"""Continuation segments inside the FP32 phase of a mixed run.  Safeguard 1
(GLU_GFIX_SAFEGUARD bit 0) restarts CG after a line search that found its
direction uphill; a continuation begins with a steepest-descent step, which
is a restart already, so its first CG iteration takes its usual beta
whatever the segment before ended on.  With segments of one iteration the
safeguard never acts, and the run is bitwise the one without it.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")


def _trace(dims, seed, mode, monkeypatch):
    monkeypatch.setenv("GLU_GFIX_SAFEGUARD", mode)
    with gl.Gfix(dims, gl.LANDAU, gl.MIXED) as g:
        g.heatbath(6.0, 4, 1, seed=seed)
        g.random_transform(seed=seed + 1)
        g.set_switch_theta(2e-2)
        g.run(gl.CG, 0.08, 1e-2, 1)  # every segment: an SD start, one CG iteration
        return g.trace()


@pytest.mark.parametrize("dims,seed", [((4, 4, 4, 4), 0), ((4, 4, 4, 4), 2), ((8, 8, 8, 8), 4), ((8, 8, 8, 8), 5)])
def test_sd_start_forgets_an_uphill_direction(dims, seed, monkeypatch):
    print(f"[continuation] {dims} {seed}", flush=True)
    off, on = (_trace(dims, seed, mode, monkeypatch) for mode in ("0", "1"))
    # an uphill direction: the parabola's vertex below half the first probe
    assert np.any(off[1:-2:2, 1] < 0.075)
    assert np.array_equal(off, on)
