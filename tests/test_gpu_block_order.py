"""The order of the workgroups that a context starts with, time slabs or, on
long lattices (T at least 8 Lz), contiguous runs: no sum depends on it, so a
run is bitwise the one of a context told its order.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")


@pytest.mark.parametrize("dims", [(16, 16, 8, 64), (16, 16, 8, 56), (32, 8, 3, 128)])
@pytest.mark.parametrize("precision", [gl.FP64, gl.MIXED])
def test_default_order_is_neutral(dims, precision, monkeypatch):
    print(f"[block order] {dims} {precision}", flush=True)
    out = []
    for order in (None, "0", "1", "2"):
        if order is not None:
            monkeypatch.setenv("GLU_GFIX_XCD", order)
        with gl.Gfix(dims, precision=precision) as g:
            g.heatbath(6.0, 4, 1, seed=3)
            g.random_transform(seed=4)
            g.run(gl.CG, 0.08, 1e-14, 12)
            out.append((g.trace(), g.get_links()))
    for trace, links in out[1:]:
        assert np.array_equal(trace, out[0][0])
        assert np.array_equal(links, out[0][1])
