"""Every extent of the shared-launch transforms (2..16, primes and composites,
on the staged axes and on t) against the oracle: a few iterations of a small
lattice, where the Fourier acceleration enters every one.

Tolerance: 1e-11 on the links after 6 iterations.  The transform rounds at
1e-15 and the parabola fit amplifies it less than 10-fold over the first
iterations (1e3 over 20, see test_gpu_facg_batch.py).
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dims", [(10, 11, 3, 13), (14, 15, 9, 2), (13, 2, 14, 11), (3, 13, 10, 15), (6, 9, 12, 14),
                                  (16, 3, 5, 7), (11, 14, 15, 10)])
def test_transform_extents(dims):
    print(f"[batch extents] {dims}", flush=True)
    L = O.Lattice(dims, nth=4)
    U = L.heatbath(6.0, 4, 1, seed=11)
    L.random_gtrans(U, seed=7, nth=4)
    W = U.copy()
    r = L.facg(W, max_iters=6)
    dev = torch.from_numpy(U.reshape(1, -1, 4, 18)).cuda()
    torch.cuda.synchronize()
    its, _ = gl.facg_batch(dims, dev.data_ptr(), 1, 0.08, 1e-14, 6)
    assert its[0] == r["iters"] == 123456789
    assert np.abs(dev.cpu().numpy()[0] - W).max() < 1e-11
