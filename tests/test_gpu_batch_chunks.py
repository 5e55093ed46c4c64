"""The batched solver's update walks a lattice in chunks of one site per thread
of its workgroup: lattices smaller than a chunk, of exactly one or several
chunks, with a time slice of exactly one chunk, with a last chunk of a few
sites, and extents of 2, whose two neighbours along an axis are one site --
against the oracle.

Tolerance: 1e-11 on the links after 6 iterations, as rounding at 1e-15 a
stage is amplified less than 10-fold over the first iterations.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (8, 8, 4, 2), (8, 8, 8, 2), (16, 16, 2, 3), (3, 3, 3, 10), (5, 4, 13, 2),
                                  (2, 16, 16, 5), (16, 16, 9, 2)])
@pytest.mark.parametrize("wg", ["512", "128"])
def test_chunks(dims, wg, monkeypatch):
    print(f"[batch chunks] {dims} {wg}", flush=True)
    monkeypatch.setenv("GLU_GFIX_BATCH_WG", wg)
    L = O.Lattice(dims, nth=4)
    U = L.heatbath(6.0, 4, 1, seed=5)
    L.random_gtrans(U, seed=3, nth=4)
    W = U.copy()
    r = L.facg(W, max_iters=6)
    dev = torch.from_numpy(np.stack([U, U]).reshape(2, -1, 4, 18)).cuda()
    torch.cuda.synchronize()
    its, _ = gl.facg_batch(dims, dev.data_ptr(), 2, 0.08, 1e-14, 6)
    assert its[0] == its[1] == r["iters"]
    out = dev.cpu().numpy()
    assert np.abs(out[0] - W).max() < 1e-11
    assert np.array_equal(out[0], out[1])
