"""The plaquette of links rounded to single precision, as a configuration read
from a single-precision file has them: SU(3) to 1e-7 only, so every product
has to be formed in full.  Both measurements against the same sums in numpy
(complex128; the library holds a link's first two columns and completes the
third), and against each other.  Up to 512 rows of 256 sites the host adds the
partial sums (16^3x32 is the largest of these), above a second launch does.

Tolerance: 1e-13 relative.  A loop is some tens of roundings of 1.1e-16 and
sums over thousands of loops average them; a product completed from two of
its rows or columns is off by 1e-7 a loop, 1e-11 to 1e-9 in these averages.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

gl = pytest.importorskip("glu_amd")
torch = pytest.importorskip("torch")


def _noalloc(U, dims):
    links = torch.from_numpy(U).cuda()
    out = torch.zeros(6, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    rc = gl.lib().glu_gfix_measure_noalloc(C.c_void_p(links.data_ptr()), (C.c_size_t * 4)(*dims),
                                           C.c_void_p(out.data_ptr()), C.c_void_p(stream.cuda_stream))
    assert rc == 0, gl.lib().glu_gfix_last_error().decode()
    stream.synchronize()
    return out.cpu().numpy()


def _plaquette(U, dims):
    m = np.ascontiguousarray(U).view(np.complex128).reshape(dims[::-1] + (4, 3, 3))
    c0, c1 = m[..., 0], m[..., 1]
    m = np.stack([c0, c1, np.cross(c0, c1).conj()], -1)
    tot = 0.0
    for mu in range(1, 4):
        for nu in range(mu):
            a = m[..., mu, :, :] @ np.roll(m[..., nu, :, :], -1, 3 - mu)
            b = m[..., nu, :, :] @ np.roll(m[..., mu, :, :], -1, 3 - nu)
            tot += (a.real * b.real + a.imag * b.imag).sum()
    return 2 * tot / (36 * np.prod(dims))


@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (6, 6, 6, 10), (16, 16, 8, 8), (16, 16, 16, 32), (12, 10, 42, 40)])
def test_plaquette_of_single_precision_links(dims):
    print(f"[rounded links] {dims}", flush=True)
    with gl.Gfix(dims, gl.LANDAU, gl.FP64) as g:
        g.heatbath(6.0, 4, 1, seed=3)
        g.random_transform(seed=4)
        U = g.get_links().astype(np.float32).astype(np.float64)
        g.set_links(U)
        got = g.measure()
    ref, na = _plaquette(U, dims), _noalloc(U, dims)
    print(f"[rounded links]   {got['plaquette'] / ref - 1:.1e} {na[0] / ref - 1:.1e}", flush=True)
    assert abs(got["plaquette"] - ref) < 1e-13 * abs(ref)
    assert abs(na[0] - ref) < 1e-13 * abs(ref)
    for k, name in enumerate(("plaquette", "link_trace", "link_max", "functional", "tlink")):
        assert abs(got[name] - na[k]) <= 1e-13 * max(abs(na[k]), 1e-3), name
