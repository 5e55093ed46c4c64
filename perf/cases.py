"""Workloads for timing the library through its public entry points.

Every case is work that a program linked against the library has it do:
gauge fixing one configuration (Landau or Coulomb), fixing many small ones
in one launch, serving a stream of requests of uneven sizes, and the
measurements around a fixing.  Links are device resident, as the library's
device entry points take them, and contexts are kept between calls, as the
library's own serving loop and benchmark keep them.

The links are SU(3) matrices scattered about unity so that the average
plaquette is that of a quenched beta = 6.0 configuration (0.59), under a
Haar-random gauge transform: a solve starts at the theta a fresh
configuration starts at and runs to theta < 1e-14 through the line-search
iterations and the fixed-step tail.  Without the long-range correlations of
a thermalised field it gets there in about 30 iterations on a trajectory
that does not amplify rounding, so its links can be compared.

`exact` follows the same algorithm (GLU's FACG and its Coulomb form) in
plain torch, complex128 throughout.
"""
import numpy as np
import torch

import glu_amd as gl

ROUGH = 0.36   # link scatter that gives plaquette 0.59
ACC = 1e-14    # GLU's default accuracy
MAX_ITERS = 1000
GF_TUNE = {"landau": 0.08, "coulomb": 0.09}  # GLU's usual fixed steps
CG_TOL = 5e-11
# FP32 -> FP64 switch of the mixed cases: below it the FP32 phase wanders at
# its rounding floor on some of these inputs, for a number of iterations and
# to links that rounding decides
SWITCH = 1e-7
ITERS = 30     # iterations such a solve takes, near enough for work()


# ---------------------------------------------------------------- the cases --
def listed():
    return [
        # one small lattice on a context of its own: launch-bound iterations
        {"name": "landau_8", "kind": "landau", "dims": "8x8x8x8", "precision": "fp64"},
        # extents with factors 5 and 7 and no common length
        {"name": "landau_ragged", "kind": "landau", "dims": "20x28x10x36", "precision": "fp64"},
        # an ordinary lattice at GLU's own precision
        {"name": "landau_24", "kind": "landau", "dims": "24x24x24x48", "precision": "fp64"},
        # the benchmark's lattice in the mixed FP32 -> FP64 schedule
        {"name": "landau_32_mixed", "kind": "landau", "dims": "32x32x32x64", "precision": "mixed"},
        # links smoothed by smearing: few iterations, so the ends of a solve count
        {"name": "smooth_16", "kind": "smooth", "dims": "16x16x16x32", "precision": "fp64"},
        # hundreds of small lattices in one launch
        {"name": "batch_8", "kind": "batch", "dims": "8x8x8x8", "count": 512},
        # the same for extents that are no powers of two, one of them odd
        {"name": "batch_ragged", "kind": "batch", "dims": "6x10x12x9", "count": 96},
        # Coulomb gauge, few small slices
        {"name": "coulomb_16", "kind": "coulomb", "dims": "16x16x16x32"},
        # Coulomb gauge at the largest size the repository is benchmarked at
        {"name": "coulomb_48", "kind": "coulomb", "dims": "48x48x48x96"},
        # a configuration read from a single-precision file: checked and reunitarised
        {"name": "report_32", "kind": "report", "dims": "32x32x32x64"},
        # gluon propagators of a smooth field
        {"name": "gluon_24", "kind": "gluon", "dims": "24x24x24x48", "max_mom": 16, "three_point": False},
        # a queue of requests of uneven sizes through the serving loop
        {"name": "serve", "kind": "serve", "shapes": "8x8x8x8 12x12x12x24 8x8x8x16 16x16x16x32 12x12x12x24 "
                                                     "8x8x8x8 16x16x16x32 8x8x8x16", "precision": "mixed"},
    ]


EXTENTS = (4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 24, 28, 30, 32, 36, 40, 42, 48, 56, 60, 64, 72, 96)


def _dims(rng, lo, hi, extents=EXTENTS):
    """Four extents with a volume spread over lo..hi on its logarithm, near
    the aspect ratios in use (the time extent the longest as a rule)."""
    while True:
        side = (lo * (hi / lo) ** rng.random()) ** 0.25
        d = [rng.choice([e for e in extents if 0.6 * side <= e <= 1.7 * side] or [min(extents)]) for _ in range(4)]
        if rng.random() < 0.5:
            d[1] = d[2] = d[0]
        if lo <= d[0] * d[1] * d[2] * d[3] <= hi:
            return "x".join(map(str, d))


def draw(rng):
    kind = rng.choice(["landau", "landau", "landau", "smooth", "batch", "batch", "coulomb", "coulomb", "report",
                       "gluon", "serve"])
    c = {"kind": kind}
    if kind in ("landau", "smooth"):
        c["dims"] = _dims(rng, 4096, 2_100_000)
        c["precision"] = rng.choice(["fp64", "mixed"]) if kind == "landau" else "fp64"
    elif kind == "batch":
        c["dims"] = _dims(rng, 1296, 16384, tuple(range(4, 17)))
        v = int(np.prod(_ext(c["dims"])))
        c["count"] = rng.randint(1, max(1, 2_000_000 // v))
    elif kind == "coulomb":
        c["dims"] = _dims(rng, 8192, 4_000_000)
    elif kind == "report":
        c["dims"] = _dims(rng, 1024, 4_000_000)
    elif kind == "gluon":
        c["dims"] = _dims(rng, 4096, 1_000_000)
        c["max_mom"], c["three_point"] = rng.randint(4, 24), rng.random() < 0.5
    else:
        c["shapes"] = " ".join(rng.choice(["8x8x8x8", "8x8x8x16", "12x12x12x24", "16x16x16x32", "10x10x10x20"])
                               for _ in range(rng.randint(3, 14)))
        c["precision"] = rng.choice(["fp64", "mixed"])
    return c


def _ext(text):
    return tuple(int(e) for e in text.split("x"))


# --------------------------------------------------------------- the inputs --
def _mul(a, b):
    return (a.unsqueeze(-1) * b.unsqueeze(-3)).sum(-2)


def _mul_dag(a, b):
    """a b^dagger"""
    return (a.unsqueeze(-2) * b.conj().unsqueeze(-3)).sum(-1)


def _complete(c0, c1):
    """SU(3) matrices from their first two columns"""
    return torch.stack([c0, c1, torch.linalg.cross(c0, c1).conj().resolve_conj()], -1)


def _gram(m):
    """Gram-Schmidt on the columns, the third completed"""
    c0, c1 = m[..., 0], m[..., 1]
    c0 = c0 / c0.abs().square().sum(-1, keepdim=True).sqrt()
    c1 = c1 - (c0.conj() * c1).sum(-1, keepdim=True) * c0
    c1 = c1 / c1.abs().square().sum(-1, keepdim=True).sqrt()
    return _complete(c0, c1)


def _gauss(shape, gen):
    return torch.view_as_complex(torch.randn(*shape, 2, dtype=torch.float64, device="cuda", generator=gen))


def _near_unity(shape, eps, gen):
    h = _gauss(shape + (3, 3), gen)
    h = 0.5 * (h + h.conj().transpose(-1, -2))
    return _gram(torch.eye(3, dtype=torch.complex128, device="cuda") + 1j * eps * h)


def _links(dims, seed, scatter, turn, batch=1):
    """Links (batch, T, Z, Y, X, 4, 3, 3): scattered about unity, then under
    a gauge transform (turn: "haar", or the size of a small one)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    shape = (batch,) + dims[::-1]
    g = _gram(_gauss(shape + (3, 3), gen)) if turn == "haar" else _near_unity(shape, turn, gen) if turn else None
    out = torch.empty(shape + (4, 3, 3), dtype=torch.complex128, device="cuda")
    for mu in range(4):
        u = _near_unity(shape, scatter, gen)
        if g is not None:
            u = _mul(g, _mul_dag(u, torch.roll(g, -1, 4 - mu)))
        out[..., mu, :, :] = u
    return out


def _glu_layout(u):
    """double[batch, V, 4, 18], x fastest, row-major re / im pairs"""
    return torch.view_as_real(u).reshape(u.shape[0], -1, 4, 18)


def _case_links(case, seed):
    kind, dims = case["kind"], _ext(case["dims"])
    if kind == "smooth":
        return _links(dims, seed, 0.1, 0.2)
    if kind == "gluon":
        return _links(dims, seed, 0.1, 0)
    if kind == "report":  # as read from a single-precision file
        return _links(dims, seed, ROUGH, 0.5).to(torch.complex64).to(torch.complex128)
    return _links(dims, seed, ROUGH, "haar", case.get("count", 1))


PRECISION = {"fp64": gl.FP64, "mixed": gl.MIXED}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        shapes = [_ext(t) for t in case["shapes"].split()]
        inputs = [_glu_layout(_links(d, 1000 * seed + k, ROUGH, "haar"))[0] for k, d in enumerate(shapes)]
        return {"kind": kind, "shapes": shapes, "inputs": inputs, "work": [torch.empty_like(u) for u in inputs],
                "precision": PRECISION[case["precision"]], "server": gl.Server(max_active=8, switch_theta=SWITCH)}
    dims = _ext(case["dims"])
    links = _glu_layout(_case_links(case, seed))
    state = {"kind": kind, "dims": dims, "links": links, "out": torch.empty_like(links)}
    if kind == "batch":
        state["count"] = case["count"]
    else:
        state["ctx"] = gl.Gfix(dims, gl.COULOMB if kind == "coulomb" else gl.LANDAU,
                               PRECISION[case.get("precision", "fp64")])
        if case.get("precision") == "mixed":
            state["ctx"].set_switch_theta(SWITCH)
    if kind == "gluon":
        state |= {"max_mom": case["max_mom"], "three_point": case["three_point"]}
    return state


# ----------------------------------------------------------------- one pass --
def run(state):
    kind = state["kind"]
    if kind == "serve":
        for u, w in zip(state["inputs"], state["work"]):
            w.copy_(u)
        torch.cuda.synchronize()  # the server reads the buffers on streams of its own
        srv = state["server"]
        tickets = [srv.submit(d, w.data_ptr(), gl.LANDAU, state["precision"], gl.CG, GF_TUNE["landau"], ACC, MAX_ITERS)
                   for d, w in zip(state["shapes"], state["work"])]
        iters = [srv.wait(t)[0] for t in tickets]
        return {"iters": np.array(iters), "links": state["work"]}
    if kind == "batch":
        state["out"].copy_(state["links"])
        iters, _ = gl.facg_batch(state["dims"], state["out"].data_ptr(), state["count"], GF_TUNE["landau"], ACC,
                                 MAX_ITERS)
        return {"iters": np.array(iters), "links": state["out"]}
    g = state["ctx"]
    g.set_links_device(state["links"].data_ptr())
    if kind == "gluon":
        f = g.gluon_exceptional if state["three_point"] else g.gluon_props
        mom, a, b, err = f("psq", state["max_mom"])
        return {"mom": mom, "a": a, "b": b, "err": err}
    if kind == "report":
        out = {**g.measure(), "theta": g.theta()}
        g.reunit()
    elif kind == "coulomb":
        g.run(gl.CG, GF_TUNE["coulomb"], ACC, MAX_ITERS)
        out = {"iters": np.array(g.slice_info()[0])}
    else:
        iters, _, restarts = g.landau(gl.CG, GF_TUNE["landau"], ACC, MAX_ITERS)
        out = {"iters": iters, "restarts": restarts}
    g.get_links_device(state["out"].data_ptr())
    out["links"] = state["out"]
    return out


# --------------------------------------------------- what a pass has to move --
def work(case):
    kind = case["kind"]
    if kind == "serve":
        each = [work({"kind": "landau", "dims": t, "precision": case["precision"]}) for t in case["shapes"].split()]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    v = float(np.prod(_ext(case["dims"]))) * case.get("count", 1)
    io = 2 * 576.0 * v  # GLU's 72 doubles a site, in and out
    if kind == "report":
        return {"bytes": io, "flops": 4500.0 * v}
    if kind == "gluon":
        # the links in; 16 packed fields out and in once for the planes, once for the columns
        return {"bytes": (576.0 + 4 * 256.0) * v, "flops": 16 * 5 * np.log2(v) * v}
    # an iteration: two columns of every link it moves read and written, and
    # the 4 packed fields -- derivative out, accelerated field in, old field
    # in, direction in and out, each 64 B a site
    if kind == "coulomb":
        per, flops, n = 3 * 96.0 + 2 * 96.0 + 5 * 64.0, 6000.0, ITERS
    else:
        half = 0.5 if case.get("precision") == "mixed" else 1.0
        per, flops = half * (2 * 384.0 + 5 * 64.0), 8000.0
        n = 9 if kind == "smooth" else ITERS
    return {"bytes": io + n * per * v, "flops": n * (flops + 4 * 2 * 5 * np.log2(v)) * v}


# ------------------------------------------- the same answers in plain torch --
def _pack(u, dims4):
    """The packed divergence of the links u[..., D, 3, 3] (axes b, T, Z, Y, X
    or b, Z, Y, X), 4 complex fields in front (Gfix/FACG.c:38-73)."""
    nd = u.shape[-3]
    delta = 0
    for mu in range(nd):
        m = u[..., mu, :, :]
        a = -0.5j * (m - m.conj().transpose(-1, -2))
        a = a - (a.diagonal(dim1=-2, dim2=-1).sum(-1) / 3)[..., None, None] * torch.eye(3, dtype=a.dtype, device=a.device)
        delta = delta + torch.roll(a, 1, dims4[mu]) - a
    f0 = torch.complex(-delta[..., 1, 1].real, delta[..., 0, 0].real)
    return torch.stack([f0, 1j * delta[..., 0, 1], 1j * delta[..., 0, 2], 1j * delta[..., 1, 2]])


def _gauge(f, alpha):
    """P(1 + alpha X) of the packed fields (Gfix/CG.c:47-100); alpha: (b)"""
    al = alpha.reshape(alpha.shape + (1,) * (f[0].dim() - 1)).to(f.dtype)
    x = al * f
    one = torch.ones_like(x[0])
    c0 = torch.stack([one + 1j * x[0].imag, -x[1].conj(), -x[2].conj()], -1)
    c1 = torch.stack([x[1], one - 1j * x[0].real, -x[3].conj()], -1)
    c0 = c0 / c0.abs().square().sum(-1, keepdim=True).sqrt()
    c1 = c1 - (c0.conj() * c1).sum(-1, keepdim=True) * c0
    return _complete(c0, c1 / c1.abs().square().sum(-1, keepdim=True).sqrt())


def _sums(f, old):
    """GLU's trace-metric <f, f> and <f, f - old> per lattice (Gfix/FACG.c:99-178)"""
    ax = tuple(range(1, f[0].dim()))
    d = f - old
    s1 = 2 * f.abs().square().sum(0) + 2 * f[0].real * f[0].imag
    s2 = 2 * (f.real * d.real + f.imag * d.imag).sum(0) + f[0].real * d[0].imag + f[0].imag * d[0].real
    return s1.sum(ax), s2.sum(ax)


def _rotate(u, g, axes):
    return torch.stack([_mul(g, _mul_dag(u[..., mu, :, :], torch.roll(g, -1, axes[mu]))) for mu in range(len(axes))], -3)


def _vertex(al, f):
    """GLU's parabola through the probes (Gfix/line_search.c:38-57)"""
    a = f[0] / ((al[0] - al[1]) * (al[0] - al[2]))
    b = f[1] / ((al[1] - al[0]) * (al[1] - al[2]))
    c = f[2] / ((al[2] - al[0]) * (al[2] - al[1]))
    s = (al[0] * (b + c) + al[1] * (a + c) + al[2] * (a + b)) / (2 * (a + b + c))
    return torch.where(s > al[2], torch.full_like(s, al[2]),
                       torch.where(~torch.isfinite(s) | (s < al[0]), torch.full_like(s, 0.08), s))


def _facg(u, landau):
    """FACG of a batch of lattices or slices u[b, ..., D, 3, 3]: the total
    transform of each."""
    nd = u.shape[-3]
    b, ext = u.shape[0], u.shape[1:1 + nd]
    axes = [nd - mu for mu in range(nd)]
    ax = tuple(range(1, nd + 1))
    vol = int(np.prod(ext))
    cos = 0
    for mu in range(nd):
        n = ext[nd - 1 - mu]
        shape = [1] * nd
        shape[nd - 1 - mu] = n
        cos = cos + torch.cos(torch.arange(n, dtype=torch.float64, device=u.device) * (2 * np.pi / n)).reshape(shape)
    psq = 2 * (nd - cos)
    psq.view(-1)[0] = 1.0
    scale = 4.0 * nd / psq  # GLU: 4 nd / vol / p^2 between unnormalised transforms
    probes = (0.0, 0.15, 0.30) if landau else (0.0, 0.17, 0.34)
    step = GF_TUNE["landau" if landau else "coulomb"]
    g = _gram(torch.eye(3, dtype=u.dtype, device=u.device).expand((b,) + tuple(ext) + (3, 3)).contiguous())
    cur = u
    live = torch.ones(b, dtype=torch.bool, device=u.device)
    inold = sn = old = None
    for k in range(MAX_ITERS):
        f = _pack(cur, axes)
        theta = (4 * f.abs().square().sum(0) - 4 * f[0].real * f[0].imag).sum(ax) / (3.0 * vol)
        f = torch.fft.ifftn(torch.fft.fftn(f, dim=tuple(a + 1 for a in ax)) * scale, dim=tuple(a + 1 for a in ax))
        s1, s2 = _sums(f, old if old is not None else torch.zeros_like(f))
        if not landau:
            theta = s1 / (3.0 * vol)
        beta = torch.zeros_like(s1)
        if k:
            beta = torch.where(theta < CG_TOL, s1 / inold, (s2 / inold).clamp(min=0.0))
            sn = f + beta.reshape((b,) + (1,) * nd) * sn
        else:
            sn = f
        tr = []
        for p in probes:
            m = _gauge(sn, torch.full_like(theta, p))
            tr.append(-sum((_mul_dag(_mul(m, cur[..., mu, :, :]), torch.roll(m, -1, axes[mu]))
                            .diagonal(dim1=-2, dim2=-1).real.sum(-1)).sum(ax) for mu in range(nd)))
        alpha = _vertex(probes, tr)
        if k:
            alpha = torch.where(theta > CG_TOL, alpha, torch.full_like(alpha, step))
        m = _gauge(sn, alpha)
        keep = live.reshape((b,) + (1,) * (nd + 2))
        g = torch.where(keep, _mul(m, g), g)
        cur = torch.where(keep.unsqueeze(-1), _rotate(cur, m, axes), cur)
        inold, old = s1, f
        if k:
            live = live & (theta > ACC)
            if not bool(live.any()):
                break
    return g


def _plaquettes(u, axes):
    tot = 0.0
    for mu in range(4):
        for nu in range(mu):
            a = _mul(u[..., mu, :, :], torch.roll(u[..., nu, :, :], -1, axes[mu]))
            c = _mul(u[..., nu, :, :], torch.roll(u[..., mu, :, :], -1, axes[nu]))
            tot += (a.real * c.real + a.imag * c.imag).sum().item()
    return tot


def _gluon(u, case):
    """G, F (or g2, g3) and GLU's momentum-space figure on the psq list
    (Cuts/glueprop.c:32-151, Cuts/MOMgg.c:94-215)"""
    dims = _ext(case["dims"])
    v = float(np.prod(dims))
    small = min(dims)
    k = np.stack(np.meshgrid(*[np.arange(n) - n // 2 for n in dims[::-1]], indexing="ij")[::-1], -1).reshape(-1, 4)
    ratio = np.array([small / n for n in dims])
    mom = k[((k * ratio) ** 2).sum(1) <= case["max_mom"]]
    n, zero = len(mom), (len(mom) - 1) // 2
    site = [torch.from_numpy(mom[:, mu] % dims[mu]).cuda() for mu in range(4)]
    at = torch.from_numpy(mom).cuda().double()
    p = torch.stack([2 * torch.sin(at[:, mu] * (np.pi / dims[mu])) for mu in range(4)], 1)
    a = []
    for mu in range(4):
        m = u[0, ..., mu, :, :]
        h = -0.5j * (m - m.conj().transpose(-1, -2))
        h = h - (h.diagonal(dim1=-2, dim2=-1).sum(-1) / 3)[..., None, None] * torch.eye(3, dtype=h.dtype, device=h.device)
        h = torch.fft.ifftn(h, dim=(0, 1, 2, 3)) * v
        phase = torch.exp(1j * np.pi * at[:, mu] / dims[mu])
        a.append(h[site[3], site[2], site[1], site[0]] * phase[:, None, None])
    a = torch.stack(a, 1)  # (n, mu, 3, 3)
    err = (a * p[..., None, None]).sum((1, 2, 3)).abs() / 3
    psq = p.square().sum(1)
    psq = torch.where(psq < 3e-14, torch.ones_like(psq), psq)
    if not case["three_point"]:
        flat = a.reshape(n, 4, 9)
        gram = (flat.unsqueeze(2) * flat.conj().unsqueeze(1)).sum(-1).real
        lo = (p.unsqueeze(2) * p.unsqueeze(1) * gram).sum((1, 2)) / psq
        tr = gram.diagonal(dim1=1, dim2=2).sum(1) - lo
        norm = torch.full((n,), 2.0 / (24.0 * v), dtype=torch.float64, device="cuda")
        norm[n >> 1] = 2.0 / (32.0 * v)
        x, y = tr * norm, lo * (2.0 / (8.0 * v))
        half = n >> 1
        x[half + 1:], y[half + 1:] = x[:n - half - 1].flip(0), y[:n - half - 1].flip(0)
    else:
        am = a.flip(0)
        tr = (a * am.transpose(-1, -2)).sum((1, 2, 3)).real
        norm = torch.full((n,), 2.0 / (24.0 * v), dtype=torch.float64, device="cuda")
        norm[zero] = 2.0 / (32.0 * v)
        x = tr * norm
        w = p[..., None, None]
        rho, aa, ap = (a[zero] * w).sum(1), _mul(a, am).sum(1), (a * w).sum(1)
        amin = (am * -w).sum(1) / psq[:, None, None]
        t3 = (_mul(aa, rho) + _mul(_mul(rho, ap), amin)).diagonal(dim1=-2, dim2=-1).sum(-1).real
        y = t3 / psq * (4.0 / (2.0 * 3 * 8 * 3 * v))
    return {"mom": None, "a": x, "b": y, "err": err.sum().item() / n}


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        links = []
        for k, t in enumerate(case["shapes"].split()):
            u = _links(_ext(t), 1000 * seed + k, ROUGH, "haar")
            links.append(_glu_layout(_rotate(u, _facg(u, True), [4, 3, 2, 1]))[0])
        return {"iters": None, "links": links}
    u = _case_links(case, seed)
    axes = [4, 3, 2, 1]
    if kind == "gluon":
        return _gluon(u, case)
    if kind == "report":
        # the library holds a link's first two columns
        u = _complete(u[..., 0], u[..., 1])
        v = u[..., 0, 0, 0].numel()
        tr = u.diagonal(dim1=-2, dim2=-1).real.sum(-1)
        f = _pack(u, axes)
        theta = (4 * f.abs().square().sum() - 4 * (f[0].real * f[0].imag).sum()).item() / (3.0 * v)
        link = tr.sum().item() / (12.0 * v)
        return {"plaquette": 2 * _plaquettes(u, axes) / (36.0 * v), "link_trace": link, "link_max": tr.max().item() / 3,
                "functional": 1 - link, "tlink": tr[..., 3].sum().item() / (3.0 * v), "theta": 2 * theta,
                "links": _glu_layout(_gram(u))}
    if kind == "coulomb":
        slices = u[0, ..., :3, :, :]  # every time slice a problem of its own
        g = _gram(_facg(slices, False))
        return {"iters": None, "links": _glu_layout(_rotate(u, g.unsqueeze(0), axes))}
    out = {"iters": None, "links": _glu_layout(_rotate(u, _facg(u, True), axes))}
    return out if kind == "batch" else {**out, "restarts": None}
