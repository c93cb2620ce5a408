"""The transforms whose speed is tracked, as a user's program calls them.

A case is one call of ``fgt2d`` or ``fgt3d``: points, charges (and dipoles) in,
potentials (and gradients, Hessians) out.  The listed cases cover the range
that the tests, the benchmark and the served request stream use: 10^3 to 2M +
2M points in 2D and 2*10^3 to 8M + 8M in 3D, precisions 1e-3 to 5e-11, uniform
and strongly clustered points, one and two densities, charges alone and with
dipoles, potentials alone and with derivatives, at the sources and at separate
targets, from GPU tensors and from host arrays, in both arithmetic modes.
"""
import math

import torch

import fgt2d_amd

SIGMA, CENTRES = 0.01, 10  # the Gaussian mixture of the clustered 2D workload


def _case(name, dim, points, ns, nt, delta, eps, nd=1, at_src=1, at_trg=0, dipoles=False,
          mixed=False, host=False):
    """at_src, at_trg: 0 nothing, 1 potentials, 2 and gradients, 3 and Hessians."""
    c = dict(dim=dim, points=points, ns=ns, nt=nt, delta=delta, eps=eps, nd=nd, at_src=at_src,
             at_trg=at_trg, dipoles=dipoles, mixed=mixed, host=host)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest request of the served stream (N from 10^3): launches and read-backs
        _case("2d_1k", 2, "uniform", 1000, 0, 1e-4, 1e-6),
        # the stream's median size as its clients and a Fortran program hand
        # it over: host arrays in and out, low accuracy
        _case("2d_30k_host", 2, "uniform", 31623, 0, 1e-3, 1e-3, host=True),
        # the 100k workload of the benchmark: its top level has orders above
        # 50, so leaves there are evaluated from their plane waves
        _case("2d_100k", 2, "uniform", 100000, 0, 1e-4, 1e-9),
        # charges and dipoles, two densities, derivatives at odd-sized targets
        _case("2d_dipoles", 2, "mixture", 123457, 76543, 1e-4, 1e-6, nd=2, at_trg=3, dipoles=True),
        # the reference test driver's size, spacing and accuracy, with the
        # gradients a particle code moves its points by
        _case("2d_1m_grad", 2, "uniform", 1000000, 0, (1 / 64.) ** 2 / (1.5 * 1.5) / 16, 5e-11,
              at_src=2),
        # the headline workload in both arithmetic modes
        _case("2d_mixture_2m", 2, "mixture", 2000000, 2000000, 1e-5, 1e-6, at_src=0, at_trg=1),
        _case("2d_mixture_2m_mixed", 2, "mixture", 2000000, 2000000, 1e-5, 1e-6, at_src=0,
              at_trg=1, mixed=True),
        # small 3D request, odd size
        _case("3d_2k", 3, "uniform", 2053, 0, 1e-3, 1e-6),
        # high accuracy with derivatives on both sides (the 3D parity test's
        # kind of call), a ragged target count
        _case("3d_50k_hess", 3, "uniform", 50000, 20011, 3e-3, 1e-9, at_src=2, at_trg=3),
        # the reference 3D test driver's configuration
        _case("3d_300k", 3, "uniform", 300000, 0, 1.2e-3, 1e-6),
        # the 1M workload of the benchmark
        _case("3d_1m", 3, "uniform", 1000000, 0, 1e-3, 1e-6),
        # the largest: 8M sources on a spherical shell, 8M uniform targets
        _case("3d_shell_8m", 3, "shell", 8000000, 8000000, 1e-5, 1e-9, at_src=0, at_trg=1),
    ]


def draw(rng):
    """A request of the served stream's ranges (delta log-uniform in [1e-6,
    1e-2], eps 1e-3, 1e-6 or 1e-9, N log-uniform), with the listed cases'
    options: the more a point costs, the fewer of them."""
    dim = rng.choice((2, 3))
    eps = rng.choice((1e-3, 1e-6, 1e-9))
    delta = 10.0 ** rng.uniform(-6, -2)
    nd = rng.choice((1, 1, 1, 2))
    dipoles = rng.random() < 0.25
    at_src, at_trg = rng.choice(((1, 0), (1, 0), (0, 1), (1, 1), (2, 0), (2, 3), (0, 2)))
    top = 2e6 if dim == 2 else (1e6 if eps > 1e-8 else 1.5e5)
    if nd > 1 or dipoles or max(at_src, at_trg) > 1:
        top /= 4
    ns = int(10.0 ** rng.uniform(3, math.log10(top))) | 1
    nt = int(ns * rng.uniform(0.2, 1.0)) + 1 if at_trg else 0
    points = rng.choice(("uniform", "uniform", "mixture" if dim == 2 else "shell"))
    host = ns < 200000 and rng.random() < 0.15
    mixed = dim == 2 and eps >= 1e-6 and rng.random() < 0.3
    return _case(None, dim, points, ns, nt, delta, eps, nd, at_src, at_trg, dipoles, mixed, host)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _points(case, g):
    """(sources, targets or None) on the GPU."""
    dim, ns, nt = case["dim"], case["ns"], case["nt"]

    def unif(n, d=dim):
        return torch.rand((n, d), generator=g, device="cuda", dtype=torch.float64)

    def normal(*s):
        return torch.randn(s, generator=g, device="cuda", dtype=torch.float64)

    if case["points"] == "mixture":
        mu = 0.1 + 0.8 * unif(CENTRES)

        def mix(n):
            k = torch.randint(0, CENTRES, (n,), generator=g, device="cuda")
            return (mu[k] + SIGMA * normal(n, dim)).clamp_(0.0, 1.0)
        return mix(ns), (mix(nt) if nt else None)
    if case["points"] == "shell":
        d = normal(ns, 3)
        d /= d.norm(dim=1, keepdim=True)
        src = 0.5 + d * (0.4 + 1e-3 * normal(ns, 1))
        return src, (unif(nt) if nt else None)
    return unif(ns), (unif(nt) if nt else None)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    src, trg = _points(case, g)
    ns, nd = case["ns"], case["nd"]
    if case["points"] == "mixture":
        chg = torch.randn((ns, nd), generator=g, device="cuda", dtype=torch.float64)
    else:
        chg = 2 * torch.rand((ns, nd), generator=g, device="cuda", dtype=torch.float64) - 1
    st = dict(case=case, src=src, trg=trg, chg=chg, normals=None, strengths=None)
    if case["dipoles"]:
        n = torch.randn((ns, case["dim"]), generator=g, device="cuda", dtype=torch.float64)
        st["normals"] = n / n.norm(dim=1, keepdim=True)
        # as large an effect as the charges': a dipole's field is 2/delta r
        # times a charge's
        st["strengths"] = math.sqrt(case["delta"]) * torch.randn(
            (ns, nd), generator=g, device="cuda", dtype=torch.float64)
    if case["host"]:
        for k, v in st.items():
            if isinstance(v, torch.Tensor):
                st[k] = v.cpu().numpy()
    return st


def run(state):
    c = state["case"]
    fgt2d_amd.set_precision("mixed" if c["mixed"] else "fp64")
    f = fgt2d_amd.fgt2d if c["dim"] == 2 else fgt2d_amd.fgt3d
    out = f(c["delta"], c["eps"], state["src"], state["chg"], state["trg"], ifpgh=c["at_src"],
            ifpghtarg=c["at_trg"], ifdipole=int(c["dipoles"]), rnormal=state["normals"],
            dipstr=state["strengths"])
    return [o for o in out if o is not None]


def _widths(case):
    """Values per point and density: potentials, gradients, Hessians."""
    d = case["dim"]
    return (1, d, 3 if d == 2 else 6)


def work(case):
    """Each input read and each output written once.  Operations: every point
    meets one expansion of the deepest leaves' order (18 in 2D, 15 in 3D)
    per density and derivative, or the points within the cutoff distance
    directly (about 20 operations a pair), whichever is less."""
    d, ns, nt, nd = case["dim"], case["ns"], case["nt"], case["nd"]
    w = _widths(case)
    outs = ns * sum(w[:case["at_src"]]) + nt * sum(w[:case["at_trg"]])
    ins = ns * (d + nd) + (ns * (d + nd) if case["dipoles"] else 0) + nt * d
    terms = 19 ** 2 if d == 2 else 16 ** 3
    expand = 2.0 * terms * nd * (ns * (1 + (d if case["dipoles"] else 0)) + outs)
    rc = math.sqrt(case["delta"] * math.log(1 / case["eps"]))
    ball = min(1.0, math.pi * rc ** 2 if d == 2 else 4.19 * rc ** 3)
    n_eval = (ns if case["at_src"] else 0) + nt
    direct = 20.0 * nd * ns * n_eval * ball
    return {"bytes": 8.0 * (ins + nd * outs), "flops": min(expand, direct)}


def tolerance(case):
    """Measured: the FP64 transform against another implementation of the same
    expansions (other recurrences, other summation orders) differs by up to
    8e-15 in the 2-norm, and by 2e-12 of the root mean square at single points
    of the order-62 Hessians; high orders of clustered draws with dipoles get
    a decade more.  The mixed mode against FP64: 3.5e-7."""
    if case["mixed"]:
        return {"rel": 1.4e-6}
    return {"rel": 1e-13, "max": 1e-11}


# ---------------------------------------------------------------------------
# the sums themselves, in 64 bits
# ---------------------------------------------------------------------------
CUT = 45.0          # pairs with r^2 > CUT delta contribute below 3e-20
MOST_PAIRS = 7e11   # about 10 seconds
TILE = 1 << 27      # pairs at once


def _sums(t, s, q, w, delta, level):
    """Potentials, gradients, Hessians (the first `level` of them) at t of the
    charges q (n, nd) and dipoles w (n, nd, d) at s; t and s are offsets from
    one centre near both."""
    d, c = t.shape[1], 2.0 / delta
    one = torch.ones_like
    left = torch.cat([t, (t * t).sum(1, keepdim=True), one(t[:, :1])], 1)
    right = torch.cat([c * s, -one(s[:, :1]) / delta, -(s * s).sum(1, keepdim=True) / delta], 1)
    k = (left @ right.t().contiguous()).exp_()

    def moment(f, axes=()):
        # sum over the sources of K f prod_i (t_i - s_i)
        if not axes:
            return k @ f
        i = axes[0]
        return t[:, i:i + 1] * moment(f, axes[1:]) - moment(s[:, i:i + 1] * f, axes[1:])

    def with_dipoles(axes):
        # sum of K (q + c w.r) prod r_i
        v = moment(q, axes)
        if w is not None:
            for j in range(d):
                v = v + c * moment(w[:, :, j].contiguous(), axes + (j,))
        return v

    def dip(j, axes):
        return moment(w[:, :, j].contiguous(), axes) if w is not None else 0.0

    out = [with_dipoles(())]
    if level >= 2:
        out.append(torch.stack([c * (dip(i, ()) - with_dipoles((i,))) for i in range(d)], 1))
    if level >= 3:
        # xx, xy, yy in 2D; xx, yy, zz, xy, xz, yz in 3D
        pairs = ((0, 0), (0, 1), (1, 1)) if d == 2 else ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2),
                                                         (1, 2))
        out.append(torch.stack([
            c * c * (with_dipoles((i, j)) - dip(j, (i,)) - dip(i, (j,)))
            - (c * out[0] if i == j else 0.0) for i, j in pairs], 1))
    return out


def _direct(trg, src, q, w, delta, level):
    """The sums at every target, by columns of cells of the cutoff's size;
    None when that would take too long."""
    rc = math.sqrt(CUT * delta)
    nc = max(1, min(48, int(1.0 / rc)))

    def cell(p):
        return (p[:, :2].clamp(0.0, 1.0 - 1e-12) * nc).long()
    ts, ss = cell(trg), cell(src)
    ti, si = ts[:, 0] * nc + ts[:, 1], ss[:, 0] * nc + ss[:, 1]
    to, so = torch.argsort(ti), torch.argsort(si)
    tn = torch.bincount(ti, minlength=nc * nc).cpu().tolist()
    sn = torch.bincount(si, minlength=nc * nc).cpu().tolist()
    ta, sa = [0], [0]
    for i in range(nc * nc):
        ta.append(ta[-1] + tn[i])
        sa.append(sa[-1] + sn[i])
    # a row of up to three neighbour cells is one run of the sorted sources
    runs = []
    for i in range(nc * nc):
        x, y = divmod(i, nc)
        y0, y1 = max(0, y - 1), min(nc - 1, y + 1)
        runs.append([(sa[a * nc + y0], sa[a * nc + y1 + 1])
                     for a in range(max(0, x - 1), min(nc - 1, x + 1) + 1)])
    if sum(tn[i] * sum(b - a for a, b in runs[i]) for i in range(nc * nc)) * level > MOST_PAIRS:
        return None
    d, nd = trg.shape[1], q.shape[1]
    outs = [torch.zeros((trg.shape[0],) + shape, device=trg.device, dtype=torch.float64)
            for shape in ((nd,), (d, nd), (3 if d == 2 else 6, nd))[:level]]
    trg, src, q = trg[to], src[so], q[so]
    w = w[so] if w is not None else None
    for i in range(nc * nc):
        if not tn[i]:
            continue
        x, y = divmod(i, nc)
        centre = torch.tensor([(x + 0.5) / nc, (y + 0.5) / nc, 0.5][:d], device=trg.device,
                              dtype=torch.float64)
        for a, b in runs[i]:
            if a == b:
                continue
            s = src[a:b] - centre
            step = max(1, TILE // (b - a))
            for t0 in range(ta[i], ta[i + 1], step):
                t1 = min(ta[i + 1], t0 + step)
                v = _sums(trg[t0:t1] - centre, s, q[a:b], w[a:b] if w is not None else None,
                          delta, level)
                for o, x_ in zip(outs, v):
                    o[to[t0:t1]] += x_
    return outs


def exact(case, seed):
    st = prepare(dict(case, host=False), seed)
    w = None
    if case["dipoles"]:
        w = st["normals"][:, None, :] * st["strengths"][:, :, None]
    out = []
    for pts, level in ((st["src"], case["at_src"]), (st["trg"], case["at_trg"])):
        if pts is None or not level:
            continue
        v = _direct(pts, st["src"], st["chg"], w, case["delta"], level)
        if v is None:
            return None
        out += v
    return [o.cpu().numpy() for o in out] if case["host"] else out
