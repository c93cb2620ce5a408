"""3D transforms whose cutoff-level boxes are formed and evaluated whole
(k_form3_top, k_eval3_top), against the 3D oracle: every width of the kernels'
plane-wave tiles (npw 12, 18, 26, 32, 38, 44, 52), values, gradients and
Hessians, charges and dipoles, several densities, leaves one to three levels
below the cutoff, leaves on the plane-wave route, boxes of less than one tile of points
and ragged segments; and dense transforms, which stay leaf by leaf.

Tolerance: both sides sum the same FP64 expansions in another order; the
largest difference over the largest value is bounded by the phases'
magnification of one rounding, exp(x^2) per axis with x^2 <= ln(1/eps)/4, which
at eps = 1e-12 is 1e9 eps_machine = 2e-7 in the worst case of one node and is
seen below 1e-12 throughout."""
import numpy as np
import pytest

import fgt2d_amd
from oracle import oracle as O

pytestmark = pytest.mark.gpu

NAMES = ["pot", "grad", "hess", "pottarg", "gradtarg", "hesstarg"]

# (points, ns, nt, delta, eps, nd, ifpgh, ifpghtarg, charges, dipoles, route)
CASES = [
    ("uniform", 6001, 1501, 1e-2, 1e-3, 1, 1, 1, True, False, True),   # npw 12
    ("uniform", 6001, 37, 1e-2, 1e-3, 2, 2, 3, True, False, True),     # npw 18, short segments
    ("uniform", 9000, 1, 1e-2, 1e-6, 1, 1, 1, True, False, True),      # npw 26, one target
    ("shell", 20001, 2003, 1e-3, 1e-6, 1, 3, 2, True, True, True),      # npw 32, dipoles
    ("shell", 7001, 0, 4e-3, 1e-6, 3, 1, 0, False, True, True),        # dipoles only, nd 3
    ("cluster", 6000, 900, 1e-5, 1e-9, 1, 2, 1, True, False, True),    # npw 38
    ("cluster", 3001, 333, 1e-5, 1e-9, 1, 1, 3, True, True, True),     # npw 44
    ("uniform", 5000, 400, 1e-2, 1e-12, 1, 2, 1, True, False, True),   # npw 52: the widest tiles
    ("uniform", 3000, 200, 2e-2, 1e-12, 1, 1, 2, True, False, True),
    ("uniform", 60000, 500, 1e-2, 1e-6, 1, 1, 1, True, False, False),  # full leaves: leaf by leaf
    # its few leaves of order 33 are all refined by the level restriction
    ("mixture", 27703, 0, 7e-3, 1e-9, 1, 2, 0, True, False, False),
]


def _points(kind, rng, n):
    if kind == "uniform":
        return rng.random((n, 3))
    if kind == "cluster":
        return 0.485 + 0.03 * rng.random((n, 3))
    if kind == "mixture":
        mu = rng.uniform(0.1, 0.9, (10, 3))
        return np.clip(mu[rng.integers(0, 10, n)] + 0.01 * rng.normal(size=(n, 3)), 0.0, 1.0)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return 0.5 + d * (0.4 + 1e-3 * rng.normal(size=(n, 1)))


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_whole_box_route_matches_oracle(case):
    kind, ns, nt, delta, eps, nd, ifs, ift, ifc, ifd, route = case
    print("case", case, flush=True)
    rng = np.random.default_rng(ns + nt)
    src = _points(kind, rng, ns)
    tg = _points(kind, rng, nt) if nt else None
    chg = rng.normal(size=(ns, nd)) if ifc else None
    rn = rng.normal(size=(ns, 3)) if ifd else None
    ds = np.sqrt(delta) * rng.normal(size=(ns, nd)) if ifd else None
    fgt2d_amd.set_timing(True)
    try:
        got = fgt2d_amd.fgt3d(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift,
                              ifdipole=int(ifd), rnormal=rn, dipstr=ds)
        kernels = {k["kernel"] for k in fgt2d_amd.kernel_launches()}
    finally:
        fgt2d_amd.set_timing(False)
    st = fgt2d_amd.last_stats()
    assert st["nlevels"] > max(st["npwlevel"], 0), st  # expansions
    assert ("form_top" in kernels) == route, (kernels, st)
    want = O.oracle_fgt3d(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift, rnormal=rn,
                          dipstr=ds)
    for k, (g, w) in enumerate(zip(got, want)):
        if (k < 3 and k < ifs) or (k >= 3 and k - 3 < ift):
            g, w = np.asarray(g), np.asarray(w)
            assert np.abs(g - w).max() < 1e-11 * np.abs(w).max(), NAMES[k]


# (extent of the points, ns, nt, delta, eps, ifpgh, ifpghtarg, dipoles)
FEW_NODES = [
    (0.25, 500, 0, 1.0, 0.1, 1, 0, False),
    (1.0, 900, 200, 6.9, 0.2, 2, 1, False),
    (1.0, 600, 100, 6.9, 0.2, 1, 0, True),
]


@pytest.mark.parametrize("case", FEW_NODES, ids=[str(i) for i in range(len(FEW_NODES))])
def test_no_plane_wave_nodes(case):
    """Boxes so small and accuracies so low that the expansions have no node
    at all: they add nothing, as in the oracle, and the call is no error."""
    ext, ns, nt, delta, eps, ifs, ift, ifd = case
    print("case", case, flush=True)
    rng = np.random.default_rng(ns)
    src, chg = ext * rng.random((ns, 3)), rng.normal(size=(ns, 1))
    tg = ext * rng.random((nt, 3)) if nt else None
    rn = rng.normal(size=(ns, 3)) if ifd else None
    ds = rng.normal(size=(ns, 1)) if ifd else None
    got = fgt2d_amd.fgt3d(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift, ifdipole=int(ifd),
                          rnormal=rn, dipstr=ds)
    st = fgt2d_amd.last_stats()
    assert st["npw"] == 0 and st["nlevels"] > st["npwlevel"], st
    want = O.oracle_fgt3d(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift, rnormal=rn,
                          dipstr=ds)
    for k, (g, w) in enumerate(zip(got, want)):
        if (k < 3 and k < ifs) or (k >= 3 and k - 3 < ift):
            assert np.array_equal(np.asarray(g), np.asarray(w)), NAMES[k]
