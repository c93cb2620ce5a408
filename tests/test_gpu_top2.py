"""2D transforms whose cutoff-level boxes are formed and evaluated whole
(k_form2_top, k_eval2_top), against the oracle: every width of the kernels'
plane-wave tiles (npw 12, 18, 26, 32, 38, 44, 52), values, gradients and
Hessians, charges and dipoles, several densities, leaves one to three levels
below the cutoff, cutoff-level leaves on the plane-wave route, segments of less
than one tile and ragged ones; and transforms that stay leaf by leaf (full
leaves, the mixed arithmetic).

Tolerance: both sides sum the same FP64 expansions in another order, as the
other parity tests."""
import numpy as np
import pytest

import fgt2d_amd
from oracle import oracle as O
from tests import _pts

pytestmark = pytest.mark.gpu

NAMES = ["pot", "grad", "hess", "pottarg", "gradtarg", "hesstarg"]

# (points, ns, nt, delta, eps, nd, ifpgh, ifpghtarg, charges, dipoles, whole boxes)
CASES = [
    ("uniform", 12001, 3001, 1e-3, 1e-3, 1, 1, 1, True, False, True),    # npw 12
    ("uniform", 9001, 17, 1e-3, 1e-3, 2, 2, 3, True, False, True),       # npw 18
    ("uniform", 30011, 1, 5e-4, 1e-6, 1, 1, 1, True, False, True),       # npw 26, one target
    ("mixture", 3011, 701, 1e-4, 1e-6, 2, 0, 3, True, True, True),       # npw 32, dipoles
    ("mixture", 3001, 0, 1e-4, 1e-6, 3, 2, 0, False, True, True),         # dipoles only
    ("uniform", 40001, 9000, 3e-4, 1e-9, 1, 1, 2, True, False, True),    # npw 38, plane-wave leaves
    ("uniform", 60013, 501, 3e-4, 1e-9, 1, 3, 1, True, False, True),     # npw 44
    ("uniform", 8000, 2000, 1e-3, 1e-12, 1, 1, 2, True, False, True),    # npw 52: the widest tiles
    ("uniform", 200000, 1000, 1e-2, 1e-6, 1, 1, 1, True, False, False),  # full leaves: leaf by leaf
    # thousands of sources a box and 12 nodes: the serial sum is the longer
    ("uniform", 25401, 2198, 1.6e-2, 1e-3, 1, 0, 2, True, False, False),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_whole_box_route_matches_oracle(case):
    kind, ns, nt, delta, eps, nd, ifs, ift, ifc, ifd, whole = case
    print("case", case, flush=True)
    rng = np.random.default_rng(ns + nt)
    points = _pts.uniform if kind == "uniform" else _pts.mixture
    src = points(rng, ns)
    tg = points(rng, nt) if nt else None
    chg = rng.normal(size=(ns, nd)) if ifc else None
    rn = rng.normal(size=(ns, 2)) if ifd else None
    ds = np.sqrt(delta) * rng.normal(size=(ns, nd)) if ifd else None
    fgt2d_amd.set_timing(True)
    try:
        got = fgt2d_amd.fgt2d(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift,
                              ifdipole=int(ifd), rnormal=rn, dipstr=ds)
        kernels = {k["kernel"] for k in fgt2d_amd.kernel_launches()}
    finally:
        fgt2d_amd.set_timing(False)
    st = fgt2d_amd.last_stats()
    assert st["nlevels"] > max(st["npwlevel"], 0), st  # expansions
    assert ("form_top" in kernels) == whole, (kernels, st)
    want = O.oracle_fgt2d(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift, rnormal=rn,
                          dipstr=ds)
    for k, (g, w) in enumerate(zip(got, want)):
        if (k < 3 and k < ifs) or (k >= 3 and k - 3 < ift):
            g, w = np.asarray(g), np.asarray(w)
            assert np.abs(g - w).max() < 1e-11 * np.abs(w).max(), NAMES[k]


def test_mixed_arithmetic_stays_leaf_by_leaf():
    """The same call, whole boxes in FP64 (third case above), by leaves in the
    mixed mode, whose expansions are half as wide."""
    rng = np.random.default_rng(3)
    src, chg = _pts.uniform(rng, 30011), rng.normal(size=(30011, 1))
    want = O.oracle_fgt2d(5e-4, 1e-6, src, chg)
    for mode, whole, tol in (("fp64", True, 1e-11), ("mixed", False, 2e-5)):
        prev = fgt2d_amd.set_precision(mode)
        fgt2d_amd.set_timing(True)
        try:
            got = fgt2d_amd.fgt2d(5e-4, 1e-6, src, chg)
            kernels = {k["kernel"] for k in fgt2d_amd.kernel_launches()}
            assert fgt2d_amd.last_precision() == mode
            assert ("form_top" in kernels) == whole and ("eval_top" in kernels) == whole, kernels
        finally:
            fgt2d_amd.set_timing(False)
            fgt2d_amd.set_precision(prev)
        assert np.abs(got[0] - want[0]).max() < tol * np.abs(want[0]).max()
