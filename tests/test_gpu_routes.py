"""Both routes of the transforms with expansions, forced by FGTPW_ROUTE.

By leaves: the oracle and golden tests of the other files again, so that the
leaf kernels of every order (formation and conversion up to order 63, the
plane-wave leaves, the chunks) are compared with the oracle also for the
inputs that the route estimate gives to the whole-box kernels.

Against each other: every form a call can have (plane-wave lengths 2 to 58,
charges, dipoles or both, several densities, sources or targets alone,
sparse and dense boxes, a single source) by leaves and by whole boxes.
Tolerance: the same FP64 sums in another order, as the tests against the
oracle."""
import numpy as np
import pytest

import fgt2d_amd
from tests import _pts
from tests import test_gpu3d as g3
from tests import test_gpu_dipole as gd
from tests import test_gpu_golden as gg
from tests import test_gpu_parity as g2

pytestmark = pytest.mark.gpu

NAMES = ["pot", "grad", "hess", "pottarg", "gradtarg", "hesstarg"]


@pytest.fixture
def leaves(monkeypatch):
    monkeypatch.setenv("FGTPW_ROUTE", "leaves")


def _n(cases):
    return dict(argvalues=cases, ids=[str(i) for i in range(len(cases))])


@pytest.mark.parametrize("case", **_n(g3.CASES))
def test_3d_by_leaves_matches_oracle(case, leaves):
    g3.test_fgt3d_matches_oracle(case)


@pytest.mark.parametrize("path", **_n(g3.GOLD3))
def test_3d_by_leaves_matches_golden(path, leaves):
    g3.test_fgt3d_matches_reference_golden(path)


@pytest.mark.parametrize("case", **_n(gd.CASES3))
def test_3d_dipoles_by_leaves_match_oracle(case, leaves):
    gd.test_dipole_transform_3d_matches_oracle(case)


@pytest.mark.parametrize("cap", ["8", "37"])
def test_3d_chunks_by_leaves_match_one_chunk(cap, leaves, monkeypatch):
    g3.test_chunked_expansions_match_one_chunk(cap, monkeypatch)


@pytest.mark.parametrize("case", **_n(g2.CASES))
def test_2d_by_leaves_matches_oracle(case, leaves):
    g2.test_transform_matches_oracle(case)


@pytest.mark.parametrize("path", **_n(gg.GOLD))
def test_2d_by_leaves_matches_golden(path, leaves):
    gg.test_gpu_matches_reference_golden(path)


@pytest.mark.parametrize("case", **_n(gd.CASES))
def test_2d_dipoles_by_leaves_match_oracle(case, leaves):
    gd.test_dipole_transform_matches_oracle(case)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_2d_finest_level_beside_the_tree_by_leaves(precision, leaves):
    g2.test_finest_level_formed_beside_the_tree_is_bit_identical(precision)


# (dim, points, ns, nt, delta, eps, nd, ifpgh, ifpghtarg, charges, dipoles)
FORMS = [
    (2, "uniform", 901, 300, 2.1, 0.1, 1, 1, 1, True, False),      # npw 2, the root alone
    (2, "uniform", 2001, 501, 1.25, 0.02, 2, 1, 1, True, False),   # npw 4
    (2, "uniform", 2003, 33, 0.71, 1e-3, 1, 2, 0, True, False),    # npw 8
    (2, "uniform", 1, 37, 0.71, 1e-3, 1, 0, 1, True, False),       # one source
    (2, "uniform", 5003, 1001, 1e-2, 1e-3, 1, 3, 3, True, True),
    (2, "cluster", 30001, 777, 1e-4, 1e-6, 2, 2, 1, False, True),  # thousands of points a box
    (2, "cluster", 20001, 0, 1e-4, 1e-9, 1, 3, 0, True, True),
    (2, "uniform", 9001, 2003, 1e-3, 1e-9, 3, 1, 2, True, False),
    (2, "uniform", 6007, 600, 1e-3, 1e-12, 1, 2, 3, True, False),  # npw 58
    (3, "uniform", 901, 300, 2.1, 0.1, 1, 1, 1, True, False),      # npw 2, the root alone
    (3, "uniform", 2001, 501, 1.25, 0.02, 2, 1, 1, True, False),   # npw 4
    (3, "uniform", 4003, 33, 0.71, 1e-3, 1, 2, 0, True, False),    # npw 8
    (3, "uniform", 1, 37, 0.71, 1e-3, 1, 0, 1, True, False),       # one source
    (3, "uniform", 5003, 1001, 2e-2, 1e-3, 1, 3, 3, True, True),
    (3, "cluster", 30001, 777, 1e-3, 1e-6, 2, 2, 1, False, True),  # thousands of points a box
    (3, "cluster", 20001, 0, 1e-3, 1e-9, 1, 3, 0, True, True),
    (3, "uniform", 9001, 2003, 2e-2, 1e-9, 3, 1, 2, True, False),
    (3, "uniform", 6007, 600, 2e-2, 1e-13, 1, 1, 1, True, False),  # npw 56, order 86 (plane-wave leaves)
]


def _points(dim, kind, rng, n):
    if kind == "uniform":
        return _pts.uniform(rng, n, dim)
    return np.clip(0.5 + 0.02 * rng.normal(size=(n, dim)), 0.0, 1.0)


@pytest.mark.parametrize("form", **_n(FORMS))
def test_routes_agree(form, monkeypatch):
    dim, kind, ns, nt, delta, eps, nd, ifs, ift, ifc, ifd = form
    print("form", form, flush=True)
    rng = np.random.default_rng(ns)
    src = _points(dim, kind, rng, ns)
    tg = _points(dim, kind, rng, nt) if nt else None
    chg = rng.normal(size=(ns, nd)) if ifc else None
    rn = rng.normal(size=(ns, dim)) if ifd else None
    ds = np.sqrt(delta) * rng.normal(size=(ns, nd)) if ifd else None
    f = fgt2d_amd.fgt2d if dim == 2 else fgt2d_amd.fgt3d
    out = {}
    fgt2d_amd.set_timing(True)
    try:
        for route in ("leaves", "boxes"):
            monkeypatch.setenv("FGTPW_ROUTE", route)
            out[route] = f(delta, eps, src, chg, tg, ifpgh=ifs, ifpghtarg=ift, ifdipole=int(ifd),
                           rnormal=rn, dipstr=ds)
            kernels = {k["kernel"] for k in fgt2d_amd.kernel_launches()}
            st = fgt2d_amd.last_stats()
            assert st["nlevels"] > st["npwlevel"] and st["npw"] >= 2, st
            assert ("form_top" in kernels) == (route == "boxes"), (kernels, st)
            print(route, st, flush=True)
    finally:
        fgt2d_amd.set_timing(False)
    for k in range(6):
        if (k < 3 and k < ifs) or (k >= 3 and k - 3 < ift):
            g, w = np.asarray(out["boxes"][k]), np.asarray(out["leaves"][k])
            assert np.abs(g - w).max() < 1e-11 * np.abs(w).max(), NAMES[k]
