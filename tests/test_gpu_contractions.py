"""The tiled contractions at the edges of their tiles: leaves of fewer points
than a chunk or a block, AO counts around the 16- and 32-row tile steps, one
to four blocks per leaf, every form (LDA, GGA, meta-GGA; one spin and two)
and both storage precisions, against the CPU oracle.

Bounds on Vxc in FP64: each leaf drops at most two terms below 1e-14 per
entry (none for a meta-GGA) and the sums round at 1e-15 of the
largest entry per leaf, so 2e-14 leaves + 1e-13 max|V|, below 1e-11 here.
FP32 AO storage rounds each value by 6e-8 relative: 1e-7 max|V|, the bound of
the batch tests."""
import numpy as np
import pytest

import oracle
from conftest import random_density
from occ_amd import AOBasis, molecules
from occ_amd.dft import XCContext, functional_ids
from occ_amd.grid import GridSettings, MolecularGrid

pytestmark = pytest.mark.gpu

SYSTEMS = {"water": lambda: molecules.water(), "methane": lambda: molecules.alkane(1),
           "water3": lambda: molecules.water_cluster(3, seed=6),
           "alkane3": lambda: molecules.alkane(3), "alkane5": lambda: molecules.alkane(5)}


def _setup(system, basis_name, method, precision, tile, nrad=19, nang=38):
    atoms = SYSTEMS[system]()
    basis = AOBasis.load(atoms, basis_name, pure=basis_name.startswith("def2"))
    pts, wts = MolecularGrid(atoms, GridSettings(radial_points=nrad, angular_points=nang)).build()
    print(f"{system} {basis_name} {method} {precision} tile {tile}: nbf={basis.nbf} "
          f"npts={len(wts)}", flush=True)
    ctx = XCContext(basis, pts, wts, functional_ids(method), precision=precision, tile_ao=tile)
    return basis, pts, wts, ctx


def _bound(precision, V):
    return 1e-11 if precision == "fp64" else 1e-7 * np.abs(V).max()


@pytest.mark.parametrize("precision", ["fp64", "fp32cache"])
@pytest.mark.parametrize("method", ["svwn5", "pbe", "tpss"])
@pytest.mark.parametrize("system,basis_name,tile", [
    ("water", "6-31g", 0), ("water", "def2-svp", 0), ("methane", "6-31g(d,p)", 32),
    ("water3", "def2-svp", 64), ("water3", "def2-tzvp", 0), ("alkane5", "def2-svp", 96),
    ("alkane5", "6-31g", 0)])
def test_build_matches_oracle(system, basis_name, tile, method, precision):
    basis, pts, wts, ctx = _setup(system, basis_name, method, precision, tile)
    D = random_density(basis.nbf, 5, 17)
    K, exc, nel = oracle.xc_build(oracle.OracleBasis.from_flat(basis.flat()), pts, wts,
                                  functional_ids(method), D)
    for _ in range(2):
        V, e, n = ctx.build(D)
        assert np.abs(V - K).max() <= _bound(precision, K)
        assert abs(e - exc) <= (1e-11 if precision == "fp64" else 1e-6)
        assert abs(n - nel) <= (1e-11 if precision == "fp64" else 1e-6)
    ctx.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32cache"])
@pytest.mark.parametrize("method", ["svwn5", "blyp", "tpss"])
@pytest.mark.parametrize("system,basis_name,tile", [
    ("water", "6-31g", 0), ("methane", "def2-svp", 32), ("water3", "def2-tzvp", 0),
    ("alkane5", "def2-svp", 64)])
def test_unrestricted_build_matches_oracle(system, basis_name, tile, method, precision):
    basis, pts, wts, ctx = _setup(system, basis_name, method, precision, tile)
    # each spin block is read in full: an unsymmetric perturbation enters as it is
    r = np.random.default_rng(3)
    D = np.concatenate([random_density(basis.nbf, 5, 21), random_density(basis.nbf, 4, 22)]) / 2
    D = np.asfortranarray(D + 1e-3 * r.normal(size=D.shape) * np.abs(D))
    K, exc, nel = oracle.xc_build_unrestricted(oracle.OracleBasis.from_flat(basis.flat()), pts,
                                               wts, functional_ids(method), D)
    V, e, n = ctx.build_unrestricted(D)
    assert np.abs(V - K).max() <= _bound(precision, K)
    assert abs(e - exc) <= (1e-11 if precision == "fp64" else 1e-6)
    assert np.abs(np.array(n) - np.array(nel)).max() <= (1e-11 if precision == "fp64" else 1e-6)
    ctx.close()


# gradients: sums over the leaf points of values up to ~1e2 (core derivatives),
# rounded at 1e-15 of them: 1e-11; FP32 storage 6e-8 of an entry, 1e-6 in all
@pytest.mark.parametrize("precision", ["fp64", "fp32cache"])
@pytest.mark.parametrize("method", ["svwn5", "pbe", "tpss"])
@pytest.mark.parametrize("system,basis_name", [
    ("water", "6-31g"), ("methane", "def2-svp"), ("water3", "def2-tzvp"), ("alkane5", "6-31g")])
def test_gradients_match_oracle(system, basis_name, method, precision):
    basis, pts, wts, ctx = _setup(system, basis_name, method, precision, 0)
    ob, n = oracle.OracleBasis.from_flat(basis.flat()), len(basis.atoms)
    tol = 1e-11 if precision == "fp64" else 1e-6
    D = random_density(basis.nbf, 5, 31)
    G = oracle.xc_gradient(ob, basis.shell_atom, n, pts, wts, functional_ids(method), D)
    first = ctx.xc_gradient(D, basis.shell_atom, n)
    assert np.abs(first - G).max() <= tol * max(1.0, np.abs(G).max())
    assert np.array_equal(first, ctx.xc_gradient(D, basis.shell_atom, n))
    Du = np.asfortranarray(np.concatenate([D, random_density(basis.nbf, 4, 32)]) / 2)
    Gu = oracle.xc_gradient_unrestricted(ob, basis.shell_atom, n, pts, wts,
                                         functional_ids(method), Du)
    got = ctx.xc_gradient_unrestricted(Du, basis.shell_atom, n)
    assert np.abs(got - Gu).max() <= tol * max(1.0, np.abs(Gu).max())
    ctx.close()


# the same with column blocks of 32 AOs whose second half holds real ones: one
# block of 17 to 32 AOs, and for a meta-GGA 64 + 32 with more than 80
@pytest.mark.parametrize("precision", ["fp64", "fp32cache"])
@pytest.mark.parametrize("method", ["svwn5", "pbe", "tpss"])
@pytest.mark.parametrize("system,basis_name", [
    ("methane", "6-31g"), ("water", "def2-svp"), ("alkane3", "def2-svp")])
def test_gradients_of_blocks_of_32(system, basis_name, method, precision):
    test_gradients_match_oracle(system, basis_name, method, precision)


# VV10: one pass over several segments of j, points within and beyond the range
# whose pairs share a reciprocal (atoms 1500 Bohr apart, a tiny b).  The sums run
# in another order than the oracle's: 1e-12 of E; Vxc as a build's, plus the
# rounding of 1e4 pair terms relative to its largest entry.
@pytest.mark.parametrize("shift,b", [(0.0, 6.0), (1500.0, 6.0), (0.0, 1e-6), (3.0, 1e-9)])
@pytest.mark.parametrize("nrad,nang", [(8, 26), (40, 50)])
def test_vv10_matches_oracle(shift, b, nrad, nang):
    atoms = molecules.water()
    if shift:
        atoms = atoms + [(z, x + shift, y, w) for z, x, y, w in molecules.water()]
    basis = AOBasis.load(atoms, "6-31g")
    pts, wts = MolecularGrid(atoms, GridSettings(radial_points=nrad, angular_points=nang)).build()
    print(f"vv10 shift {shift} b {b} npts={len(wts)}", flush=True)
    D = random_density(basis.nbf, 5, 41)
    e, V = oracle.vv10(oracle.OracleBasis.from_flat(basis.flat()), pts, wts, D, b=b, C=0.01)
    ctx = XCContext(basis, pts, wts, functional_ids("pbe"))
    got, K = ctx.nlc_vv10(D, b=b, C=0.01)
    ctx.close()
    assert abs(got - e) <= 1e-12 * abs(e)
    assert np.abs(K - V).max() <= 1e-11 + 1e-11 * np.abs(V).max()


# More than 32,768 points, where segments of j are longer than eight tiles: 135
# tiles (15 segments of 9, the last block's second tile missing) and 136, the
# last input points next to the nuclei.  Bounds as above.
@pytest.mark.parametrize("npts", [34305, 34400, 34816])
def test_vv10_segments_with_live_last_points(npts):
    atoms = molecules.water()
    basis = AOBasis.load(atoms, "6-31g")
    pts, wts = MolecularGrid(atoms, GridSettings(radial_points=75, angular_points=302)).build()
    d = np.min([np.linalg.norm(pts - np.array(a[1:]), axis=1) for a in atoms], axis=0)
    near = np.argsort(-d, kind="stable")[-npts:]  # the nearest npts points, far to near
    pts, wts = np.ascontiguousarray(pts[near]), np.ascontiguousarray(wts[near])
    print(f"vv10 npts={len(wts)}", flush=True)
    D = random_density(basis.nbf, 5, 43)
    e, V = oracle.vv10(oracle.OracleBasis.from_flat(basis.flat()), pts, wts, D, b=6.0, C=0.01)
    ctx = XCContext(basis, pts, wts, functional_ids("pbe"))
    got, K = ctx.nlc_vv10(D, b=6.0, C=0.01)
    ctx.close()
    assert abs(got - e) <= 1e-12 * abs(e)
    assert np.abs(K - V).max() <= 1e-11 + 1e-11 * np.abs(V).max()


# A meta-GGA's potential is added in full: with weights of 1e-16 of a grid's all
# entries are that small, and none may be left out (1e-11 of the largest, as
# above).
@pytest.mark.parametrize("tile", [0, 32, 64])
@pytest.mark.parametrize("precision", ["fp64", "fp32cache"])
def test_meta_gga_potential_is_added_in_full(precision, tile):
    basis, pts, wts, ctx = _setup("water3", "def2-svp", "tpss", precision, tile)
    ctx.close()
    wts = 1e-16 * wts
    ctx = XCContext(basis, pts, wts, functional_ids("tpss"), precision=precision, tile_ao=tile)
    D = random_density(basis.nbf, 5, 17)
    ob, ids = oracle.OracleBasis.from_flat(basis.flat()), functional_ids("tpss")
    tol = 1e-11 if precision == "fp64" else 1e-7
    K = oracle.xc_build(ob, pts, wts, ids, D)[0]
    assert np.abs(ctx.build(D)[0] - K).max() <= tol * np.abs(K).max()
    Du = np.asfortranarray(np.concatenate([D, random_density(basis.nbf, 4, 22)]) / 2)
    K = oracle.xc_build_unrestricted(ob, pts, wts, ids, Du)[0]
    assert np.abs(ctx.build_unrestricted(Du)[0] - K).max() <= tol * np.abs(K).max()
    ctx.close()


# The host entry points keep one 2 nbf x nbf matrix beside what the device ones
# keep (allocated whole or not at all), D going in and Vxc coming out of it.
@pytest.mark.parametrize("method", ["pbe", "tpss"])
def test_unrestricted_host_build_keeps_one_matrix(method):
    from occ_amd.device import DeviceArray
    basis, pts, wts, ctx = _setup("water3", "6-31g", method, "fp64", 0)
    n = basis.nbf
    D = np.asfortranarray(np.concatenate([random_density(n, 5, 21), random_density(n, 4, 22)]) / 2)
    dD, dV, dr = DeviceArray(2 * n * n), DeviceArray(2 * n * n), DeviceArray(3)
    dD.upload(D)
    ctx.build_unrestricted_device(dD.ptr, dV.ptr, dr.ptr)
    ctx.synchronize()
    on_device = ctx.info()["device_bytes"]
    first, second = ctx.build_unrestricted(D), ctx.build_unrestricted(D)
    assert ctx.info()["device_bytes"] - on_device == 16 * n * n
    # FP64 atomics: equal to rounding
    for V, e, nel in (first, second):
        assert np.abs(V - dV.download((2 * n, n))).max() <= 1e-13
        assert [e, *nel] == list(dr.download())
    ctx.close()
