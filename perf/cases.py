"""What the performance of this framework is measured on: XC builds, gradients,
non-local correlation and set-up through the entry points that an SCF program
calls, from one water molecule to (H2O)128.

A case names a path and its sizes:

  path       what runs (see `run`): "build" (restricted build on device buffers),
             "host" (DFT.compute_vxc on host arrays), "uks" (unrestricted build),
             "gradient" / "ugradient" (XC nuclear gradient), "vv10" (non-local
             correlation), "batch" (many molecules in one context), "geometry"
             (grid, context and first build of a new geometry)
  family, n  water cluster of n molecules or alkane with n carbons
             (a batch: n molecules of 1..`top` units of both families)
  basis, method, precision, radial, angular   as the entry points take them

Inputs come from the seed alone: the geometry (water clusters), and a density
C C^T of orthonormal orbitals that are localised on the atoms.  `exact` is the
same mathematics in 64-bit torch: dense AO values, spin-resolved energy
densities, and automatic differentiation for the potentials and gradients.
"""
import functools
import math
import random

import numpy as np
import torch

from occ_amd import AOBasis, alkane, water_cluster
from occ_amd.dft import DFT, XCBatch, XCContext, functional_ids, grid_hierarchy
from occ_amd.grid import GridSettings, MolecularGrid

BASES = {"sto-3g": False, "6-31g": False, "6-31g(d,p)": False, "def2-svp": True,
         "def2-tzvp": True}  # name: spherical


def _case(name, path, family, n, basis, method, precision, radial, angular, top=0):
    return dict(name=name, path=path, family=family, n=n, basis=basis, method=method,
                precision=precision, radial=radial, angular=angular, top=top)


def listed():
    return [
        # the smallest build there is, as in the inner loop of a small molecule's
        # SCF: launches and latency
        _case("water_svwn5", "build", "water", 1, "6-31g", "svwn5", "fp64", 75, 302),
        # one SCF iteration of a host program on a small molecule: host arrays in
        # and out, a wait at its end, Cartesian d shells
        _case("dimer_pbe_host", "host", "water", 2, "6-31g(d,p)", "pbe", "fp64", 75, 302),
        # the ordinary production build in full precision
        _case("water32_pbe_fp64", "build", "water", 32, "def2-svp", "pbe", "fp64", 75, 302),
        # the largest: the cluster build of the benchmark, in the mode it is quoted in
        _case("water128_blyp_fp32", "build", "water", 128, "def2-svp", "blyp", "fp32", 75, 302),
        # a long chain (elongated leaves, other screening) with 32-bit AO storage
        _case("alkane30_blyp_fp32cache", "build", "alkane", 30, "def2-svp", "blyp", "fp32cache",
              75, 302),
        # many small molecules at once, replayed as a graph (data generation)
        _case("batch24_pbe_fp32", "batch", "mixed", 24, "def2-svp", "pbe", "fp32", 50, 194, 16),
        # open shells: both spins' densities and potentials
        _case("water32_uks_pbe", "uks", "water", 32, "def2-svp", "pbe", "fp64", 75, 302),
        # meta-GGA: three more contractions per stage
        _case("water32_tpss", "build", "water", 32, "def2-svp", "tpss", "fp64", 75, 302),
        # a geometry optimisation's step: the XC nuclear gradient
        _case("water32_pbe_gradient", "gradient", "water", 32, "def2-svp", "pbe", "fp64", 75, 302),
        # the same for a radical with a meta-GGA: every gradient term there is
        _case("alkane11_tpss_ugradient", "ugradient", "alkane", 11, "def2-svp", "tpss", "fp64",
              50, 194),
        # VV10 on its own coarser grid: the sum over point pairs
        _case("water16_vv10", "vv10", "water", 16, "def2-svp", "pbe", "fp64", 50, 110),
        # what a new geometry costs before its second iteration: Becke grid, leaf
        # layout, AO values (f shells) and the first build
        _case("water5_tzvp_geometry", "geometry", "water", 5, "def2-tzvp", "pbe", "fp64", 50, 194),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    path = rng.choice(["build", "build", "build", "host", "batch", "uks", "build", "gradient",
                       "ugradient", "vv10", "geometry"])
    family = rng.choice(["water", "water", "alkane"])
    method = rng.choice(["svwn5", "pbe", "blyp", "bpbe", "tpss"])
    radial, angular = rng.choice([(75, 302), (50, 194), (40, 110), (61, 146), (75, 302)])
    precision = rng.choice(["fp64", "fp64", "fp32cache", "fp32"])
    basis = rng.choice(["def2-svp", "def2-svp", "6-31g", "6-31g(d,p)", "def2-tzvp"])
    top, hi = 0, 48
    if path == "batch":
        family, top, n = "mixed", rng.choice([3, 8, 16]), _log_int(rng, 3, 32)
    else:
        if path == "vv10":
            radial, angular, hi = 50, rng.choice([50, 74, 110]), 24
        elif path == "geometry":
            hi = 16
        elif path in ("uks", "gradient", "ugradient") or method == "tpss":
            hi = 32
        if basis == "def2-tzvp":
            hi = min(hi, 12)
        n = _log_int(rng, 1, hi)
    # FP32 contractions are for restricted LDA / GGA builds
    if precision == "fp32" and (method == "tpss" or path not in ("build", "host", "batch")):
        precision = "fp32cache"
    if path == "vv10" and method == "svwn5":
        method = "pbe"
    c = _case("", path, family, n, basis, method, precision, radial, angular, top)
    del c["name"]
    return c


# --- inputs -----------------------------------------------------------------


def _molecules(case, seed):
    """[(atoms, basis name)] of a case."""
    rng = random.Random(seed)
    if case["path"] != "batch":
        n = case["n"]
        atoms = alkane(n) if case["family"] == "alkane" else water_cluster(n, seed=seed)
        return [(atoms, case["basis"])]
    out = []
    for i in range(case["n"]):
        # sizes are the case's, so that another seed is the same amount of work
        units = 1 + (i * 5 + 2) % case["top"]
        atoms = alkane(units) if i % 2 else water_cluster(units, seed=rng.randrange(1 << 30))
        out.append((atoms, case["basis"] if i % 4 < 2 else "6-31g"))
    return out


def _basis(atoms, name):
    return AOBasis.load(atoms, name, pure=BASES[name])


def _grid(case, atoms):
    return MolecularGrid(atoms, GridSettings(radial_points=case["radial"] + 1,
                                             angular_points=case["angular"]))


def _orbitals(basis, nocc, seed):
    """nocc orthonormal orbitals, each localised on one of the atoms."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rng = np.random.default_rng(seed)
    xyz = np.array([a[1:] for a in basis.atoms])
    of = np.concatenate([[a] * s.size() for a, s in zip(basis.shell_atom, basis.shells)])
    d = np.linalg.norm(xyz[of][:, None] - xyz[np.arange(nocc) % len(xyz)][None], axis=2)
    C = torch.from_numpy(rng.normal(size=d.shape) * np.exp(-0.5 * d)).to(dev)
    e, U = torch.linalg.eigh(C.T @ C)
    return C @ (U * e.clamp_min(1e-12).rsqrt()) @ U.T


def _occupied(basis):
    return max(1, min(basis.nbf, sum(int(a[0]) for a in basis.atoms) // 2))


def _density(basis, seed):
    """D = C C^T, symmetric."""
    C = _orbitals(basis, _occupied(basis), seed)
    return C @ C.T


def _spin_densities(basis, seed):
    """C_s C_s^T / 2 of a cation: one beta electron fewer."""
    n = _occupied(basis)
    C = _orbitals(basis, n, seed)
    A = torch.from_numpy(np.random.default_rng(seed + 1).normal(size=(n, n))).to(C.device)
    B = C @ torch.linalg.qr(A)[0][:, :max(n - 1, 1)]
    return 0.5 * C @ C.T, 0.5 * B @ B.T


@functools.lru_cache(maxsize=1)
def _stream():
    """The program's own stream, which its builds are queued on."""
    return torch.cuda.Stream()


def _buffer(n):
    return torch.zeros(int(n), dtype=torch.float64, device="cuda")


def prepare(case, seed):
    path = case["path"]
    mols = _molecules(case, seed)
    ids = functional_ids(case["method"])
    bases = [_basis(*m) for m in mols]
    b = bases[0]
    st = {"path": path, "basis": b}
    if path == "geometry":
        st.update(case=dict(case), ids=ids, D=_density(b, seed).cpu().numpy())
        return st
    grids = [_grid(case, m[0]).build() for m in mols]
    st["stream"] = _stream().cuda_stream
    if path == "batch":
        ctx = XCBatch(bases, grids, ids, precision=case["precision"])
        ctx.set_graph(True)
        D = torch.cat([_density(x, seed + i).reshape(-1) for i, x in enumerate(bases)])
        st.update(ctx=ctx, D=D.cuda(), V=_buffer(D.numel()), r=_buffer(2 * len(mols)))
        return st
    pts, wts = grids[0]
    if path == "host":
        st["dft"] = DFT(case["method"], b, pts, wts, precision=case["precision"])
        st["D"] = np.asfortranarray(_density(b, seed).cpu().numpy())
        return st
    st["ctx"] = XCContext(b, pts, wts, ids, precision=case["precision"])
    if path in ("uks", "ugradient"):
        da, db = _spin_densities(b, seed)
        # 2 nbf x nbf column-major, alpha block over beta block
        st["D"] = torch.cat([da, db], dim=1).contiguous().cuda()
        st["V"], st["r"] = _buffer(2 * b.nbf ** 2).view(b.nbf, 2 * b.nbf), _buffer(3)
    else:
        st["D"] = _density(b, seed).contiguous().cuda()
        st["V"], st["r"] = _buffer(b.nbf ** 2).view(b.nbf, b.nbf), _buffer(2)
    st["G"] = _buffer(3 * len(b.atoms)).view(len(b.atoms), 3)
    return st


def run(st):
    path, b = st["path"], st["basis"]
    if path == "geometry":
        case = st["case"]
        pts, wts = _grid(case, b.atoms).build()
        ctx = XCContext(b, pts, wts, st["ids"], precision=case["precision"])
        V, exc, nel = ctx.build(st["D"])
        ctx.close()
        return {"weights": wts, "vxc": V, "scalars": [exc, nel]}
    if path == "host":
        V = st["dft"].compute_vxc(st["D"])
        return {"vxc": V, "scalars": [st["dft"].exchange_correlation_energy(),
                                      st["dft"].total_density()]}
    ctx, s = st["ctx"], st["stream"]
    D = st["D"].data_ptr()
    if path in ("gradient", "ugradient"):
        call = ctx.xc_gradient_device if path == "gradient" else ctx.xc_gradient_unrestricted_device
        call(D, b.shell_atom, len(b.atoms), st["G"].data_ptr(), stream=s)
        return {"gradient": st["G"]}
    V, r = st["V"].data_ptr(), st["r"].data_ptr()
    if path == "uks":
        ctx.build_unrestricted_device(D, V, r, stream=s)
    elif path == "vv10":
        ctx.nlc_vv10_device(D, V, r, stream=s)
    else:
        ctx.build_device(D, V, r, stream=s)
    return {"vxc": st["V"], "scalars": st["r"]}


def tolerance(case):
    # sums of up to 1e7 terms in 64 bits, in another order; FP32 AO values differ
    # by their rounding (6e-8 each, averaged over the points)
    if case["precision"] == "fp64":
        return {"rel": 1e-11, "max": 1e-9}
    return {"rel": 1e-6, "max": 1e-4}


# --- work -------------------------------------------------------------------


def _extents(basis, threshold=1e-10):
    """Distance at which each shell's values fall below the threshold (Bohr)."""
    r = np.arange(0.5, 30.0, 0.1)
    out = []
    for s in basis.shells:
        v = np.abs(s.coefficients @ np.exp(-s.exponents[:, None] * r * r)) * r ** s.l
        above = np.nonzero(v > threshold)[0]
        out.append(r[above[-1]] if len(above) else 0.5)
    return np.array(out)


@functools.lru_cache(maxsize=64)
def _sums(key):
    """(points, nbf^2, atoms, sum n m, sum n m^2) over the 128-point leaves of a
    case's grids, m the AOs that reach a leaf."""
    case = dict(key)
    npts = nn = nat = n1 = n2 = 0.0
    for atoms, name in _molecules(case, 0):
        b = _basis(atoms, name)
        pts, wts, _ = _grid(case, atoms).unpartitioned()
        h = grid_hierarchy(pts, wts)
        R = np.array([s.origin for s in b.shells])
        ext, size = _extents(b), np.array([float(s.size()) for s in b.shells])
        cnt, rad = h["count"].astype(float), h["radius"]
        for lo in range(0, len(cnt), 4096):
            c = h["center"][lo:lo + 4096]
            d2 = (c * c).sum(1)[:, None] + (R * R).sum(1)[None] - 2.0 * c @ R.T
            reach = np.sqrt(np.maximum(d2, 0.0)) - ext[None] < rad[lo:lo + 4096, None]
            m = reach @ size
            n1 += float((cnt[lo:lo + 4096] * m).sum())
            n2 += float((cnt[lo:lo + 4096] * m * m).sum())
        npts, nn, nat = npts + len(wts), nn + b.nbf ** 2, nat + len(atoms)
    return npts, nn, nat, n1, n2


def work(case):
    path, method = case["path"], case["method"]
    npts, nn, nat, n1, n2 = _sums(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    lda, mgga = method == "svwn5", method == "tpss"
    spins = 2 if path in ("uks", "ugradient") else 1
    comps = 1 if lda else 4
    size = 8 if case["precision"] == "fp64" else 4
    # matrix products of 2 n m^2 per leaf; symmetric ones (an LDA's, and those of
    # tau) need half of that
    density = 1.0 * n2 if lda else 2.0 * n2
    vxc = 1.0 * n2 if lda else 2.0 * n2
    if mgga:
        density, vxc = density + 3.0 * n2, vxc + 3.0 * n2
    flops, extra = spins * (density + vxc), 0.0
    if path in ("gradient", "ugradient"):
        # phi P is the density's; the derivative rows' product and, for tau, the
        # full products of the three planes
        flops = spins * (2.0 * n2 + (0.0 if lda else 2.0 * n2) + (6.0 * n2 if mgga else 0.0))
        extra = (3 if lda else 6) * 8.0 * n1
        nn = nn / 2.0
    elif path == "vv10":
        flops = 4.0 * n2 + 27.0 * npts * (npts - 1) / 2.0
    elif path == "geometry":
        flops += 12.0 * npts * nat * nat
        extra = 64.0 * npts
    return {"bytes": comps * size * n1 + extra + 16.0 * spins * nn + 32.0 * npts, "flops": flops}


# --- 64-bit reference ---------------------------------------------------------

_S = math.sqrt
# components of a shell as sums of c x^i y^j z^k, spherical m = -l..l (Racah)
_SPH = {0: [[(1.0, 0, 0, 0)]],
        1: [[(1.0, 0, 1, 0)], [(1.0, 0, 0, 1)], [(1.0, 1, 0, 0)]],
        2: [[(_S(3), 1, 1, 0)], [(_S(3), 0, 1, 1)],
            [(1.0, 0, 0, 2), (-0.5, 2, 0, 0), (-0.5, 0, 2, 0)],
            [(_S(3), 1, 0, 1)], [(_S(3) / 2, 2, 0, 0), (-_S(3) / 2, 0, 2, 0)]],
        3: [[(3 * _S(5 / 8), 2, 1, 0), (-_S(5 / 8), 0, 3, 0)], [(_S(15), 1, 1, 1)],
            [(4 * _S(3 / 8), 0, 1, 2), (-_S(3 / 8), 2, 1, 0), (-_S(3 / 8), 0, 3, 0)],
            [(1.0, 0, 0, 3), (-1.5, 2, 0, 1), (-1.5, 0, 2, 1)],
            [(4 * _S(3 / 8), 1, 0, 2), (-_S(3 / 8), 3, 0, 0), (-_S(3 / 8), 1, 2, 0)],
            [(_S(15) / 2, 2, 0, 1), (-_S(15) / 2, 0, 2, 1)],
            [(_S(5 / 8), 3, 0, 0), (-3 * _S(5 / 8), 1, 2, 0)]]}
_CART = {l: [[(1.0, i, j, l - i - j)] for i in range(l, -1, -1) for j in range(l - i, -1, -1)]
         for l in range(4)}


class _AOs:
    """phi and grad phi of a basis at points, differentiable in the centres."""

    def __init__(self, basis, dev):
        first = basis.first_bf()
        groups = {}
        for k, s in enumerate(basis.shells):
            groups.setdefault((s.l, s.pure, len(s.exponents)), []).append(k)
        self.groups, order = [], []
        t = functools.partial(torch.tensor, dtype=torch.float64, device=dev)
        for (l, pure, _), ks in groups.items():
            fac = _S((2 * l + 1) / (4 * math.pi)) if pure or l < 2 else 1.0
            comp = _SPH[l] if pure else _CART[l]
            a = t(np.array([basis.shells[k].exponents for k in ks]))
            c = t(np.array([basis.shells[k].coefficients for k in ks])) * fac
            at = torch.tensor([basis.shell_atom[k] for k in ks], device=dev)
            self.groups.append((comp, a, c, at))
            order += [first[k] + q for q in range(len(comp)) for k in ks]
        self.inv = torch.argsort(torch.tensor(order, device=dev))

    def __call__(self, pts, centres, deriv):
        out = [[] for _ in range(4 if deriv else 1)]
        for comp, a, c, at in self.groups:
            d = pts[:, None, :] - centres[at][None]
            e = c * torch.exp(-a * (d * d).sum(-1, keepdim=True))
            R = e.sum(-1)
            R1 = (-2.0 * a * e).sum(-1) if deriv else None
            pw = [[None, d[..., k], d[..., k] ** 2, d[..., k] ** 3] for k in range(3)]

            def mono(p):
                v = None
                for k in range(3):
                    if p[k]:
                        v = pw[k][p[k]] if v is None else v * pw[k][p[k]]
                return torch.ones_like(R) if v is None else v

            for terms in comp:
                S = sum(q * mono(p) for q, *p in terms)
                out[0].append(S * R)
                for k in range(3 if deriv else 0):
                    g = S * d[..., k] * R1
                    for q, *p in terms:
                        if p[k]:
                            low = [x - (j == k) for j, x in enumerate(p)]
                            g = g + q * p[k] * mono(low) * R
                    out[k + 1].append(g)
        return [torch.cat(o, 1)[:, self.inv] for o in out]


def _limit(x, lo=None, hi=None):
    """x held between lo and hi, its derivative kept."""
    y = x if lo is None else torch.maximum(x, torch.as_tensor(lo, dtype=x.dtype, device=x.device))
    y = y if hi is None else torch.minimum(y, hi)
    return x + (y - x).detach()


_PI = math.pi
_CX = 0.75 * (3.0 / _PI) ** (1.0 / 3.0)
_BETA, _GAMMA = 0.06672455060314922, (1.0 - math.log(2.0)) / _PI ** 2


def _opz(x, p):
    return x.clamp_min(2.220446049250313e-16) ** p


def _f_zeta(z):
    return (_opz(1 + z, 4 / 3) + _opz(1 - z, 4 / 3) - 2) / (2 ** (4 / 3) - 2)


def _interpolate(rs, z, e0, e1, ac, fpp):
    f, z4 = _f_zeta(z), z ** 4
    return e0 + ac * f * (1 - z4) / fpp + (e1 - e0) * f * z4


def _pw92(rs, z):
    def G(A, a1, b1, b2, b3, b4):
        s = rs.sqrt()
        return -2 * A * (1 + a1 * rs) * torch.log1p(
            1 / (2 * A * (b1 * s + b2 * rs + b3 * rs * s + b4 * rs * rs)))
    return _interpolate(rs, z, G(0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294),
                        G(0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517),
                        -G(0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671),
                        1.709920934161365617563962776245)


def _vwn5(rs, z):
    def V(A, b, c, x0):
        x = rs.sqrt()
        X, X0, Q = x * x + b * x + c, x0 * x0 + b * x0 + c, _S(4 * c - b * b)
        at = torch.atan(Q / (2 * x + b))
        return A * (torch.log(x * x / X) + 2 * b / Q * at - b * x0 / X0 * (
            torch.log((x - x0) ** 2 / X) + 2 * (b + 2 * x0) / Q * at))
    return _interpolate(rs, z, V(0.0310907, 3.72744, 12.9352, -0.10498),
                        V(0.01554535, 7.06042, 18.0578, -0.32500),
                        V(-1 / (6 * _PI ** 2), 1.13107, 13.0045, -0.0047584),
                        4 / (9 * (2 ** (1 / 3) - 1)))


def _pbe_c(ra, rb, sig):
    """n eps_c of PBE."""
    n = ra + rb
    z = (ra - rb) / n
    ec = _pw92((3 / (4 * _PI * n)) ** (1 / 3), z)
    phi = 0.5 * (_opz(1 + z, 2 / 3) + _opz(1 - z, 2 / 3))
    t2 = sig / (4 * phi ** 2 * (4 / _PI) * (3 * _PI ** 2 * n) ** (1 / 3) * n * n)
    A = _BETA / _GAMMA / torch.expm1(-ec / (_GAMMA * phi ** 3))
    At = A * t2
    H = _GAMMA * phi ** 3 * torch.log1p(_BETA / _GAMMA * t2 * (1 + At) / (1 + At + At * At))
    return n * (ec + H)


def _lyp(ra, rb, saa, sab, sbb):
    a, b, c, d = 0.04918, 0.132, 0.2533, 0.349
    cf = 0.3 * (3 * _PI ** 2) ** (2 / 3)
    n, g = ra + rb, saa + 2 * sab + sbb
    r = n ** (-1 / 3)
    den = 1 + d * r
    om = torch.exp(-c * r) / den * n ** (-11 / 3)
    de = c * r + d * r / den
    q = ra * rb * (2 ** (11 / 3) * cf * (ra ** (8 / 3) + rb ** (8 / 3)) +
                   (47 / 18 - 7 / 18 * de) * g - (2.5 - de / 18) * (saa + sbb) -
                   (de - 11) / 9 * (ra / n * saa + rb / n * sbb))
    q = q - 2 / 3 * n * n * g + (2 / 3 * n * n - ra * ra) * sbb + (2 / 3 * n * n - rb * rb) * saa
    return -4 * a / den * ra * rb / n - a * b * om * q


def _exchange(kind, r, s, t):
    """One spin's exchange energy, E_x[2 r, 4 s, 2 t] / 2."""
    n = 2 * r
    lda = -_CX * n ** (4 / 3)
    if kind == "lda":
        return 0.5 * lda
    if kind == "b88":
        r43 = r ** (4 / 3)
        x = s.sqrt() / r43
        return 0.5 * lda - 0.0042 * r43 * x * x / (1 + 6 * 0.0042 * x * torch.asinh(x))
    p = 4 * s / (4 * (3 * _PI ** 2) ** (2 / 3) * n ** (8 / 3))
    k = 0.804
    if kind == "pbe":
        return 0.5 * lda * (1 + k - k / (1 + _BETA * _PI ** 2 / 3 * p / k))
    b, c, e, mu, ge = 0.40, 1.59096, 1.537, 0.21951, 10 / 81
    sig, tau = 4 * s, 2 * t
    tw = sig / (8 * n)
    z = tw / tau
    al = (tau - tw) / (0.3 * (3 * _PI ** 2) ** (2 / 3) * n ** (5 / 3))
    qb = 0.45 * (al - 1) / (1 + b * al * (al - 1)).sqrt() + 2 * p / 3
    z2 = z * z
    x = ((ge + c * z2 / (1 + z2) ** 2) * p + 146 / 2025 * qb ** 2 -
         73 / 405 * qb * (0.5 * (9 / 25 * z2 + p * p)).sqrt() + ge * ge / k * p * p +
         2 * _S(e) * ge * 9 / 25 * z2 + e * mu * p ** 3) / (1 + _S(e) * p) ** 2
    return 0.5 * lda * (1 + k - k / (1 + x / k))


def _tpss_c(ra, rb, saa, sab, sbb, ta, tb):
    n = ra + rb
    zeta = (ra - rb) / n
    sig = saa + 2 * sab + sbb
    ep = _pbe_c(ra, rb, sig) / n
    zero = torch.zeros_like(ra)
    par = 0.0
    for r, s in ((ra, saa), (rb, sbb)):
        e = _pbe_c(r, zero, s) / r
        par = par + r / n * torch.where(e > ep, e, ep)
    z = _limit(sig / (8 * n * (ta + tb)), None, torch.ones_like(n))
    xi2 = (4 * (rb * rb * saa - 2 * ra * rb * sab + ra * ra * sbb) / n ** 4 /
           (4 * (3 * _PI ** 2 * n) ** (2 / 3)))
    q = zeta * zeta
    C = (0.53 + 0.87 * q + 0.5 * q * q + 2.26 * q ** 3) / (
        1 + xi2 * (_opz(1 + zeta, -4 / 3) + _opz(1 - zeta, -4 / 3)) / 2) ** 4
    f = (1 + C * z * z) * ep - (1 + C) * z * z * par
    return n * f * (1 + 2.8 * f * z ** 3)


def _energy_density(method, ra, rb, saa, sab, sbb, ta, tb):
    """n eps_xc of a spin-polarised density."""
    n = ra + rb
    if method == "svwn5":
        x = _exchange("lda", ra, None, None) + _exchange("lda", rb, None, None)
        return x + n * _vwn5((3 / (4 * _PI * n)) ** (1 / 3), (ra - rb) / n)
    saa, sbb = _limit(saa, 1e-40), _limit(sbb, 1e-40)
    if method == "tpss":
        ta, tb = _limit(ta, 1e-20), _limit(tb, 1e-20)
        saa, sbb = _limit(saa, None, 8 * ra * ta), _limit(sbb, None, 8 * rb * tb)
        top = 0.5 * (saa + sbb)
        sab = _limit(sab, -top.detach(), top)
        x = _exchange("tpss", ra, saa, ta) + _exchange("tpss", rb, sbb, tb)
        return x + _tpss_c(ra, rb, saa, sab, sbb, ta, tb)
    kind = "b88" if method in ("blyp", "bpbe") else "pbe"
    x = _exchange(kind, ra, saa, None) + _exchange(kind, rb, sbb, None)
    if method == "blyp":
        return x + _lyp(ra, rb, saa, sab, sbb)
    return x + _pbe_c(ra, rb, saa + 2 * sab + sbb)


def _densities(ao, P, tau):
    """rho, grad rho (3) and tau of the density matrix P (factor 2 inside)."""
    T = ao[0] @ P
    rho = (T * ao[0]).sum(1)
    g = [2 * (T * a).sum(1) for a in ao[1:]]
    t = 0.5 * sum(((a @ P) * a).sum(1) for a in ao[1:]) if tau else None
    return rho, g, t


def _dot(u, v):
    return sum(a * b for a, b in zip(u, v))


def _xc(basis, pts, wts, method, Ps, centres_grad=False, chunk=0):
    """Exc, electrons per matrix, dExc/dP (or dExc/dR) of the spin matrices Ps
    (one: closed shell)."""
    dev = Ps[0].device
    ao = _AOs(basis, dev)
    chunk = chunk or max(256, min(8192, (1 << 22) // basis.nbf // (3 if centres_grad else 1)))
    R = torch.tensor([a[1:] for a in basis.atoms], dtype=torch.float64, device=dev)
    R.requires_grad_(centres_grad)
    Ps = [P.detach().clone().requires_grad_(not centres_grad) for P in Ps]
    pts = torch.from_numpy(np.asarray(pts).reshape(-1, 3)).to(dev)
    wts = torch.from_numpy(np.asarray(wts)).to(dev)
    lda, mgga = method == "svwn5", method == "tpss"
    exc, nel = 0.0, [0.0] * len(Ps)
    for lo in range(0, len(wts), chunk):
        w = wts[lo:lo + chunk]
        a = ao(pts[lo:lo + chunk], R, not lda)
        q = [_densities(a, P, mgga) for P in Ps]
        for k in range(len(Ps)):
            nel[k] += float((w * q[k][0].detach()).sum())
        total = sum(x[0] for x in q)
        keep = total.detach() >= 1e-15
        sc = 0.5 if len(q) == 1 else 1.0
        u, v = q[0], q[-1]
        ra, rb = sc * u[0][keep], sc * v[0][keep]
        ga, gb = [sc * x[keep] for x in u[1]], [sc * x[keep] for x in v[1]]
        s = [None] * 3 if lda else [_dot(ga, ga), _dot(ga, gb), _dot(gb, gb)]
        t = [sc * u[2][keep], sc * v[2][keep]] if mgga else [None, None]
        e = (w[keep] * _energy_density(method, ra, rb, *s, *t)).sum()
        exc += float(e.detach())
        e.backward()
    if centres_grad:
        return exc, nel, R.grad
    return exc, nel, [0.5 * (P.grad + P.grad.T) for P in Ps]


def _vv10(basis, pts, wts, P, b=6.0, C=0.01):
    """VV10 energy and potential; a point's sums run over the points before it."""
    dev = P.device
    aof = _AOs(basis, dev)
    R = torch.tensor([a[1:] for a in basis.atoms], dtype=torch.float64, device=dev)
    x = torch.from_numpy(np.asarray(pts).reshape(-1, 3)).to(dev)
    w = torch.from_numpy(np.asarray(wts)).to(dev)
    step = max(256, (1 << 22) // basis.nbf)
    parts = [_densities(aof(x[lo:lo + step], R, True), P, False) for lo in range(0, len(w), step)]
    rho = torch.cat([p[0] for p in parts])
    g = [torch.cat([p[1][k] for p in parts]) for k in range(3)]
    sig = _dot(g, g)
    beta = (3.0 / b ** 2) ** 0.75 / 32.0
    live = rho >= 1e-8
    tmp = C * (sig / rho ** 2) ** 2
    om = (tmp + 4 * _PI / 3 * rho).sqrt()
    ka = b * 1.5 * _PI * (9 * _PI) ** (-1 / 6) * rho ** (1 / 6)
    i = torch.nonzero(live).reshape(-1)
    xl, wl, oml, kal = x[i], 2 * (rho * w)[i], om[i], ka[i]
    F = 0.5 * wl / (2 * kal ** 3)
    U = F * (1 / kal + 1 / (2 * kal))
    W = torch.zeros_like(F)
    m = len(i)
    rows = 2048
    for lo in range(0, m, rows):
        hi = min(m, lo + rows)
        for jo in range(0, hi, 8192):
            je = min(hi, jo + 8192)
            r2 = sum((xl[lo:hi, None, k] - xl[None, jo:je, k]) ** 2 for k in range(3))
            gi = r2 * oml[lo:hi, None] + kal[lo:hi, None]
            gj = r2 * oml[None, jo:je] + kal[None, jo:je]
            t = wl[None, jo:je] / (gi * gj * (gi + gj))
            if je > lo:
                t = t.masked_fill(torch.arange(lo, hi, device=dev)[:, None] <=
                                  torch.arange(jo, je, device=dev)[None], 0.0)
            u = t * (1 / gi + 1 / (gi + gj))
            F[lo:hi] += t.sum(1)
            U[lo:hi] += u.sum(1)
            W[lo:hi] += (u * r2).sum(1)
    F = -1.5 * F
    full = torch.zeros((3, len(w)), dtype=torch.float64, device=dev)
    full[:, i] = torch.stack([F, U, W])
    F, U, W = full
    ex = (beta + 0.5 * F) * w
    dor = (2 * _PI / 3 * rho - 2 * tmp) / om
    vr = torch.where(live, (beta + F + 1.5 * (U * ka / 6 + W * dor)) * w, beta * w)
    vs = torch.where(live & (sig > 0), 1.5 * W * tmp * rho / (sig * om) * w, torch.zeros_like(w))
    V = torch.zeros_like(P)
    for lo in range(0, len(w), step):
        a = aof(x[lo:lo + step], R, True)
        A = 0.5 * vr[lo:lo + step, None] * a[0]
        for k in range(3):
            A = A + (2 * vs * g[k])[lo:lo + step, None] * a[k + 1]
        V += a[0].T @ A
    return float((ex * rho).sum()), float((rho * w).sum()), V + V.T


def _becke(grid, dev):
    """Partitioned weights of a molecular grid (Becke cells, Treutler-Ahlrichs)."""
    pts, wts, own = grid.unpartitioned()
    xyz, rad = grid.atom_arrays()
    x, q = torch.from_numpy(pts).to(dev), torch.from_numpy(xyz).to(dev)
    d = torch.linalg.vector_norm(x[:, None] - q[None], dim=2)
    R = torch.linalg.vector_norm(q[:, None] - q[None], dim=2)
    P = torch.ones_like(d)
    for i in range(len(rad)):
        for j in range(i):
            mu = (d[:, i] - d[:, j]) / R[i, j]
            if abs(rad[i] - rad[j]) > 1e-14:
                chi = _S(rad[i] / rad[j])
                u = (chi - 1) / (chi + 1)
                mu = mu + u / (u * u - 1) * (1 - mu * mu)
            for _ in range(3):
                mu = 0.5 * (3 - mu * mu) * mu
            P[:, i] *= 0.5 * (1 - mu)
            P[:, j] *= 0.5 * (1 + mu)
    own = torch.from_numpy(own).to(dev).long()
    return pts, (torch.from_numpy(wts).to(dev) * P.gather(1, own[:, None])[:, 0] / P.sum(1)).cpu()


def exact(case, seed):
    path, method = case["path"], case["method"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    npts, nn, nat, n1, n2 = _sums(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    per = 12 if path in ("gradient", "ugradient") else 4
    if path != "batch" and npts * math.sqrt(nn) * per > 1.5e10:
        return None
    mols = _molecules(case, seed)
    vxc, scalars = [], []
    for k, (atoms, name) in enumerate(mols):
        b = _basis(atoms, name)
        if path == "geometry":
            pts, wts = _becke(_grid(case, atoms), dev)
            wts = wts.numpy()
        else:
            pts, wts = _grid(case, atoms).build()
        if path in ("uks", "ugradient"):
            Ps = [2 * d for d in _spin_densities(b, seed)]
        else:
            Ps = [2 * _density(b, seed + k if path == "batch" else seed)]
        if path in ("gradient", "ugradient"):
            return {"gradient": _xc(b, pts, wts, method, Ps, centres_grad=True)[2]}
        if path == "vv10":
            e, nel, V = _vv10(b, pts, wts, Ps[0])
            return {"vxc": V, "scalars": torch.tensor([e, nel], dtype=torch.float64)}
        e, nel, V = _xc(b, pts, wts, method, Ps)
        vxc.append(V)
        scalars += [e] + nel
    if path == "batch":
        vxc = torch.cat([V[0].reshape(-1) for V in vxc])
    else:
        vxc = torch.cat(vxc[0], dim=1)
    if path in ("host", "geometry"):
        out = {"vxc": vxc.cpu().numpy(), "scalars": scalars}
        if path == "geometry":
            out["weights"] = wts
        return out
    return {"vxc": vxc, "scalars": torch.tensor(scalars, dtype=torch.float64)}
