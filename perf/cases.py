"""Performance cases of the CheFSI library: H applications, Chebyshev filters
(single operators and batches), the subspace step and whole SCF runs, on
device-resident blocks through the public entry points (``lynx_amd.core``,
``lynx_amd.scf`` and the C ABI that they wrap).

The operators are generic: an FD12 grid of about 0.34 Bohr spacing, one atom
per 135 Bohr^3 (silicon's density) with Kleinman-Bylander projectors on
spheres of 1.4 Bohr (8 projectors) or 2.9 Bohr (32 projectors), and a smooth
potential.  ``exact`` restates the same operators in plain torch and numpy.
"""
from __future__ import annotations

import ctypes
import math
import os

import numpy as np
import torch

from lynx_amd import _lib as L
from lynx_amd import core
from lynx_amd.scf import Calculator

H0 = 0.342                 # grid spacing, Bohr
A_SI = 10.26               # silicon lattice constant, Bohr
FCC = 0.5 * np.array([[0.0, 1.0, 1.0], [1.0, 0.0, 1.0], [1.0, 1.0, 0.0]])
DIAMOND = np.array([[0.00, 0.00, 0.00], [0.25, 0.25, 0.25], [0.50, 0.50, 0.00], [0.75, 0.75, 0.25],
                    [0.50, 0.00, 0.50], [0.75, 0.25, 0.75], [0.00, 0.50, 0.50], [0.25, 0.75, 0.75]])
PSP = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(L.__file__))), "tests", "golden", "psp", "C.pot")
TORCH = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16, "c128": torch.complex128,
         "c64": torch.complex64}
CODE = {"f64": L.F64, "f32": L.F32, "bf16": L.BF16, "c128": L.C128, "c64": L.C64}
SIZE = {"f64": 8, "f32": 4, "bf16": 2, "c128": 16, "c64": 8}
KPT = (0.17, 0.29, -0.11)  # a general Bloch vector, 1/Bohr


def listed():
    return [
        # one H application on a small molecule-sized cell: call latency
        dict(name="apply_small_f64", kind="apply", cell="orth", nx=20, ny=20, nz=20, ncol=12, dtype="f64"),
        # the filter of a medium insulator supercell (64 atoms) in each storage type that the passes use
        dict(name="filter_64atoms_f64", kind="filter", cell="orth", nx=60, ny=60, nz=60, ncol=160, dtype="f64",
             degree=20),
        dict(name="filter_64atoms_bf16", kind="filter", cell="orth", nx=60, ny=60, nz=60, ncol=160, dtype="bf16",
             degree=20),
        # the reduced-precision filter of a large supercell (216 atoms)
        dict(name="filter_216atoms_f32", kind="filter", cell="orth", nx=90, ny=90, nz=90, ncol=480, dtype="f32",
             degree=20),
        # an orthorhombic cell with odd grid sizes and an odd block width
        dict(name="filter_ragged_f64", kind="filter", cell="orth", nx=47, ny=45, nz=51, ncol=61, dtype="f64",
             degree=18),
        # one k-point of an orthogonal cell (Bloch phases)
        dict(name="filter_kpoint_c128", kind="filter", cell="orth", nx=40, ny=40, nz=40, ncol=48, dtype="c128",
             degree=20),
        # a non-orthogonal cell at Gamma
        dict(name="filter_skew_f64", kind="filter", cell="fcc", nx=48, ny=48, nz=48, ncol=64, dtype="f64", degree=20),
        # all k-points of a primitive cell in one batch (6 x 6 x 6 grid)
        dict(name="batch_kpoints_c64", kind="batch_kpt", cell="fcc", nx=24, ny=24, nz=24, nk=112, ncol=12,
             dtype="c64", degree=20),
        # a batch of different structures, as in data generation for force fields
        dict(name="batch_frames_f64", kind="batch_mix", n8=32, n16=16, noxide=8, nbox=8, dtype="f64", degree=20),
        # Cholesky-QR and projection of a large block: the dense half of a pass
        dict(name="subspace_216atoms_f64", kind="subspace", cell="orth", nx=90, ny=90, nz=90, ncol=480, dtype="f64"),
        # whole self-consistent runs: a small cubic cell, and a primitive cell with k-points
        dict(name="scf_si8", kind="scf", cell="orth", n=30, nstates=24, kgrid=1),
        dict(name="scf_si2_kpoints", kind="scf", cell="fcc", n=24, nstates=12, kgrid=6),
    ]


def draw(rng):
    kind = rng.choice(["apply", "filter", "filter", "filter", "filter", "kpt", "skew", "skew", "batch_kpt",
                       "batch_mix", "subspace", "scf"])

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def dims(lo, hi, even=False):
        n = log(lo, hi)
        d = [max(lo, min(hi, int(round(n * rng.uniform(0.75, 1.3))))) for _ in range(3)]
        if even:
            d[0] += d[0] % 2
        return dict(nx=d[0], ny=d[1], nz=d[2])

    def columns(c, most, size):
        """A block of at most 2.8 GB, columns in proportion to the cell."""
        nd = c["nx"] * c["ny"] * c["nz"]
        return max(4, min(int(nd * 7e-4 * rng.uniform(0.7, 2.0)) + 4, most, int(1.4e9 / (nd * size))))

    degree = rng.randint(14, 24)
    if kind == "apply":
        c = dict(kind="apply", cell=rng.choice(["orth", "orth", "fcc"]), **dims(14, 48))
        return dict(c, ncol=rng.randint(1, 32), dtype=rng.choice(["f64", "f64", "f32", "c128"]))
    if kind == "filter":
        dtype = rng.choice(["f64", "f64", "f32", "bf16"])
        c = dict(kind="filter", cell="orth", **dims(20, 84, even=dtype == "bf16"))
        return dict(c, ncol=columns(c, 480, SIZE[dtype]), dtype=dtype, degree=degree)
    if kind in ("kpt", "skew"):
        dtype = "c128" if kind == "kpt" else rng.choice(["f64", "c128", "f32"])
        c = dict(kind="filter", cell="orth" if kind == "kpt" else "fcc", **dims(20, 56))
        return dict(c, ncol=columns(c, 160, SIZE[dtype]), dtype=dtype, degree=degree)
    if kind == "batch_kpt":
        c = dict(kind="batch_kpt", cell=rng.choice(["fcc", "orth"]), **dims(16, 32))
        return dict(c, nk=log(4, 112), ncol=rng.randint(6, 16), dtype=rng.choice(["c64", "c128"]), degree=degree)
    if kind == "batch_mix":
        return dict(kind="batch_mix", n8=log(2, 32), n16=log(1, 16), noxide=log(1, 8), nbox=log(1, 8),
                    dtype=rng.choice(["f64", "f32"]), degree=degree)
    if kind == "subspace":
        dtype = rng.choice(["f64", "f64", "c128"])
        c = dict(kind="subspace", cell="orth", **dims(28, 80))
        return dict(c, ncol=columns(c, 400, SIZE[dtype]), dtype=dtype)
    return dict(kind="scf", cell="orth", n=rng.randint(24, 32), nstates=rng.randint(20, 28), kgrid=1)


# ------------------------------------------------------------- operators --
class System:
    """Host description of one operator: lattice, potential and projectors."""

    def __init__(self, cell, n, seed, natom=None, heavy=0):
        rng = np.random.default_rng(seed)
        self.n = np.array(n)
        self.nd = int(np.prod(self.n))
        self.orth = cell == "orth"
        if self.orth:
            self.latvec = np.diag(self.n * H0)
        else:                                      # rhombohedral cell with the spacing of a primitive fcc cell
            self.latvec = (self.n * H0)[:, None] * FCC * math.sqrt(2.0)
        self.length = np.linalg.norm(self.latvec, axis=1)
        self.h = self.length / self.n
        self.unit = self.latvec / self.length[:, None]
        inv = np.linalg.inv(self.unit)
        self.metric = inv.T @ inv
        volume = abs(np.linalg.det(self.latvec))
        self.dv = volume / self.nd
        natom = max(1, round(volume / 135.0)) if natom is None else natom
        m = math.ceil(natom ** (1.0 / 3.0) - 1e-9)
        sites = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
        sites = sites[rng.permutation(len(sites))[:natom]]
        self.frac = ((sites + 0.5 + rng.uniform(-0.08, 0.08, sites.shape)) / m) % 1.0
        self.veff = self._potential(rng)
        self._projectors(natom, heavy)

    def _potential(self, rng):
        g = [2 * np.pi * np.arange(k) / k for k in self.n]
        v = np.full(self.n[::-1], -0.3)
        for _ in range(6):
            q = rng.integers(1, 4, 3)
            p = rng.uniform(0, 2 * np.pi, 3)
            v += rng.uniform(0.05, 0.2) * (np.cos(q[2] * g[2] + p[2])[:, None, None]
                                           * np.cos(q[1] * g[1] + p[1])[None, :, None]
                                           * np.cos(q[0] * g[0] + p[0])[None, None, :])
        return np.ascontiguousarray(v).ravel()

    def _projectors(self, natom, heavy):
        """Per atom two radial functions for each l (l <= 1 within 1.44 Bohr;
        the `heavy` first atoms l <= 3 within 2.9 Bohr), normalised on the
        grid; sphere points by periodic image."""
        self.img_atom, self.img_ndc, self.img_nproj, self.img_shift = [], [], [], []
        self.atoms = []                            # per atom: points, chi (points x projectors), image shifts
        gpos, chis, gammas, displ = [], [], [], [0]
        ext = np.linalg.norm(np.linalg.inv(self.unit), axis=0)
        for a in range(natom):
            lmax, rc = (3, 2.9) if a < heavy else (1, 1.44)
            pos = self.frac[a] * self.length
            rng = [np.arange(math.ceil((pos[i] - rc * ext[i]) / self.h[i]),
                             math.floor((pos[i] + rc * ext[i]) / self.h[i]) + 1) for i in range(3)]
            k, j, i = (t.ravel() for t in np.meshgrid(rng[2], rng[1], rng[0], indexing="ij"))
            ijk = np.stack([i, j, k], 1)
            d = (ijk * self.h - pos) @ self.unit
            r = np.linalg.norm(d, axis=1)
            keep = r <= rc
            ijk, d, r = ijk[keep], d[keep], r[keep]
            image = -np.floor_divide(ijk, self.n)
            order = np.lexsort(image.T)
            ijk, d, r, image = ijk[order], d[order], r[order], image[order]
            chi, gamma = _channels(d, r, rc, lmax)
            chi /= np.sqrt(self.dv * (chi * chi).sum(axis=0))
            w = ijk % self.n
            g = w[:, 0] + self.n[0] * (w[:, 1] + self.n[1] * w[:, 2])
            first = np.flatnonzero(np.r_[True, np.any(image[1:] != image[:-1], axis=1)])
            for b, e in zip(first, np.r_[first[1:], len(g)]):
                self.img_atom.append(a)
                self.img_ndc.append(e - b)
                self.img_nproj.append(chi.shape[1])
                self.img_shift.append(image[b] * self.length)
                chis.append(np.asfortranarray(chi[b:e]).ravel(order="F"))
            gpos.append(g)
            gammas.append(gamma)
            displ.append(displ[-1] + chi.shape[1])
            self.atoms.append((g, chi, image * self.length, gamma))
        self.raw = dict(img_atom=self.img_atom, img_ndc=self.img_ndc, img_nproj=self.img_nproj,
                        gpos=np.concatenate(gpos), chi=np.concatenate(chis), img_shift=np.array(self.img_shift).ravel(),
                        n_atom=natom, ip_displ=displ, gamma=np.concatenate(gammas))

    def hamiltonian(self):
        lat = core.Lattice(self.latvec, core.CellType.Orthogonal if self.orth else core.CellType.NonOrthogonal)
        grid = core.FDGrid(*(int(k) for k in self.n), lat)
        st = core.FDStencil(12, grid, lat)
        dom = core.Domain(grid)
        vnl = core.NonlocalProjector().setup_raw(**self.raw)
        H = core.Hamiltonian(0).setup(st, dom, grid, core.HaloExchange(dom, st.FDn()), vnl)
        H.set_veff(self.veff)
        return H

    def bounds(self):
        """(lambda_cutoff, eig_min, eig_max) from the potential's range and
        the stencil's symbol, filtering out the upper three quarters."""
        t = [np.linspace(0, 2 * np.pi, 33)[:-1]] * 3
        t = np.stack(np.meshgrid(*t, indexing="ij"), -1)
        top = 0.5 * self.symbol(t).max() + self.veff.max() + 2.0
        low = self.veff.min() - 1.0
        return low + 0.25 * (top - low), low, top

    def symbol(self, theta):
        """-laplacian of exp(i theta . index) on the grid."""
        w1, w2 = _weights()
        k = np.arange(1, 7)
        lap, d = 0.0, []
        for a in range(3):
            c = np.cos(theta[..., a, None] * k)
            lap = lap - self.metric[a, a] / self.h[a] ** 2 * (w2[0] + 2 * (c * w2[1:]).sum(-1))
            d.append(2 * (np.sin(theta[..., a, None] * k) * w1[1:]).sum(-1) / self.h[a])
        for a, b in ((0, 1), (0, 2), (1, 2)):
            lap = lap + 2 * self.metric[a, b] * d[a] * d[b]
        return lap


def _weights(n=6):
    """Central difference weights of order 2n: first and second derivative."""
    f = math.factorial
    w1 = [0.0] + [(-1) ** (k + 1) * f(n) ** 2 / (k * f(n - k) * f(n + k)) for k in range(1, n + 1)]
    w2 = [-2 * sum(1.0 / k ** 2 for k in range(1, n + 1))]
    w2 += [2 * (-1) ** (k + 1) * f(n) ** 2 / (k ** 2 * f(n - k) * f(n + k)) for k in range(1, n + 1)]
    return np.array(w1), np.array(w2)


def _channels(d, r, rc, lmax):
    x, y, z = d.T
    one = np.ones_like(x)
    angular = [[one], [y, z, x], [x * y, y * z, 2 * z * z - x * x - y * y, x * z, x * x - y * y],
               [y * (3 * x * x - y * y), x * y * z, y * (4 * z * z - x * x - y * y),
                z * (2 * z * z - 3 * x * x - 3 * y * y), x * (4 * z * z - x * x - y * y), z * (x * x - y * y),
                x * (x * x - 3 * y * y)]]
    cols, gamma = [], []
    for l in range(lmax + 1):
        for p, g in ((0, 0.9), (1, -0.4)):
            u = (1 - (r / rc) ** 2) ** 2 * np.exp(-(1.0 + 2.0 * p) * (r / rc) ** 2)
            for s in angular[l]:
                cols.append(u * s)
                gamma.append(g / (l + 1))
    return np.stack(cols, 1), np.array(gamma)


def _block(case, seed, rows, nd):
    """rows x nd uniform values in [-0.5, 0.5]: rows columns of nd points."""
    dt = TORCH[case["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    real = torch.float64 if dt in (torch.float64, torch.complex128) else torch.float32
    shape = (rows, nd, 2) if dt.is_complex else (rows, nd)
    x = torch.rand(shape, generator=g, device="cuda", dtype=real) - 0.5
    return torch.view_as_complex(x) if dt.is_complex else x.to(dt)


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _kpoint(case):
    return KPT if case["dtype"] in ("c128", "c64") else (0.0, 0.0, 0.0)


def _kpoints(case, length, seed):
    """nk k-points of the Brillouin zone."""
    return np.random.default_rng(seed + 17).uniform(-0.5, 0.5, (case["nk"], 3)) * 2 * np.pi / length


def _frames(case, seed):
    """(group, system, columns) of a batch of structures: 8-atom and 16-atom
    cells, perovskite-like cells with two heavy atoms, and a molecule in a box."""
    out = []
    for group, count, n, ncol, kw in (("n8", case["n8"], (30, 30, 30), 24, {}),
                                      ("n16", case["n16"], (30, 30, 60), 40, {}),
                                      ("noxide", case["noxide"], (28, 28, 28), 30, dict(natom=5, heavy=2)),
                                      ("nbox", case["nbox"], (50, 50, 50), 8, dict(natom=1))):
        out += [(group, System("orth", n, 1000 * seed + 100 * len(out) + i, **kw), ncol) for i in range(count)]
    return out


# ---------------------------------------------------------------- passes --
def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind)
    if kind == "scf":
        rng = np.random.default_rng(seed)
        orth = case["cell"] == "orth"
        base = DIAMOND if orth else DIAMOND[:2]
        latvec = A_SI * (np.eye(3) if orth else FCC)
        frac = base + rng.normal(0.0, 0.05 / A_SI, base.shape)
        n = case["n"]
        config = {"lattice": {"vectors": latvec.tolist(), "cell_type": "orthogonal" if orth else "nonorthogonal"},
                  "grid": {"Nx": n, "Ny": n, "Nz": n, "fd_order": 12},
                  "atoms": [{"pseudo_file": PSP, "fractional": True, "coordinates": frac.tolist()}],
                  "electronic": {"xc": "GGA_PBE", "smearing": "fermi-dirac", "temperature": 1000.0,
                                 "Nstates": case["nstates"]},
                  "scf": {"tolerance": 1e-6, "cheb_degree": 20},
                  "kpoints": {"grid": [case["kgrid"]] * 3}}
        s["calc"] = Calculator().set_config(config).setup()
    elif kind == "batch_kpt":
        m = System(case["cell"], _dims(case), seed)
        nk, nc = case["nk"], case["ncol"]
        s["H"] = m.hamiltonian()
        s["batch"] = core.BatchFilter([(s["H"], k) for k in _kpoints(case, m.length, seed)])
        s["x"] = _block(case, seed, nk * nc, m.nd).view(nk, nc, m.nd)
        s["y"] = torch.empty_like(s["x"])
        s["args"] = ([t.data_ptr() for t in s["x"]], [t.data_ptr() for t in s["y"]], [m.nd] * nk, [nc] * nk,
                     case["degree"], *m.bounds())
        s["dtype"] = case["dtype"]
    elif kind == "batch_mix":
        frames = _frames(case, seed)
        s["H"] = [m.hamiltonian() for _, m, _ in frames]
        s["batch"] = core.BatchFilter([(H, None) for H in s["H"]])
        s["x"], s["y"] = {}, {}
        for group in ("n8", "n16", "noxide", "nbox"):
            mine = [(m, nc) for g, m, nc in frames if g == group]
            m, nc = mine[0]
            s["x"][group] = _block(case, seed + len(s["x"]), len(mine) * nc, m.nd).view(len(mine), nc, m.nd)
            s["y"][group] = torch.empty_like(s["x"][group])
        xs = [t.data_ptr() for b in s["x"].values() for t in b]
        ys = [t.data_ptr() for b in s["y"].values() for t in b]
        lc, lo, hi = zip(*(m.bounds() for _, m, _ in frames))
        s["args"] = (xs, ys, [m.nd for _, m, _ in frames], [nc for _, _, nc in frames], case["degree"], lc, lo, hi)
        s["dtype"] = case["dtype"]
    else:
        m = System(case["cell"], _dims(case), seed)
        s["H"] = m.hamiltonian()
        s["H"].set_kpoint(_kpoint(case))
        s["code"], s["nd"], s["ncol"] = CODE[case["dtype"]], m.nd, case["ncol"]
        s["x"] = _block(case, seed, case["ncol"], m.nd)
        if kind == "subspace":
            s["hs"] = np.zeros((case["ncol"],) * 2, np.complex128 if case["dtype"] == "c128" else np.float64)
        else:
            s["y"] = torch.empty_like(s["x"])
            s["degree"], s["bounds"] = case.get("degree"), m.bounds()
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "scf":
        energy = s["calc"].run()
        eig, occ, rho, _ = s["calc"].scf.state()
        return {"energy": energy, "fermi": s["calc"].fermi_energy(), "eig": eig, "occ": occ, "rho": rho}
    if kind in ("batch_kpt", "batch_mix"):
        s["batch"].filter_device({"f64": np.float64, "f32": np.float32, "c64": np.complex64,
                                  "c128": np.complex128}[s["dtype"]], *s["args"])
        return s["y"]
    lib, ctx, nd, nc, x = L.lib(), s["H"].ctx, s["nd"], s["ncol"], s["x"].data_ptr()
    if kind == "apply":
        y = s["y"].data_ptr()
        L.check(lib.lynx_h_apply(ctx, s["code"], x, nd, y, nd, nc, 0.0, L.MEM_DEVICE), ctx)
        return s["y"]
    if kind == "filter":
        lc, lo, hi = s["bounds"]
        y = s["y"].data_ptr()
        L.check(lib.lynx_cheb_filter(ctx, s["code"], x, nd, y, nd, nc, s["degree"], lc, lo, hi, L.MEM_DEVICE), ctx)
        return s["y"]
    L.check(lib.lynx_orthogonalize(ctx, s["code"], x, nd, nc, L.MEM_DEVICE), ctx)
    L.check(lib.lynx_project_hamiltonian(ctx, s["code"], x, nd, nc, ctypes.c_void_p(s["hs"].ctypes.data),
                                         L.MEM_DEVICE), ctx)
    return {"x": s["x"], "hs": s["hs"]}


# ------------------------------------------------------------------ work --
def _apply_flops(nd, ncol, cell, cplx):
    """One H application: 13-point second differences in three directions
    (with the three mixed terms of a skew cell as differences of first
    differences), the potential and 8 projectors on a tenth of the points."""
    point = 18 + 2 * 19 + 2 + (6 * 18 if cell == "fcc" else 0) + 0.1 * 4 * 8
    return point * nd * ncol * (2 if cplx else 1)


def work(case):
    kind = case["kind"]
    if kind == "scf":
        nd = case["n"] ** 3
        nk = 1 if case["kgrid"] == 1 else case["kgrid"] ** 3 // 2 + 4
        cplx = case["kgrid"] > 1
        passes = 20 * nk
        nb = case["nstates"]
        flops = passes * (21 * _apply_flops(nd, nb, case["cell"], cplx) + 8 * nd * nb * nb * (4 if cplx else 1))
        return {"bytes": 8.0 * (3 * nd + 2 * nk * nb), "flops": float(flops)}
    if kind == "batch_mix":
        units = [(27000, 24, case["n8"]), (54000, 40, case["n16"]), (21952, 30, case["noxide"]),
                 (125000, 8, case["nbox"])]
        size = SIZE[case["dtype"]]
        return {"bytes": float(sum(k * (2 * size * nd * nc + 8 * nd) for nd, nc, k in units)),
                "flops": float(sum(k * case["degree"] * _apply_flops(nd, nc, "orth", False) for nd, nc, k in units))}
    nd = case["nx"] * case["ny"] * case["nz"]
    nc = case["ncol"] * case.get("nk", 1)
    cplx = case["dtype"] in ("c64", "c128")
    size = SIZE[case["dtype"]]
    one = _apply_flops(nd, nc, case["cell"], cplx)
    if kind == "subspace":
        # overlap and projection (their upper halves), the rotation by a triangular factor, one H application
        return {"bytes": float(2 * size * nd * nc + 8 * nd + size * nc * nc),
                "flops": float(3 * nd * nc * nc * (4 if cplx else 1) + one)}
    return {"bytes": float(2 * size * nd * nc + 8 * nd), "flops": float(one * case.get("degree", 1))}


# ----------------------------------------------------------------- exact --
class Exact:
    """The operator of a System on the GPU in 64-bit torch."""

    def __init__(self, m, kpt=None):
        self.m = m
        cplx = kpt is not None
        self.theta = np.asarray(kpt) * m.length if cplx else None
        self.veff = torch.from_numpy(m.veff).cuda()
        self.atoms = []
        for g, chi, shift, gamma in m.atoms:
            c = torch.from_numpy(chi).cuda()
            if cplx:
                c = c * torch.from_numpy(np.exp(-1j * (shift @ np.asarray(kpt)))).cuda()[:, None]
            self.atoms.append((torch.from_numpy(g).cuda(), c, torch.from_numpy(gamma).cuda() * m.dv))

    def shift(self, x, a, k):
        """x at index + k along axis a of (columns, nz, ny, nx)."""
        ax = 3 - a
        y = torch.roll(x, -k, ax)
        if self.theta is not None:
            w = y.narrow(ax, x.shape[ax] - k, k) if k > 0 else y.narrow(ax, 0, -k)
            w *= complex(np.exp(1j * math.copysign(1.0, k) * self.theta[a]))
        return y

    def first(self, x, a):
        w1, _ = _weights()
        return sum(w1[k] / self.m.h[a] * (self.shift(x, a, k) - self.shift(x, a, -k)) for k in range(1, 7))

    def apply(self, x):
        m = self.m
        _, w2 = _weights()
        v = x.view(x.shape[0], *(int(k) for k in m.n[::-1]))
        lap = torch.zeros_like(v)
        for a in range(3):
            c = m.metric[a, a] / m.h[a] ** 2
            lap += c * w2[0] * v
            for k in range(1, 7):
                lap += c * w2[k] * (self.shift(v, a, k) + self.shift(v, a, -k))
        if not m.orth:
            lap += 2 * m.metric[0, 1] * self.first(self.first(v, 1), 0)
            dz = self.first(v, 2)
            lap += 2 * m.metric[0, 2] * self.first(dz, 0)
            lap += 2 * m.metric[1, 2] * self.first(dz, 1)
        y = -0.5 * lap.view(x.shape) + self.veff * x
        for g, chi, gamma in self.atoms:
            coeff = (x[:, g] @ chi) * gamma
            y.index_add_(1, g, coeff @ chi.conj().T.contiguous())
        return y

    def filter(self, x, degree, cut, low, top):
        e, c = (top - cut) / 2, (top + cut) / 2
        s1 = s = e / (low - c)
        old, y = x, (self.apply(x) - c * x) * (s / e)
        for _ in range(degree - 1):
            t = 1 / (2 / s1 - s)
            old, y = y, (self.apply(y) - c * y) * (2 * t / e) - s * t * old
            s = t
        return y


def _wide(x):
    return x.to(torch.complex128 if x.is_complex() else torch.float64)


def _columns(f, x):
    """f over groups of columns that keep the temporaries small."""
    out = torch.empty_like(x, dtype=torch.complex128 if x.is_complex() else torch.float64)
    step = max(1, int(3e7) // x.shape[1])
    for b in range(0, x.shape[0], step):
        out[b:b + step] = f(_wide(x[b:b + step]))
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "scf":
        return None
    if kind == "batch_mix":
        out = {}
        frames = _frames(case, seed)
        for group in ("n8", "n16", "noxide", "nbox"):
            mine = [(m, nc) for g, m, nc in frames if g == group]
            m, nc = mine[0]
            x = _block(case, seed + len(out), len(mine) * nc, m.nd).view(len(mine), nc, m.nd)
            out[group] = torch.stack([Exact(m).filter(_wide(b), case["degree"], *m.bounds())
                                      for (m, _), b in zip(mine, x)])
        return out
    m = System(case["cell"], _dims(case), seed)
    if kind == "batch_kpt":
        x = _block(case, seed, case["nk"] * case["ncol"], m.nd).view(case["nk"], case["ncol"], m.nd)
        return torch.stack([Exact(m, k).filter(_wide(b), case["degree"], *m.bounds())
                            for k, b in zip(_kpoints(case, m.length, seed), x)])
    x = _block(case, seed, case["ncol"], m.nd)
    op = Exact(m, _kpoint(case) if x.is_complex() else None)
    if kind == "apply":
        return _columns(op.apply, x)
    if kind == "filter":
        return _columns(lambda v: op.filter(v, case["degree"], *m.bounds()), x)
    r = torch.linalg.cholesky(m.dv * (x.conj() @ x.T.contiguous()), upper=True)   # x holds columns as rows
    inv = torch.linalg.solve_triangular(r, torch.eye(len(r), dtype=r.dtype, device="cuda"), upper=True)
    q = inv.T.contiguous() @ x
    hs = m.dv * (q.conj() @ _columns(op.apply, q).T.contiguous())
    hs = 0.5 * (hs + hs.conj().T)
    return {"x": q, "hs": hs.T.contiguous().cpu().numpy()}
