"""Cases whose time is followed from change to change: the calls that a plane-wave
program makes to this library, through ``cpw2000_amd.hk_psi``, on synthetic
crystals of the sizes that the tests and the benchmark use.

A case names a cell (diamond silicon-like, ``fcc`` primitive or ``r1 x r2 x r3``
conventional cells of lattice parameter ``a`` bohr), a cutoff ``ecut`` (Ha), a
number of bands, a k-point (``shift`` along a general direction) and the call
(``kind``):

``apply``    H|psi> of one k-point on resident arrays, library defaults or (``tune``) after ``Plan.tune``
``mixed``    the same in FP32-mixed arithmetic with the kernel choice pinned (``Plan.set_variant``)
``kgraph``   H|psi> of several k-points of one cell in one ``Graph`` launch
``spin``     two-component H|psi> with a non-collinear potential
``density``  electron density of the occupied bands
``forces``   forces and non-local energy of the occupied bands
``rr``       Rayleigh-Ritz of a block of bands
``dropin``   ``hk_psi_c16`` on host arrays (the Fortran call)
``step``     after the atoms moved: projectors rebuilt on the device, then a diagonalisation from the small-matrix start
"""

import functools
import math

import numpy as np
import torch

from cpw2000_amd import hk_psi

TWOPI = 2.0 * math.pi
RC = 1.8                     # radius of the Gaussian projectors (bohr)
D_S, D_P = 1.5, 0.8          # strengths of the s and p projectors (Ha)
DELQ = 0.002                 # step of the tabulated projectors (1/bohr)
QV = 3.0                     # largest |q| of the position-dependent local potential (1/bohr)


# ---------------------------------------------------------------------------
# cells and plane waves
# ---------------------------------------------------------------------------

def _lengths(kmax):
    """FFT lengths 2^a, 2^a 9, 2^a 25, 2^a 27, 2^a 5, 2^a 3 that hold -kmax..kmax, as the program's size table has them."""
    small, large = (2, 4, 6, 8, 10, 12, 16, 18, 20, 24, 32), (36, 40, 48, 50, 54, 64)
    table = list(small) + [f * n for f in (1, 2, 4, 8) for n in large]
    return tuple(next(n for n in table if n >= 2 * int(k) + 1) for k in kmax)


def _cell(case):
    """Lattice vectors (columns) and undisplaced fractional positions."""
    a = case["a"]
    if case["fcc"]:
        return 0.5 * a * np.array([[0.0, 1, 1], [1, 0, 1], [1, 1, 0]]), np.array([[0.0, 0, 0], [0.25, 0.25, 0.25]])
    r = (case["r1"], case["r2"], case["r3"])
    base = np.array([[0, 0, 0], [0, .5, .5], [.5, 0, .5], [.5, .5, 0]])
    base = np.concatenate([base, base + 0.25])
    pos = np.concatenate([(base + np.array([i, j, k])) / r for i in range(r[0]) for j in range(r[1]) for k in range(r[2])])
    return np.diag([a * n for n in r]), pos


def _natom(case):
    return 2 if case["fcc"] else 8 * case["r1"] * case["r2"] * case["r3"]


@functools.lru_cache(maxsize=None)
def _gvectors(fcc, a, r1, r2, r3, ecut):
    avec, _ = _cell(dict(fcc=fcc, a=a, r1=r1, r2=r2, r3=r3))
    bvec = TWOPI * np.linalg.inv(avec).T
    gcut = 2.0 * math.sqrt(2.0 * ecut)
    lim = [int(gcut * np.linalg.norm(avec[:, j]) / TWOPI) + 1 for j in range(3)]
    g = np.stack(np.meshgrid(*[np.arange(-m, m + 1) for m in lim], indexing="ij"), -1).reshape(-1, 3)
    g2 = ((g @ bvec.T) ** 2).sum(1)
    keep = g2 <= gcut * gcut
    g, g2 = g[keep], g2[keep]
    order = np.lexsort((g[:, 2], g[:, 1], g[:, 0], np.round(g2, 9)))
    return g[order].astype(np.int32), bvec, _lengths(np.abs(g).max(axis=0))


@functools.lru_cache(maxsize=None)
def _basis(fcc, a, r1, r2, r3, ecut, shift):
    """Plane waves of the k-point shift * (1, 1/2, -1/3): (k, isort, ekin, number of (x, y) columns)."""
    g, bvec, _ = _gvectors(fcc, a, r1, r2, r3, ecut)
    k = shift * np.array([1.0, 0.5, -1.0 / 3.0])
    ekin = 0.5 * (((g + k) @ bvec.T) ** 2).sum(1)
    order = np.arange(len(g)) if shift == 0 else np.argsort(ekin, kind="stable")
    m = int(np.searchsorted(ekin[order] > ecut, True)) if shift else int(np.argmax(ekin > ecut))
    isort = (order[:m] + 1).astype(np.int32)
    columns = len(np.unique(g[isort - 1][:, :2].astype(np.int64) @ np.array([100003, 1])))
    return k, isort, np.ascontiguousarray(ekin[order[:m]]), columns


def _key(case):
    return case["fcc"], case["a"], case["r1"], case["r2"], case["r3"], case["ecut"]


def _shifts(case):
    """The k-points of a case: one, or kgraph's, spread over the zone."""
    if case["kind"] != "kgraph":
        return [case["shift"]]
    return [case["shift"] + 0.5 * i / case["nk"] for i in range(case["nk"])]


class _Point:
    """Inputs of one k-point, on the GPU and (geometry) on the host, all from the generator of one seed."""

    def __init__(self, case, gen, shift, pos=None, v=None):
        self.g, self.bvec, self.n = _gvectors(*_key(case))
        self.k, self.isort, self.ekin, _ = _basis(*_key(case), shift)
        self.avec, base = _cell(case)
        self.m = len(self.isort)
        self.case, self.gen = case, gen
        dev = torch.device("cuda")
        self.gm = torch.from_numpy(self.g[self.isort - 1].astype(np.int64)).to(dev)
        self.q = (self.gm.double() + torch.from_numpy(self.k).to(dev)) @ torch.from_numpy(self.bvec.T.copy()).to(dev)
        self.ek = torch.from_numpy(self.ekin).to(dev)
        if pos is None:      # thermal displacements
            pos = base + np.linalg.solve(self.avec, 0.1 * torch.randn(len(base), 3, generator=gen, dtype=torch.float64, device=dev).cpu().numpy().T).T
        self.pos = pos
        n1, n2, n3 = self.n
        self.idx = (self.gm[:, 2] % n3, self.gm[:, 1] % n2, self.gm[:, 0] % n1)
        self.v = self.potential() if v is None else v
        self.kmscr = np.array([*np.abs(self.g).max(axis=0), n1, n2, n3, n1], np.int32)

    def potential(self, scale=0.3):
        """A smooth real potential on the mesh (Ha), as (n3, n2, n1)."""
        n1, n2, n3 = self.n
        noise = torch.randn(n3, n2, n1, generator=self.gen, dtype=torch.float64, device="cuda")
        f = [torch.fft.fftfreq(k, 1.0 / k, dtype=torch.float64, device="cuda") for k in (n1, n2, n3)]
        b = torch.from_numpy(self.bvec).cuda()
        g2 = sum((b[i, 0] * f[0][None, None, :] + b[i, 1] * f[1][None, :, None] + b[i, 2] * f[2][:, None, None]) ** 2 for i in range(3))
        v = torch.fft.ifftn(torch.fft.fftn(noise) * torch.exp(-g2 / 2.0)).real
        return (v * (scale / v.std())).contiguous()

    def bands(self, nb, rows=1):
        """Random bands (nb, rows * m) decaying with the kinetic energy, of unit norm."""
        z = torch.randn(nb, rows * self.m, generator=self.gen, dtype=torch.complex128, device="cuda")
        z *= torch.exp(-self.ek / 4.0).repeat_interleave(rows)
        return z / torch.linalg.vector_norm(z, dim=1, keepdim=True)

    def projectors(self):
        """(4 natom, m) s and p projectors, type -> l -> m (y, z, x) -> atom, and their strengths."""
        na = len(self.pos)
        omega = abs(np.linalg.det(self.avec))
        tau = torch.from_numpy(self.pos).cuda()
        phase = torch.polar(torch.ones((), dtype=torch.float64, device="cuda"), -TWOPI * (tau @ self.gm.double().T))
        rad = torch.exp(-0.5 * RC * RC * (self.q ** 2).sum(1)) / math.sqrt(omega)
        out = torch.empty(4 * na, self.m, dtype=torch.complex128, device="cuda")
        for i, y in enumerate((None, self.q[:, 1], self.q[:, 2], self.q[:, 0])):
            out[i * na:(i + 1) * na] = phase * (rad if y is None else 1j * y * rad)
        d = torch.tensor([D_S] * na + [D_P] * (3 * na), dtype=torch.float64, device="cuda")
        return out, d

    def plan(self):
        p = hk_psi.Plan(self.m, len(self.g), self.g.T, self.ekin, self.isort, self.kmscr)
        p.set_potential(self.v.reshape(-1).cpu().numpy())
        return p

    def to_mesh(self, psi):
        """psi(r) = sum_G psi(G) exp(iG.r)."""
        n1, n2, n3 = self.n
        box = torch.zeros(psi.shape[0], n3, n2, n1, dtype=torch.complex128, device="cuda")
        box[(slice(None), *self.idx)] = psi
        return torch.fft.ifftn(box, dim=(1, 2, 3), norm="forward")

    def from_mesh(self, f):
        return torch.fft.fftn(f, dim=(1, 2, 3), norm="forward")[(slice(None), *self.idx)]

    def chunks(self, nb):
        """Bands in pieces of at most about 2 GB of mesh."""
        step = max(1, int(1.2e8 // math.prod(self.n)))
        return [slice(b, min(nb, b + step)) for b in range(0, nb, step)]

    def h(self, psi, beta, d):
        """H psi in plain torch, 64 bits."""
        out = ((psi @ beta.conj().T) * d) @ beta + self.ek * psi
        for s in self.chunks(psi.shape[0]):
            out[s] += self.from_mesh(self.to_mesh(psi[s]) * self.v)
        return out

    def local_form(self):
        """q vectors (integers, 0 < |q| <= QV) and form factor (nq, 1) of the position-dependent local potential."""
        g = self.g.astype(np.int64)
        q2 = ((g @ self.bvec.T) ** 2).sum(1)
        keep = (q2 > 0) & (q2 <= QV * QV)
        f = -8.0 * np.exp(-0.72 * q2[keep]) / abs(np.linalg.det(self.avec))
        return g[keep].astype(np.int32), f[:, None]


def _points(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    pts = []
    for s in _shifts(case):
        pts.append(_Point(case, gen, s, *((pts[0].pos, pts[0].v) if pts else ())))
    return pts


def _occupations(case, seed):
    """Two electrons a band, fading over the highest ones (Fermi occupations)."""
    x = np.linspace(-8.0, 2.0, case["bands"]) + 0.05 * np.random.default_rng(seed).standard_normal(case["bands"])
    return 2.0 / (1.0 + np.exp(x))


def _spin_parts(pt, case):
    """Four potential components, spin-rotated projectors (2 nanl, 2 m) with strengths, two-component bands."""
    v = torch.stack([pt.v] + [pt.potential(0.1) for _ in range(3)])
    beta, d = pt.projectors()
    c, s, e = math.cos(0.35), math.sin(0.35), complex(math.cos(1.3), math.sin(1.3))
    u = ((c, -s * e.conjugate()), (s * e, c))
    sp = torch.empty(2 * beta.shape[0], 2 * pt.m, dtype=torch.complex128, device="cuda")
    for j in range(2):
        for i in range(2):
            sp[j::2, i::2] = beta * u[i][j]
    return v, sp, torch.stack([d, 0.5 * d], 1).reshape(-1), pt.bands(case["bands"], rows=2)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _case(name, kind, bands, ecut, r=(0, 0, 0), a=10.26, shift=0.0, **more):
    c = dict(kind=kind, fcc=r == (0, 0, 0), a=a, r1=r[0], r2=r[1], r3=r[2], ecut=ecut, bands=bands, shift=shift, **more)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one k-point of a primitive cell, 24^3: the smallest call, a few launches of microseconds each
        _case("apply_prim_16", "apply", 16, 10.0, shift=0.15, tune=False),
        # a 32-atom slab supercell on a long mesh of its own lengths
        _case("apply_slab_72", "apply", 72, 11.0, r=(1, 1, 4), tune=False),
        # the 64-atom cell, 72^3, 128 bands, tuned once as a self-consistency loop does
        _case("apply_64_tuned", "apply", 128, 15.0, r=(2, 2, 2), tune=True),
        # the same in FP32-mixed, with the choice that the tuner makes for it kept from an earlier run
        _case("mixed_64", "mixed", 128, 15.0, r=(2, 2, 2), plane=10, proj=2, back=4, splitk=256, sched=0),
        # 216 atoms, 108^3, 512 bands: the largest cell, as a program calls it that does not tune
        _case("apply_216", "apply", 512, 15.0, r=(3, 3, 3), tune=False),
        # six k-points of the 8-atom cell, 36^3, replayed as one graph: many small kernels
        _case("kgraph_8", "kgraph", 20, 15.0, r=(1, 1, 1), shift=0.1, nk=6),
        # non-collinear magnetism: 64 spinor bands of the 64-atom cell
        _case("spin_64", "spin", 64, 15.0, r=(2, 2, 2)),
        # the density after a diagonalisation
        _case("density_64", "density", 128, 15.0, r=(2, 2, 2)),
        # forces after self-consistency
        _case("forces_64", "forces", 128, 15.0, r=(2, 2, 2), a=10.5),
        # the subspace step of a caller's own eigensolver
        _case("rr_64", "rr", 128, 15.0, r=(2, 2, 2)),
        # the Fortran program's call with host arrays, blocks of bands as its diagonaliser passes them
        _case("dropin_64", "dropin", 128, 15.0, r=(2, 2, 2)),
        # an ionic step of the 64-atom cell in FP32-mixed: new projectors, then the lowest 64 bands
        _case("step_64", "step", 64, 15.0, r=(2, 2, 2), shift=0.2),
    ]


_SPECIAL = (24, 48, 64, 72, 80, 96, 108)


def draw(rng):
    kind = rng.choice(("apply", "apply", "apply", "mixed", "kgraph", "spin", "density", "forces", "rr", "dropin", "step"))
    while True:
        ecut = round(rng.uniform(7.0, 15.0), 2)
        a = round(rng.uniform(9.8, 10.8), 3)
        shift = rng.choice((0.0, round(rng.uniform(0.02, 0.4), 3)))
        shapes = {"apply": [(0, 0, 0), (1, 1, 1), (1, 1, 2), (1, 1, 3), (1, 2, 2), (2, 2, 1), (2, 2, 2), (2, 2, 3), (3, 3, 3)],
                  "mixed": [(1, 1, 1), (2, 2, 1), (2, 2, 2), (2, 2, 3)],
                  "kgraph": [(0, 0, 0), (1, 1, 1), (1, 1, 2)], "rr": [(1, 1, 1), (2, 2, 1), (2, 2, 2)],
                  "step": [(2, 2, 1), (2, 2, 2)]}
        r = rng.choice(shapes.get(kind, [(2, 2, 1), (2, 2, 2)]))
        most = {"kgraph": 40, "spin": 64, "rr": 160, "step": 64, "apply": 256}.get(kind, 128)
        bands = int(round(math.exp(rng.uniform(math.log(4), math.log(most)))))
        more = {}
        if kind == "apply":
            more["tune"] = rng.random() < 0.3 and r != (3, 3, 3)
        if kind == "kgraph":
            more["nk"] = rng.randint(2, 10)
        if kind == "mixed":
            more = dict(plane=rng.choice((7, 10)), proj=rng.choice((1, 2, 4)), back=rng.choice((0, 4)), splitk=rng.choice((128, 256, 512)), sched=rng.randint(0, 2))
        if kind == "step":
            bands = max(bands, 16)
        c = _case(None, kind, bands, ecut, r=r, a=a, shift=shift, **more)
        n = _lengths([int(2 * math.sqrt(2 * ecut) * np.linalg.norm(v) / TWOPI) for v in _cell(c)[0].T])
        if kind in ("spin", "density", "forces") and not (n[0] == n[1] and n[0] in _SPECIAL and n[2] in _SPECIAL):
            continue     # these paths are built for the special lengths
        if kind == "mixed" and not (n[0] == n[1] and n[0] in (24, 48, 64, 72, 80, 96) and n[2] in _SPECIAL):
            continue     # the pinned register kernels are built for these lengths
        return c


def prepare(case, seed):
    kind, nb = case["kind"], case["bands"]
    pts = _points(case, seed)
    pt = pts[0]
    s = {"kind": kind}
    if kind in ("apply", "mixed", "kgraph"):
        plans, psis = [], []
        for p in pts:
            beta, d = p.projectors()
            psis.append(p.bands(nb))
            torch.cuda.synchronize()
            plans.append(p.plan())
            plans[-1].set_projectors_device(beta, d)
        hs = [torch.zeros_like(x) for x in psis]
        s.update(plan=plans[0], psi=psis[0], hpsi=hs[0], prec=hk_psi.PREC_FP64)
        if kind == "kgraph":
            s.update(graph=hk_psi.Graph(plans, psis, hs), hs=hs)
        elif kind == "mixed":
            s["prec"] = hk_psi.PREC_FP32
            for what, key in ((hk_psi.TUNE_PLANE, "plane"), (hk_psi.TUNE_PROJ, "proj"), (hk_psi.TUNE_BACK, "back"), (hk_psi.TUNE_SPLITK, "splitk"), (hk_psi.TUNE_SCHED, "sched")):
                plans[0].set_variant(hk_psi.PREC_FP32, what, case[key])
        elif case["tune"]:
            plans[0].tune(psis[0], hs[0], hk_psi.PREC_FP64)
    elif kind == "spin":
        v, sp, d, psi = _spin_parts(pt, case)
        s.update(plan=pt.plan(), psi=psi, hpsi=torch.zeros_like(psi))
        s["plan"].set_potential_spin(v.reshape(4, -1).cpu().numpy().T, 4)
        s["plan"].set_projectors_spin(sp.cpu().numpy().T, d.cpu().numpy())
    elif kind in ("density", "forces"):
        s.update(plan=pt.plan(), psi=pt.bands(nb), occ=_occupations(case, seed))
        if kind == "forces":
            beta, d = pt.projectors()
            torch.cuda.synchronize()
            s["plan"].set_projectors_device(beta, d)
            q, f = pt.local_form()
            na = len(pt.pos)
            s["args"] = (pt.pos, pt.avec, np.tile(np.arange(na, dtype=np.int32), 4), q, f, np.zeros(na, np.int32))
    elif kind == "rr":
        psi = pt.bands(nb)
        s.update(psi=psi, hpsi=pt.h(psi, *pt.projectors()))
    elif kind == "dropin":
        beta, d = pt.projectors()
        psi = pt.bands(nb).cpu().numpy().T
        s["args"] = (pt.m, nb, psi, np.zeros_like(psi), True, len(pt.g), np.asfortranarray(pt.g.T), pt.ekin, pt.isort, pt.v.reshape(-1).cpu().numpy(), pt.kmscr,
                     beta.cpu().numpy().T, d.cpu().numpy(), beta.shape[0], pt.m, nb, beta.shape[0], len(pt.g), pt.v.numel())
    elif kind == "step":
        na = len(pt.pos)
        nq = int((math.sqrt(2.0 * case["ecut"]) + 3.0) / DELQ) + 4
        vkb = np.zeros((nq + 2, 4, 3, 1), order="F")
        vkb[:, 0, 1, 0] = vkb[:, 1, 1, 0] = np.exp(-0.5 * (RC * DELQ * np.arange(-2, nq)) ** 2)
        nkb = np.zeros((4, 3, 1), np.int32, order="F")
        nkb[:2, 1, 0] = 1
        psi = torch.zeros(nb, pt.m, dtype=torch.complex128, device="cuda")
        s.update(plan=pt.plan(), psi=psi, hpsi=torch.zeros_like(psi))
        s["kb"] = (pt.k, 4 * na, np.array([nq], np.int32), np.array([DELQ]), vkb, nkb, 1, np.array([na], np.int32), np.asfortranarray(pt.pos.T[:, :, None]),
                   np.asfortranarray(pt.avec.T @ pt.avec))
    return s


def run(s):
    kind = s["kind"]
    if kind in ("apply", "mixed"):
        return s["plan"].apply(s["psi"], s["hpsi"], s["prec"])
    if kind == "kgraph":
        s["graph"].launch()
        return s["hs"]
    if kind == "spin":
        return s["plan"].apply_spin(s["psi"], s["hpsi"], hk_psi.PREC_FP64)
    if kind == "density":
        return s["plan"].density(s["psi"], s["occ"])
    if kind == "forces":
        force, enl = s["plan"].forces(s["psi"], *s["args"], occ=s["occ"])
        return {"force": force, "enl": enl}
    if kind == "rr":     # the caller keeps its block: the step rotates a copy
        x, hx = s["psi"].clone(), s["hpsi"].clone()
        eig, res = hk_psi.rayleigh_ritz(x, hx)
        return {"eig": eig, "res": res, "x": x, "hx": hx}
    if kind == "dropin":
        return hk_psi.hk_psi_c16(*s["args"])
    s["plan"].build_projectors_kb(*s["kb"])
    # eigenvectors are fixed only up to the stopping residual and a phase: the eigenvalues are what can be compared
    ei, ifail, _ = s["plan"].ditsp(s["psi"], s["hpsi"], prec=hk_psi.PREC_FP32)
    return {"ei": ei, "ifail": ifail}


def work(case):
    """Bytes: bands and projectors read, results written, the potential read, once each.  Operations: both projector
    products, 5 per point and log2 of the length for the transforms of the occupied columns, planes and rows."""
    _, _, n = _gvectors(*_key(case))
    kind, nb, nanl = case["kind"], case["bands"], 4 * _natom(case)
    nbytes = flops = 0.0
    for shift in _shifts(case):
        _, isort, _, columns = _basis(*_key(case), shift)
        m, mesh = len(isort), math.prod(n)
        box = min(n[0], 2 * math.sqrt(columns / math.pi) + 1)     # occupied x lines
        fft = 5.0 * (columns * n[2] * math.log2(n[2]) + box * n[1] * n[2] * math.log2(n[1]) + mesh * math.log2(n[0]))
        gemm = 8.0 * m * nanl * nb
        if kind == "density":
            nbytes, flops = nbytes + 16.0 * m * nb + 8.0 * mesh, flops + fft * nb
        elif kind == "forces":
            nbytes, flops = nbytes + 16.0 * m * (nb + nanl), flops + fft * nb + 4 * gemm
        elif kind == "rr":
            nbytes, flops = nbytes + 64.0 * m * nb, flops + 4 * 8.0 * m * nb * nb
        elif kind == "spin":
            nbytes, flops = nbytes + 32.0 * m * (2 * nb + 2 * nanl) + 32.0 * mesh, flops + 2 * 2 * fft * nb + 2 * 2 * 2 * gemm
        elif kind == "step":      # about 150 products per band take the residual from the start to the tolerance
            nbytes, flops = nbytes + 16.0 * m * (2 * nb + nanl) + 8.0 * mesh, flops + 150 * (2 * fft * nb + 2 * gemm)
        else:
            nbytes, flops = nbytes + 16.0 * m * (2 * nb + nanl) + 8.0 * mesh, flops + 2 * fft * nb + 2 * gemm
    return {"bytes": nbytes, "flops": flops}


def exact(case, seed):
    kind, nb = case["kind"], case["bands"]
    if kind == "step":       # thousands of plane waves: a dense diagonalisation takes minutes
        return None
    pts = _points(case, seed)
    pt = pts[0]
    if kind in ("apply", "mixed", "kgraph"):
        hs = []
        for p in pts:
            beta, d = p.projectors()
            hs.append(p.h(p.bands(nb), beta, d))
        return hs if kind == "kgraph" else hs[0]
    if kind == "spin":
        v, sp, d, psi = _spin_parts(pt, case)
        out = ((psi @ sp.conj().T) * d) @ sp + pt.ek.repeat_interleave(2) * psi
        for s in pt.chunks(nb):
            up, dn = pt.to_mesh(psi[s, 0::2]), pt.to_mesh(psi[s, 1::2])
            out[s, 0::2] += pt.from_mesh((v[0] + v[1]) * up + (v[2] - 1j * v[3]) * dn)
            out[s, 1::2] += pt.from_mesh((v[0] - v[1]) * dn + (v[2] + 1j * v[3]) * up)
        return out
    if kind == "dropin":
        beta, d = pt.projectors()
        return pt.h(pt.bands(nb), beta, d).cpu().numpy().T
    if kind in ("density", "forces"):
        psi = pt.bands(nb)
        occ = torch.from_numpy(_occupations(case, seed)).cuda()
        rho = sum((occ[s, None, None, None] * pt.to_mesh(psi[s]).abs() ** 2).sum(0) for s in pt.chunks(nb))
        if kind == "density":
            return rho.reshape(-1)
        beta, d = pt.projectors()
        q, f = pt.local_form()
        n1, n2, n3 = pt.n
        qd = torch.from_numpy(q).cuda().long()
        rq = torch.fft.fftn(rho, norm="forward")[qd[:, 2] % n3, qd[:, 1] % n2, qd[:, 0] % n1]
        tau = torch.from_numpy(pt.pos).cuda()
        w = (1j * torch.exp(-1j * TWOPI * (tau @ qd.double().T)) * (torch.from_numpy(f[:, 0]).cuda() * rq.conj())).real
        force = TWOPI * w @ qd.double()
        p0 = psi @ beta.conj().T
        enl = float((occ[:, None] * d * p0.abs() ** 2).sum())
        for j in range(3):
            pj = (psi * pt.gm[:, j]) @ beta.conj().T
            t = (2.0 * occ[:, None] * d * (-1j * pj * p0.conj()).real).sum(0)
            force[:, j] += TWOPI * t.reshape(4, -1).sum(0)
        return {"force": force.cpu().numpy() @ np.linalg.inv(pt.avec), "enl": enl}
    # rr
    psi = pt.bands(nb)
    h = pt.h(psi, *pt.projectors())
    smat, hmat = (psi.conj() @ psi.T).cpu().numpy(), (psi.conj() @ h.T).cpu().numpy()
    li = np.linalg.inv(np.linalg.cholesky(smat))
    a = li @ hmat @ li.conj().T
    eig, u = np.linalg.eigh(0.5 * (a + a.conj().T))
    c = torch.from_numpy(li.conj().T @ u).cuda()
    e = torch.from_numpy(eig).cuda()
    res = ((c.T @ h - e[:, None] * (c.T @ psi)).abs() ** 2).sum(1)
    return {"eig": eig, "res": res.cpu().numpy(), "x": None, "hx": None}
