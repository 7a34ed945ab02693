"""The advection work this library is used for, as measurable cases.

A case is a dict of plain values; `prepare` puts its inputs on the GPU (fields
evaluated from analytic profiles and a seeded hash, the construction of
maestroex_amd.workloads), `run` makes one call as a stepping program makes it,
and `exact` evaluates the same formulas in plain torch on the undivided
domain, without the library.  Kinds:

  pass     one advection pass over a level (MakeUtrans .. MakeRhoHFlux)
  levels   one pass over an AMR hierarchy, as a captured graph
  cons     MakeEdgeScal of the species in its conservative form (predict_rhoX)
  step     the differentiable scalar step on a periodic box, with its gradients
  boxstep  the same over a box list with outflow top and bottom
  update   UpdateScal (species, enthalpy) and UpdateVel
  fill     FillPatch of every scalar at level 0

Geometry of every kind but `step`: periodic but for the vertical direction
(y in 2-D, z in 3-D), which is outflow; a spherical case is outflow on every
side.  dx = 1 / (longest edge).
"""
import math
import random

import torch

import maestroex_amd as mx
from maestroex_amd import _abi
from maestroex_amd.adjoint import BoxStepper, ScalStepFn, ScalStepper
from maestroex_amd.fabs import BaseState, FaceMultiFab, Geometry, MultiFab, make_params

DEV = "cuda:0"
F64 = torch.float64
NG = 4  # ghost cells of the state


def listed():
    return [
        # a 2-D planar run at its usual base resolution: one small box, so
        # the launches and the host path count
        dict(name="pass2d-256", kind="pass", dim=2, nx=256, ny=256, nz=1, parts=1, ppm=1, nspec=3,
             sph=False),
        # the smallest 3-D level worth a call: one 32^3 box
        dict(name="pass3d-32", kind="pass", dim=3, nx=32, ny=32, nz=32, parts=1, ppm=1, nspec=3,
             sph=False),
        # an ordinary level of uneven boxes with odd edges and ppm_type 2
        dict(name="pass3d-ragged-ppm2", kind="pass", dim=3, nx=101, ny=84, nz=117, parts=3, ppm=2,
             nspec=3, sph=False),
        # the benchmark level: 256^3 as 8 boxes of 128^3, the default ppm_type 1
        dict(name="pass3d-256", kind="pass", dim=3, nx=256, ny=256, nz=256, parts=2, ppm=1,
             nspec=3, sph=False),
        # the same level with ppm_type 2
        dict(name="pass3d-256-ppm2", kind="pass", dim=3, nx=256, ny=256, nz=256, parts=2, ppm=2,
             nspec=3, sph=False),
        # a star in a box: spherical base state, outflow sides, ppm_type 2
        dict(name="star-192-ppm2", kind="pass", dim=3, nx=192, ny=192, nz=192, parts=3, ppm=2,
             nspec=3, sph=True),
        # an AMR hierarchy of many small uneven boxes on three levels, the
        # pass replayed as a graph as a stepping program does
        dict(name="levels3-ppm1", kind="levels", n0=128, parts=4, nbox1=40, nbox2=50, ppm=1,
             nspec=3),
        # conservative edge states of three species (species_pred_type 2)
        dict(name="cons-128", kind="cons", nx=128, ny=128, nz=128, parts=2, ppm=1, nspec=3),
        # forward and backward of the differentiable step: 128^3, 4 scalars
        dict(name="step-grad-128", kind="step", n=128, nc=4, ppm=1),
        # forward and backward over uneven boxes with outflow sides, ppm_type 2
        dict(name="boxstep-grad-ppm2", kind="boxstep", nx=90, ny=75, nz=110, parts=2, nc=2, ppm=2),
        # the update that closes a step
        dict(name="update-192", kind="update", nx=192, ny=192, nz=192, parts=2, nspec=3),
        # the ghost fill before a pass, on uneven boxes
        dict(name="fill-ragged", kind="fill", nx=190, ny=171, nz=203, parts=3, nspec=3),
    ]


def draw(rng):
    """One more case: edges spread over their logarithm, box lists of 1 to 4
    parts per direction, ppm_type and the number of species as used."""
    def edge(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pass", "pass", "pass", "pass2d", "star", "levels", "cons", "step",
                       "boxstep", "update", "fill"])
    if kind == "step":
        return dict(kind="step", n=edge(24, 136), nc=rng.randint(1, 4), ppm=rng.choice([1, 2]))
    if kind == "levels":
        return dict(kind="levels", n0=edge(48, 144), parts=rng.choice([2, 3, 4]),
                    nbox1=rng.randint(4, 40), nbox2=rng.randint(4, 50), ppm=rng.choice([1, 2]),
                    nspec=rng.randint(2, 4))
    if kind == "pass2d":
        return dict(kind="pass", dim=2, nx=edge(64, 1500), ny=edge(64, 1500), nz=1,
                    parts=rng.choice([1, 1, 2, 4]), ppm=rng.choice([0, 1, 1, 2]),
                    nspec=rng.randint(2, 5), sph=False)
    if kind == "star":
        n = edge(48, 200)
        return dict(kind="pass", dim=3, nx=n, ny=n, nz=n, parts=rng.choice([1, 2, 3]),
                    ppm=rng.choice([1, 2]), nspec=rng.randint(2, 3), sph=True)
    parts = rng.choice([1, 2, 2, 3])
    if kind == "pass":
        return dict(kind="pass", dim=3, nx=edge(24, 240), ny=edge(24, 240), nz=edge(24, 240),
                    parts=parts, ppm=rng.choice([0, 1, 1, 1, 2, 2, 2]), nspec=rng.randint(2, 4),
                    sph=False)
    if kind == "boxstep":
        return dict(kind=kind, nx=edge(24, 130), ny=edge(24, 130), nz=edge(24, 130),
                    parts=rng.choice([1, 2]), nc=rng.randint(1, 3), ppm=rng.choice([1, 2]))
    c = dict(kind=kind, nx=edge(24, 240), ny=edge(24, 240), nz=edge(24, 240), parts=parts,
             nspec=rng.randint(2, 5))
    if kind == "cons":
        c["ppm"] = rng.choice([1, 2])
    return c


# ---------------------------------------------------------------------------
# geometry


def _edges(case):
    return [case["nx"], case["ny"], case["nz"]] if "nx" in case else [case.get("n", 0)] * 3


def _cuts(n, parts, rng):
    """[0, n) in `parts` segments whose lengths differ by up to a third."""
    parts = max(1, min(parts, n // 12))
    cut = [round(n * p / parts) for p in range(parts + 1)]
    jit = n // parts // 6
    if n % parts:  # an even split stays even: it is how a level of equal boxes is made
        for p in range(1, parts):
            cut[p] += rng.randint(-jit, jit)
    return [(cut[p], cut[p + 1] - 1) for p in range(parts)]


def _boxes(case):
    n = _edges(case)
    rng = random.Random(n[0] * 7 + n[1] * 5 + n[2] * 3)
    seg = [_cuts(n[d], case["parts"], rng) if n[d] > 1 else [(0, 0)] for d in range(3)]
    return [((x[0], y[0], z[0]), (x[1], y[1], z[1])) for z in seg[2] for y in seg[1]
            for x in seg[0]]


def _geom(n, dim, sph, h):
    per = [0 if (sph or d == dim - 1) else 1 for d in range(dim)]
    bc = [_abi.PHYS_INTERIOR if p else _abi.PHYS_OUTFLOW for p in per]
    return Geometry(dim, n[:dim], [h] * dim, per, bc, bc), per


# ---------------------------------------------------------------------------
# inputs: every field is a function of the cell (or face) index, so that a box,
# its ghost cells and the whole domain see the same values


class Fields:
    """The fields of one level with cell width h and n cells."""

    def __init__(self, n, dim, per, h, nspec, sph, seed):
        self.n, self.dim, self.per, self.h = n, dim, per, h
        self.nspec, self.sph = nspec, sph
        self.vert = dim - 1
        rng = random.Random(seed)
        self.salt = rng.random()
        self.modes = []
        length = [n[d] * h for d in range(3)]
        for _ in range(8):
            k = [rng.randint(-3, 3) / length[d] if d < dim and per[d] else rng.uniform(-2.0, 2.0)
                 for d in range(3)]
            a = [rng.gauss(0, 1) for _ in range(3)]
            if dim == 2:
                c = [-k[1] * a[0], k[0] * a[0], 0.0]
            else:
                c = [k[1] * a[2] - k[2] * a[1], k[2] * a[0] - k[0] * a[2],
                     k[0] * a[1] - k[1] * a[0]]
            self.modes.append((k, c, rng.uniform(0, 2 * math.pi)))
        self.scale = 1.0 / max(sum(abs(c[d]) for _, c, _ in self.modes) for d in range(dim))
        self.centre = [0.5 * length[d] for d in range(3)]

    def index(self, lo, hi):
        """Index vectors lo..hi (per direction) mapped as the ghost fill maps
        them: periodic images, or the nearest valid cell beyond an outflow side."""
        out = []
        for d in range(3):
            i = torch.arange(lo[d], hi[d] + 1, device=DEV)
            if d >= self.dim:
                i = torch.zeros(1, dtype=torch.long, device=DEV)
            elif self.per[d]:
                i = i % self.n[d]
            else:
                i = i.clamp(0, self.n[d] - 1)
            out.append(i)
        return out

    def pos(self, idx, face=-1):
        x = [(idx[d].to(F64) + (0.0 if d == face else 0.5)) * self.h for d in range(3)]
        return [x[0][None, None, :], x[1][None, :, None], x[2][:, None, None]]

    def radius(self, x):
        if self.sph:
            return torch.sqrt(sum((x[d] - self.centre[d]) ** 2 for d in range(3)))
        return x[self.vert]

    @staticmethod
    def rho0(r):
        return torch.exp(-r / 0.3)

    def w0r(self, r):
        return 0.05 * r * (1.0 - r) if self.sph else 0.01 * r

    def w0vec(self, x, d):
        if not self.sph:
            return self.w0r(x[self.vert]) if d == self.vert else torch.zeros((), device=DEV,
                                                                             dtype=F64)
        r = self.radius(x)
        return torch.where(r > 0, self.w0r(r) * (x[d] - self.centre[d]) / r.clamp(min=1e-30), 0.0)

    def full(self, idx, parts):
        shp = [len(idx[2]), len(idx[1]), len(idx[0])]
        return torch.stack([torch.as_tensor(p, dtype=F64, device=DEV).expand(shp) for p in parts])

    def velocity(self, idx):
        x = self.pos(idx)
        u = [0.0] * self.dim
        for k, c, phi in self.modes:
            w = torch.cos(2 * math.pi * sum(k[d] * x[d] for d in range(self.dim)) + phi)
            for d in range(self.dim):
                u[d] = u[d] + (c[d] * self.scale) * w
        return self.full(idx, u)

    def w0_cart(self, idx):
        x = self.pos(idx)
        return self.full(idx, [self.w0vec(x, d) for d in range(self.dim)])

    def hash01(self, idx, c):
        a = (idx[0].to(F64) * 12.9898)[None, None, :] + (idx[1].to(F64) * 78.233)[None, :, None] \
            + (idx[2].to(F64) * 37.719)[:, None, None]
        v = torch.sin(a + 3.1 * c + 57.0 * self.salt) * 43758.5453
        return v - torch.floor(v)

    def density(self, idx):
        x = self.pos(idx)
        r = self.radius(x)
        d2 = sum((x[d] - self.centre[d]) ** 2 for d in range(self.dim))
        rho = self.rho0(r) * (1.0 + 0.1 * torch.exp(-d2 / 0.05 ** 2))
        return rho, r

    def scalars(self, idx):
        """rho', (rho h)', Temp and Pi (zero), mass fractions."""
        rho, r = self.density(idx)
        p = rho - self.rho0(r)
        X = [0.05 + self.hash01(idx, c) for c in range(self.nspec)]
        tot = sum(X)
        z = torch.zeros((), dtype=F64, device=DEV)
        return self.full(idx, [p, p * (2.0 - r), z, z] + [v / tot for v in X])

    def vel_force(self, idx):
        x = self.pos(idx)
        arg = 2 * math.pi * sum((d + 1) * x[d] for d in range(self.dim))
        rho, r = self.density(idx)
        f = [0.05 * torch.cos(arg + c) for c in range(self.dim)]
        f[self.vert] = f[self.vert] - 0.1 * (rho - self.rho0(r)) / rho
        return self.full(idx, f)

    def scal_force(self, idx):
        x = self.pos(idx)
        arg = 2 * math.pi * sum((d + 1) * x[d] for d in range(self.dim))
        return self.full(idx, [0.02 * torch.sin(arg + 0.5 * c) for c in range(4 + self.nspec)])

    def face(self, idx, d, which):
        x = self.pos(idx, face=d)
        r = self.radius(x)
        v = {"w0mac": lambda: self.w0vec(x, d), "r0mac": lambda: self.rho0(r),
             "h0mac": lambda: 2.0 - r, "rh0mac": lambda: self.rho0(r) * (2.0 - r)}[which]()
        return self.full(idx, [v])

    def base(self, nrow=0):
        """Planar base-state rows: w0 and edge states (n + 1), cell states."""
        nr = self.n[self.vert]
        zc = (torch.arange(nr, dtype=F64) + 0.5) * self.h
        ze = torch.arange(nr + 1, dtype=F64) * self.h
        if self.sph:
            w0 = torch.zeros(nr + 1, dtype=F64)
        else:
            w0 = self.w0r(ze)
        e = self.rho0(ze)
        c = self.rho0(zc)
        return dict(w0=w0, rho0=c, rhoh0=c * (2.0 - zc), rho0_edge=e, rhoh0_edge=e * (2.0 - ze),
                    rho0_predicted_edge=e.clone())

    @property
    def umax(self):
        return 1.01 if not self.sph else 1.05


def _pack(pieces):
    """Box arrays end to end in one buffer, each at a multiple of 256 bytes."""
    return torch.cat([torch.nn.functional.pad(a.reshape(-1), (0, -a.numel() % 32))
                      for a in pieces])


def _multifab(boxes, nc, ng, dim, bk, nodal_dir=-1):
    """A MultiFab whose boxes lie in one allocation (mf.flat), as an arena
    gives them to a program."""
    mf = MultiFab(boxes, nc, ng, dim, bk, nodal_dir=nodal_dir)
    mf.flat = _pack(mf.arrays)
    off = 0
    for b, a in enumerate(mf.arrays):
        mf.arrays[b] = mf.flat[off:off + a.numel()].view(a.shape)
        off += a.numel() + -a.numel() % 32
    return mf


def _facefab(boxes, nc, ng, dim, bk):
    fm = FaceMultiFab.__new__(FaceMultiFab)
    fm.dim = dim
    fm.d = [_multifab(boxes, nc, ng, dim, bk, nodal_dir=d) for d in range(dim)]
    return fm


def _flat(fm):
    return [fm[d].flat for d in range(fm.dim)]


def _level(F, boxes, bk, nlev=1, lev=0, nrow=0):
    """Inputs and outputs of one level of the pass as the library takes them."""
    dim, nscal = F.dim, 4 + F.nspec

    def cells(fn, nc, ng):
        mf = _multifab(boxes, nc, ng, dim, bk)
        for b, (lo, hi) in enumerate(boxes):
            mf.arrays[b].copy_(fn(F.index([q - ng for q in lo], [q + ng for q in hi])))
        return mf

    f = dict(utilde=cells(F.velocity, dim, NG),
             ufull=cells(lambda i: F.velocity(i) + F.w0_cart(i), dim, NG),
             w0_cart=cells(F.w0_cart, dim, 2), vel_force=cells(F.vel_force, dim, 1),
             scal=cells(F.scalars, nscal, NG), scal_force=cells(F.scal_force, nscal, 1))
    for name in ("w0mac", "r0mac", "rh0mac", "h0mac"):
        f[name] = None
        if F.sph:
            f[name] = fm = _facefab(boxes, 1, 1, dim, bk)
            for d in range(dim):
                for b, (lo, hi) in enumerate(boxes):
                    idx = [torch.arange(lo[q] - 1, hi[q] + 2 + (q == d), device=DEV)
                           for q in range(3)]
                    fm[d].arrays[b].copy_(F.face(idx, d, name))
    for name, v in F.base().items():
        rows = torch.zeros((nlev, max(nrow, len(v))), dtype=F64)
        rows[lev, :len(v)] = v
        f[name] = BaseState(rows.numpy(), bk)
    f["utrans"] = _facefab(boxes, 1, 1, dim, bk)
    f["umac"] = _facefab(boxes, 1, 1, dim, bk)
    f["sedge"] = _facefab(boxes, nscal, 0, dim, bk)
    f["sflux"] = _facefab(boxes, nscal, 0, dim, bk)
    f["etarhoflux"] = _multifab(boxes, 1, 1, dim, bk, nodal_dir=dim - 1)
    return f


def _outputs(f, sph=False):
    """What the pass writes.  With outflow on every side the face fill reads, in
    the domain's corners, ghost faces that it does not itself set (an earlier
    call's), so there the face velocities stand behind the edge states and
    fluxes computed from them."""
    names = ("sedge", "sflux") if sph else ("utrans", "umac", "sedge", "sflux")
    out = {name: _flat(f[name]) for name in names}
    out["etarhoflux"] = f["etarhoflux"].flat
    return out


# ---------------------------------------------------------------------------
# prepare and run


def _pass_setup(case, seed):
    n, dim = _edges(case), case["dim"]
    h = 1.0 / max(n)
    geom, per = _geom(n, dim, case["sph"], h)
    F = Fields(n, dim, per, h, case["nspec"], case["sph"], seed)
    dt, eps = 0.5 * h / F.umax, 1e-8 * F.umax
    return n, dim, h, geom, per, F, dt, eps


def _prep_pass(case, seed):
    n, dim, h, geom, per, F, dt, eps = _pass_setup(case, seed)
    boxes = _boxes(case)
    bk = mx.device_backend(DEV)
    p = make_params(geom, ppm_type=case["ppm"], nspec=case["nspec"], dt=dt, rel_eps=eps,
                    spherical=1 if case["sph"] else 0)
    f = _level(F, boxes, bk)
    return dict(m=mx.gpu_maestro(p, [boxes]), f=f, sph=case["sph"])


def _run_pass(st):
    st["m"].advance_pass(0, st["f"])
    return _outputs(st["f"], st["sph"])


def _overlaps(a, b, others):
    return any(all(a[d] <= q[1][d] and q[0][d] <= b[d] for d in range(3)) for q in others)


def _level_boxes(case):
    """Level 0 tiles the domain; a level-1 box lies anywhere, a level-2 box in
    a level-1 box with a coarse cell to spare; even corners and edges."""
    rng = random.Random(case["n0"] * 131 + case["nbox1"] * 17 + case["nbox2"])
    n0 = case["n0"] - case["n0"] % 2
    seg = []
    for _ in range(3):
        cut = [2 * round(n0 * p / case["parts"] / 2) for p in range(case["parts"] + 1)]
        for p in range(1, case["parts"]):
            cut[p] += 2 * rng.randint(-2, 2)
        seg.append([(cut[p], cut[p + 1] - 1) for p in range(case["parts"])])
    out = [[((x[0], y[0], z[0]), (x[1], y[1], z[1])) for z in seg[2] for y in seg[1]
            for x in seg[0]], [], []]
    n1 = 2 * n0
    for _ in range(4000):
        if len(out[1]) == case["nbox1"]:
            break
        e = [2 * rng.randint(8, 24) for _ in range(3)]
        a = tuple(2 * rng.randint(0, (n1 - e[d]) // 2) for d in range(3))
        b = tuple(a[d] + e[d] - 1 for d in range(3))
        if not _overlaps(a, b, out[1]):
            out[1].append((a, b))
    for _ in range(4000):
        if len(out[2]) == case["nbox2"]:
            break
        plo, phi = out[1][rng.randrange(len(out[1]))]
        room = [2 * (phi[d] - plo[d] + 1) - 4 for d in range(3)]
        e = [2 * rng.randint(4, min(32, room[d]) // 2) for d in range(3)]
        a = tuple(2 * plo[d] + 2 + 2 * rng.randint(0, (room[d] - e[d]) // 2) for d in range(3))
        b = tuple(a[d] + e[d] - 1 for d in range(3))
        if not _overlaps(a, b, out[2]):
            out[2].append((a, b))
    return n0, out


def _prep_levels(case, seed):
    n0, boxes = _level_boxes(case)
    bk = mx.device_backend(DEV)
    ns = [[n0 * 2 ** l] * 3 for l in range(3)]
    geoms = [_geom(n, 3, False, 1.0 / n[0]) for n in ns]
    F = [Fields(n, 3, g[1], 1.0 / n[0], case["nspec"], False, seed) for n, g in zip(ns, geoms)]
    dt, eps = 0.5 / ns[2][0] / F[0].umax, 1e-8 * F[0].umax
    p = make_params(geoms[0][0], ppm_type=case["ppm"], nspec=case["nspec"], dt=dt, rel_eps=eps,
                    extra_levels=[g[0] for g in geoms[1:]])
    fs = [_level(F[l], boxes[l], bk, nlev=3, lev=l, nrow=ns[2][0] + 1) for l in range(3)]
    m = mx.gpu_maestro(p, boxes)
    return dict(m=m, fs=fs, graph=m.pass_graph(fs))


def _run_levels(st):
    st["graph"].launch()
    return [_outputs(f) for f in st["fs"]]


def _prep_cons(case, seed):
    n = _edges(case)
    h = 1.0 / max(n)
    geom, per = _geom(n, 3, False, h)
    F = Fields(n, 3, per, h, case["nspec"], False, seed)
    boxes = _boxes(case)
    bk = mx.device_backend(DEV)
    p = make_params(geom, ppm_type=case["ppm"], nspec=case["nspec"], dt=0.5 * h / F.umax,
                    rel_eps=1e-8 * F.umax, species_pred_type=2)
    m = mx.gpu_maestro(p, [boxes])
    f = _level(F, boxes, bk)
    # the MAC velocity of the level: a MakeUtrans of the fields, ghosts filled
    m.MakeUtrans(0, f["utilde"], f["ufull"], f["umac"], None, f["w0_cart"])
    bcs, _ = m.bc_setup()
    return dict(m=m, f=f, bcs=bcs, nspec=case["nspec"])


def _run_cons(st):
    f, ns = st["f"], st["nspec"]
    st["m"].MakeEdgeScal(0, f["scal"], f["sedge"], f["umac"], f["scal_force"], False, st["bcs"],
                         4, 4, ns, True)
    return _flat(f["sedge"])


def _step_inputs(n, per, nc, seed):
    """Smooth-plus-rough scalars and a smooth MAC velocity, dense; faces
    0..n-1 along a periodic direction, 0..n along an outflow one."""
    h = [1.0 / q for q in n]
    F = Fields(n, 3, per, 1.0 / max(n), max(nc, 2), False, seed)
    idx = [torch.arange(q, device=DEV) for q in n]
    rho, r = F.density(idx)
    s = F.full(idx, [rho * (1.0 + 0.1 * c) + 0.05 * F.hash01(idx, c) for c in range(nc)])
    u = []
    for d in range(3):
        fi = [torch.arange(n[q] + (1 if q == d and not per[q] else 0), device=DEV)
              for q in range(3)]
        x = F.pos(fi, face=d)
        v = 0.0
        for k, c, phi in F.modes:
            v = v + (c[d] * F.scale) * torch.cos(
                2 * math.pi * sum(k[q] * x[q] for q in range(3)) + phi)
        u.append(v.expand([len(fi[2]), len(fi[1]), len(fi[0])]).contiguous())
    g = F.full(idx, [torch.cos(3.0 * c + F.hash01(idx, c + 9) * 6.0) for c in range(nc)])
    return s.contiguous(), u, g.contiguous(), 0.5 * min(h), 1e-8


def _prep_step(case, seed):
    s, u, g, dt, eps = _step_inputs([case["n"]] * 3, [1, 1, 1], case["nc"], seed)
    st = ScalStepper(case["n"], case["nc"], dt, eps, device=DEV, ppm_type=case["ppm"])
    return dict(st=st, s=s.requires_grad_(), u=[x.requires_grad_() for x in u], g=g)


def _run_step(st):
    out = ScalStepFn.apply(st["st"], st["s"], *st["u"])
    return [out.detach()] + list(torch.autograd.grad(out, [st["s"], *st["u"]], st["g"]))


def _prep_boxstep(case, seed):
    n, per = _edges(case), [1, 1, 0]
    s, u, g, dt, eps = _step_inputs(n, per, case["nc"], seed)
    st = BoxStepper(_boxes(case), n, per, case["nc"], dt, eps, ppm_type=case["ppm"], device=DEV)
    st._put_cells(st.s, s)
    st._put_cells(st.g, g)
    st._put_faces(st.u, u)
    return dict(st=st)


def _run_boxstep(state):
    st = state["st"]
    st.step_mf(st.s, st.u, st.snew)
    st.vjp_mf(st.s, st.u, st.g, st.sb, st.ub)
    return [st.snew.arrays, st.sb.arrays, [st.ub[d].arrays for d in range(3)]]


def _update_fields(case, seed, boxes, bk):
    nc = 4 + case["nspec"]
    gen = torch.Generator(device=DEV).manual_seed(seed)
    f = dict(sold=_multifab(boxes, nc, 0, 3, bk), snew=_multifab(boxes, nc, 0, 3, bk),
             force=_multifab(boxes, nc, 0, 3, bk), sflux=_facefab(boxes, nc, 0, 3, bk),
             uold=_multifab(boxes, 3, 0, 3, bk), unew=_multifab(boxes, 3, 0, 3, bk),
             vforce=_multifab(boxes, 3, 0, 3, bk), umac=_facefab(boxes, 1, 0, 3, bk),
             uedge=_facefab(boxes, 3, 0, 3, bk), w0c=_multifab(boxes, 3, 1, 3, bk))
    for key in ("force", "uold", "vforce", "w0c"):
        for a in f[key].arrays:
            a.uniform_(-1.0, 1.0, generator=gen)
    for key in ("sflux", "umac", "uedge"):
        for d in range(3):
            for a in f[key][d].arrays:
                a.uniform_(-0.01, 0.01, generator=gen)
    for a in f["sold"].arrays:
        a.uniform_(0.2, 1.0, generator=gen)
        a[0] = a[4:].sum(0)  # rho is the sum of the partial densities
    return f


def _prep_update(case, seed):
    n = _edges(case)
    h = 1.0 / max(n)
    geom, _ = _geom(n, 3, False, h)
    boxes = _boxes(case)
    bk = mx.device_backend(DEV)
    m = mx.gpu_maestro(make_params(geom, nspec=case["nspec"], dt=0.05 * h), [boxes])
    return dict(m=m, f=_update_fields(case, seed, boxes, bk), nspec=case["nspec"])


def _run_update(st):
    m, f = st["m"], st["f"]
    m.UpdateScal(0, f["sold"], f["snew"], f["sflux"], f["force"], 4, st["nspec"], None, 1e-3)
    m.UpdateScal(0, f["sold"], f["snew"], f["sflux"], f["force"], 1, 1, None, 1e-3)
    m.UpdateVel(0, f["uold"], f["unew"], f["umac"], f["uedge"], f["vforce"], None, None, f["w0c"],
                False)
    return [f["snew"].flat, f["unew"].flat]


def _prep_fill(case, seed):
    n = _edges(case)
    geom, per = _geom(n, 3, False, 1.0 / max(n))
    boxes = _boxes(case)
    bk = mx.device_backend(DEV)
    p = make_params(geom, nspec=case["nspec"])
    m = mx.gpu_maestro(p, [boxes])
    bcs, _ = m.bc_setup()
    nc = 4 + case["nspec"]
    mf = _multifab(boxes, nc, NG, 3, bk)
    F = Fields(n, 3, per, 1.0 / max(n), nc, False, seed)
    for b, (lo, hi) in enumerate(boxes):
        idx = F.index(lo, hi)
        mf.arrays[b][(slice(None),) + mf.valid_region(b)] = \
            torch.stack([F.hash01(idx, c) for c in range(nc)])
    return dict(m=m, mf=mf, bcs=bcs, nc=nc)


def _run_fill(st):
    st["m"].FillPatch(0, st["mf"], st["mf"], 0, 0, st["nc"], 0, st["bcs"], 0)
    return st["mf"].flat


_PREP = dict(cons=_prep_cons, step=_prep_step, boxstep=_prep_boxstep, update=_prep_update,
             fill=_prep_fill, levels=_prep_levels)
_PREP["pass"] = _prep_pass
_RUN = dict(cons=_run_cons, step=_run_step, boxstep=_run_boxstep, update=_run_update,
            fill=_run_fill, levels=_run_levels)
_RUN["pass"] = _run_pass


def prepare(case, seed):
    st = _PREP[case["kind"]](case, seed)
    st["kind"] = case["kind"]
    return st


def run(state):
    return _RUN[state["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    """Inputs read once and outputs written once (valid points, FP64), and the
    operations of the formulas with neighbours' terms shared: 331 per cell and
    component for 3-D edge states with ppm_type 1 (tests/test_oracle.py counts
    them), about half again with ppm_type 2, and about 0.6 of it in 2-D."""
    kind = case["kind"]
    if kind == "levels":
        _, boxes = _level_boxes(case)
        cells = sum(math.prod(hi[d] - lo[d] + 1 for d in range(3)) for b in boxes for lo, hi in b)
        dim, sph = 3, False
    else:
        cells, dim, sph = math.prod(_edges(case)), case.get("dim", 3), case.get("sph", False)
    ops = {0: 220, 1: 331, 2: 500}[case.get("ppm", 1)] * (0.6 if dim == 2 else 1.0)
    if kind in ("pass", "levels"):
        nc = case["nspec"] + 2
        d8 = 3 * dim + 1 + 2 * nc + 2 * dim + 2 * dim * nc + 1 + (9 if sph else 0)
        return dict(bytes=8 * d8 * cells, flops=int((ops * (nc + dim) + 60 * dim) * cells))
    if kind == "cons":
        nc = case["nspec"]
        return dict(bytes=8 * (nc * 5 + 3) * cells, flops=int((ops + 40) * nc * cells))
    if kind in ("step", "boxstep"):
        nc = case["nc"]
        # forward: s, u, snew; backward: s, u, gbar, sbar, ubar
        return dict(bytes=8 * (5 * nc + 9) * cells, flops=int(4 * ops * nc * cells))
    if kind == "update":
        ns = case["nspec"]
        d8 = (2 + 6 * ns) + 6 + 3 * 3 + 3 + 9 + 1
        return dict(bytes=8 * d8 * cells, flops=(12 * ns + 12 + 45) * cells)
    nc = 4 + case["nspec"]
    ghost = sum(math.prod(hi[d] - lo[d] + 1 + 2 * NG for d in range(3))
                - math.prod(hi[d] - lo[d] + 1 for d in range(3)) for lo, hi in _boxes(case))
    return dict(bytes=16 * nc * ghost, flops=0)


def tolerance(case):
    """FP64 throughout.  Plain torch, with some sums in another order, differs
    from the level stages by up to 2e-17 of the result's norm (most values are
    the same bits) and from the gradients by up to 4e-16; copies (fill) are the
    same values.  Four times that is below FP64's unit roundoff times a few:"""
    if case["kind"] == "fill":
        return "exact"
    return dict(rel=2e-15 if case["kind"] in ("step", "boxstep") else 1e-15)


# ---------------------------------------------------------------------------
# the same formulas in plain torch, on the undivided domain.  Arrays are
# (..., z, y, x); a face array holds at index i the face below cell i.


def _sh(a, d, o):
    return torch.roll(a, -o, dims=-(d + 1)) if o else a


def _mn(a, b):
    return torch.where(b < a, b, a)


def _mx(a, b):
    return torch.where(a < b, b, a)


def _vl(a, b, c):
    dl, dr, dc = 2.0 * (b - a), 2.0 * (c - b), 0.5 * (c - a)
    m = _mn(dc.abs(), _mn(dl.abs(), dr.abs()))
    return torch.where(dl * dr > 0, torch.where(dc < 0, -m, m), torch.zeros_like(m))


def _cs_face(a, b, c, d):
    e = (7.0 / 12.0) * (b + c) - (1.0 / 12.0) * (a + d)
    d2, dl, dr = 3.0 * (b - 2.0 * e + c), a - 2.0 * b + c, b - 2.0 * c + d
    sg = torch.where(d2.detach() < 0, -1.0, 1.0)
    lim = sg * _mx(_mn(1.25 * sg * dl, _mn(1.25 * sg * dr, sg * d2)), torch.zeros_like(e))
    return torch.where((e - b) * (c - e) < 0, 0.5 * (b + c) - lim / 6.0, e)


def _cs_side(al, other, del_, big):
    """The limited `al` of the Colella-Sekora cell where |al| > 2 |other|."""
    sg = torch.where(other.detach() < 0, -1.0, 1.0)
    den = 4.0 * (al + other)
    amax = -al * al / torch.where(big, den, 1.0)
    first = sg * amax >= sg * del_
    room = sg * (del_ - other) >= 1.e-10
    arg = del_ * del_ - del_ * other
    take = big & first
    root = torch.sqrt(torch.where(take & room, arg, 1.0))
    return torch.where(take, torch.where(room, -2.0 * del_ - 2.0 * sg * root, -2.0 * other), al)


def _ppm(s, d, ppm):
    """Edge values (sm, sp) of every cell along d."""
    sm1, sp1 = _sh(s, d, -1), _sh(s, d, 1)
    if ppm == 1:
        dl = _vl(sm1, s, sp1)
        f = 0.5 * (s + sm1) - (dl - _sh(dl, d, -1)) / 6.0
        f = _mx(f, _mn(s, sm1))
        f = _mn(f, _mx(s, sm1))
        sm, sp = f, _sh(f, d, 1)
        flat = (sp - s) * (s - sm) <= 0
        hi = (sp - s).abs() >= 2.0 * (sm - s).abs()
        lo = (sm - s).abs() >= 2.0 * (sp - s).abs()
        return (torch.where(flat, s, torch.where(~hi & lo, 3.0 * s - 2.0 * sp, sm)),
                torch.where(flat, s, torch.where(hi, 3.0 * s - 2.0 * sm, sp)))
    f = _cs_face(_sh(s, d, -2), sm1, s, sp1)
    fm, fp, fpp = _sh(f, d, -1), _sh(f, d, 1), _sh(f, d, 2)
    ap, am = fp - s, f - s
    bigp, bigm = ap.abs() > 2.0 * am.abs(), am.abs() > 2.0 * ap.abs()
    dfm, dfp, dbm, dbp = f - fm, fpp - fp, s - sm1, sp1 - s
    use_f = _mn(dfm.abs(), dfp.abs()) >= _mn(dbm.abs(), dbp.abs())
    chk = torch.where(use_f, dfm, dbm) * torch.where(use_f, dfp, dbp) <= 0
    ext = (am * ap >= 0) | ((bigp | bigm) & chk)
    d2 = 6.0 * (am + ap)
    sm2, sp2 = _sh(s, d, -2), _sh(s, d, 2)
    d2l, d2r, d2c = sm2 - 2.0 * sm1 + s, s - 2.0 * sp1 + sp2, sm1 - 2.0 * s + sp1
    sg = torch.where(d2.detach() < 0, -1.0, 1.0)
    lim = _mx(_mn(sg * d2, _mn(1.25 * sg * d2l, _mn(1.25 * sg * d2r, 1.25 * sg * d2c))),
              torch.zeros_like(s))
    d2a = _mx(d2.abs(), torch.full_like(s, 1.e-10))
    ap2 = _cs_side(ap, am, sm1 - s, bigp & ~ext)
    am2 = _cs_side(am, ap, sp1 - s, bigm & ~ext)
    return (s + torch.where(ext, am * lim / d2a, am2), s + torch.where(ext, ap * lim / d2a, ap2))


def _trace(s, d, ppm, uhi, ulo, dt, h, eps):
    """Ip (at the high face) and Im (at the low face) of every cell along d."""
    sm, sp = _ppm(s, d, ppm)
    s6 = 6.0 * s - 3.0 * (sm + sp)
    sg = uhi.abs() * dt / h
    Ip = torch.where(uhi > eps, sp - 0.5 * sg * (sp - sm - (1.0 - 2.0 / 3.0 * sg) * s6), s)
    sg = ulo.abs() * dt / h
    Im = torch.where(ulo < -eps, sm + 0.5 * sg * (sp - sm + (1.0 - 2.0 / 3.0 * sg) * s6), s)
    return Ip, Im


def _slope4(s, d):
    """Limited fourth-order slopes (ppm_type 0)."""
    def second(a, b, c):
        cen = 0.5 * (c - a)
        l, r = 2.0 * (b - a), 2.0 * (c - b)
        lim = torch.where(r * l > 0, _mn(l.abs(), r.abs()), torch.zeros_like(l))
        return cen, lim, torch.where(cen < 0, -1.0, 1.0)

    cen, lim, sg = second(_sh(s, d, -1), s, _sh(s, d, 1))
    two = sg * _mn(lim, cen.abs())
    ds = 4.0 / 3.0 * cen - (_sh(two, d, 1) + _sh(two, d, -1)) / 6.0
    return sg * _mn(ds.abs(), lim)


class Ref:
    """Grid of the reference: g ghost cells on every side (0 when every
    direction is periodic: the shifts wrap)."""

    def __init__(self, n, dim, per, h, dt, eps, ppm):
        self.n, self.dim, self.per, self.dt, self.eps, self.ppm = n, dim, per, dt, eps, ppm
        self.h = h if isinstance(h, list) else [h] * 3
        self.g = 0 if all(per[:dim]) else NG
        self.lo, self.hi = [None] * 3, [None] * 3
        for d in range(dim):
            if not per[d]:
                i = torch.arange(-self.g, n[d] + self.g, device=DEV)
                shp = [1, 1, 1]
                shp[2 - d] = len(i)
                self.lo[d], self.hi[d] = (i == 0).view(shp), (i == n[d]).view(shp)

    def refill(self, a, face=-1):
        """Ghost points from the valid ones: images, or the nearest point."""
        if self.g == 0:
            return a
        for d in range(self.dim):
            i = torch.arange(-self.g, self.n[d] + self.g, device=DEV)
            i = i % self.n[d] if self.per[d] else i.clamp(0, self.n[d] - 1 + (d == face))
            a = a.index_select(a.dim() - 1 - d, i + self.g)
        return a

    def outflow(self, d, l, r, normal=False):
        if self.lo[d] is None:
            return l, r
        z = torch.zeros((), dtype=F64, device=DEV)
        rr = _mn(r, z) if normal else r
        l, r = torch.where(self.lo[d], rr, l), torch.where(self.lo[d], rr, r)
        ll = _mx(l, z) if normal else l
        return torch.where(self.hi[d], ll, l), torch.where(self.hi[d], ll, r)

    def edge(self, s, f, um, cons=False):
        """Edge states of one component (MakeEdgeScal)."""
        dt, eps, dim, h = self.dt, self.eps, self.dim, self.h

        def pick(l, r, u, thr):
            return torch.where(u.abs() > thr, torch.where(u > 0, l, r), 0.5 * (l + r))

        def diff(d, x):
            return _sh(x, d, 1) - x

        def term(t, H, c_adv, c_cons):
            """Per-cell transverse correction by direction t."""
            u = um[t]
            if cons:
                return (c_cons / h[t]) * diff(t, H * u)
            return (c_adv / h[t]) * (_sh(u, t, 1) + u) * diff(t, H)

        L, R, H = [], [], []
        for d in range(dim):
            if self.ppm == 0:
                sl = _slope4(s, d)
                cu = dt * um[d] / h[d]
                l = _sh(s, d, -1) + 0.5 * (1.0 - cu) * _sh(sl, d, -1)
                r = s - 0.5 * (1.0 + cu) * sl
            else:
                Ip, r = _trace(s, d, self.ppm, _sh(um[d], d, 1), um[d], dt, h[d], eps)
                l = _sh(Ip, d, -1)
            l, r = self.outflow(d, l, r)
            L.append(l)
            R.append(r)
            H.append(pick(l, r, um[d], 0.0 if dim == 3 else eps))
        if cons:
            div = sum(diff(d, um[d]) for d in range(dim)) / h[0]
        T = {}
        if dim == 3:
            for t in range(3):
                x = term(t, H[t], dt / 6.0, dt / 3.0)
                for d in range(3):
                    if d == t:
                        continue
                    if cons:
                        b, c = (dt / 3.0) * s * div, (dt / 3.0 / h[t]) * s * diff(t, um[t])
                        l = L[d] - _sh(x, d, -1) - _sh(b, d, -1) + _sh(c, d, -1)
                        r = R[d] - x - b + c
                    else:
                        l, r = L[d] - _sh(x, d, -1), R[d] - x
                    l, r = self.outflow(d, l, r)
                    T[d, t] = pick(l, r, um[d], eps)
        out = []
        for d in range(dim):
            l, r = L[d], R[d]
            for t in range(dim):
                if t != d:
                    x = term(t, T[t, 3 - d - t] if dim == 3 else H[t], 0.25 * dt, 0.5 * dt)
                    l, r = l - _sh(x, d, -1), r - x
            if cons:
                x = (0.5 * dt / h[d]) * s * diff(d, um[d])
                l, r = l - _sh(x, d, -1), r - x
            if f is not None:
                l, r = l + 0.5 * dt * _sh(f, d, -1), r + 0.5 * dt * f
            e = pick(l, r, um[d], eps)
            if self.lo[d] is not None:
                e = torch.where(self.lo[d], r, torch.where(self.hi[d], l, e))
            out.append(e)
        return out

    def riemann(self, l, r, w):
        if w is None:
            test = ((l <= 0) & (r >= 0)) | ((l + r).abs() < self.eps)
            res = torch.where(0.5 * (l + r) > 0, l, r)
        else:
            test = ((l + w <= 0) & (r + w >= 0)) | ((l + r + 2.0 * w).abs() < self.eps)
            res = torch.where(0.5 * (l + r) + w > 0, l, r)
        return torch.where(test, torch.zeros_like(res), res)

    def vel_states(self, u, uf):
        """Left and right states of every velocity component on d-faces."""
        L, R = [], []
        for d in range(self.dim):
            l, r = [], []
            for c in range(self.dim):
                if self.ppm == 0:
                    sl = _slope4(u[c], d)
                    z = torch.zeros((), dtype=F64, device=DEV)
                    cu = 0.5 * self.dt / self.h[d]
                    a = _sh(u[c] + (0.5 - cu * _mx(z, uf[d])) * sl, d, -1)
                    b = u[c] - (0.5 + cu * _mn(z, uf[d])) * sl
                else:
                    a, b = _trace(u[c], d, self.ppm, uf[d], uf[d], self.dt, self.h[d], self.eps)
                    a = _sh(a, d, -1)
                l.append(a)
                r.append(b)
            L.append(l)
            R.append(r)
        return L, R

    def velocities(self, u, uf, force, w, w0):
        """(utrans, umac) with w0 added and the ghost faces filled; w[d] the
        velocity the Riemann solve adds on d-faces (or None)."""
        dim, dt, h = self.dim, self.dt, self.h
        L, R = self.vel_states(u, uf)
        tr = []
        for d in range(dim):
            l, r = self.outflow(d, L[d][d], R[d][d], normal=True)
            v = self.refill(self.riemann(l, r, w[d]), d)
            tr.append(v if w0[d] is None else self.refill(v + w0[d], d))

        def avg(t, l, r):
            return torch.where(t.abs() < self.eps, 0.5 * (l + r), torch.where(t > 0, l, r))

        U = []
        for d in range(dim):
            for c in range(dim):
                L[d][c], R[d][c] = self.outflow(d, L[d][c], R[d][c], normal=c == d)
            U.append([avg(tr[d], L[d][c], R[d][c]) for c in range(dim)])

        def term(c0, t, x):
            return (c0 / h[t]) * (_sh(tr[t], t, 1) + tr[t]) * (_sh(x, t, 1) - x)

        T = {}
        if dim == 3:
            for d in range(3):
                for t in range(3):
                    if t != d:
                        o = 3 - d - t
                        x = term(dt / 6.0, t, U[t][o])
                        l, r = self.outflow(d, L[d][o] - _sh(x, d, -1), R[d][o] - x)
                        T[d, t] = avg(tr[d], l, r)
        um = []
        for d in range(dim):
            l, r = L[d][d], R[d][d]
            for t in range(dim):
                if t != d:
                    x = term(0.25 * dt, t, T[t, 3 - d - t] if dim == 3 else U[t][d])
                    l, r = l - _sh(x, d, -1), r - x
            l, r = l + 0.5 * dt * _sh(force[d], d, -1), r + 0.5 * dt * force[d]
            v = self.riemann(l, r, w[d])
            if self.lo[d] is not None:
                z = torch.zeros((), dtype=F64, device=DEV)
                v = torch.where(self.lo[d], _mn(r, z), torch.where(self.hi[d], _mx(l, z), v))
            um.append(self.refill(v if w0[d] is None else v + w0[d], d))
        return tr, um


def _box_faces(a, g, boxes, d, ng, dim):
    """Box pieces of a d-face array (..., z, y, x) with g ghosts, grown by ng."""
    out = []
    for lo, hi in boxes:
        sl = [slice(lo[q] - ng + g, hi[q] + 1 + ng + (q == d) + g) if q < dim else slice(0, 1)
              for q in (2, 1, 0)]
        out.append(a[(Ellipsis,) + tuple(sl)])
    return out


def _ghost_faces(faces, g, boxes, n, dim, per):
    """faces[d] cut into boxes with one ghost face.  Beyond the (one) pair of
    outflow sides the ghosts are those of the face fill, which runs over the
    cells of the grown box: a last ghost face along its own direction stays
    unset (zero) there."""
    out = []
    t = dim - 1
    for d in range(dim):
        out.append([])
        for lo, hi in boxes:
            a = _box_faces(faces[d], g, [(lo, hi)], d, 1, dim)[0].clone()[None]
            if d != t:
                last = a.select(3 - d, a.shape[3 - d] - 1)
                ax = [q for q in (2, 1, 0) if q != d].index(t) + 1
                if lo[t] == 0:
                    last.select(ax, 0).zero_()
                if hi[t] == n[t] - 1:
                    last.select(ax, last.shape[ax] - 1).zero_()
            out[d].append(a)
    return out


def _exact_pass(case, seed):
    n, dim, h, geom, per, F, dt, eps = _pass_setup(case, seed)
    boxes = _boxes(case)
    G = Ref(n, dim, per, h, dt, eps, case["ppm"])
    g = G.g
    idx = F.index([-g] * 3, [n[d] - 1 + g for d in range(3)])
    fidx = [torch.arange(-g, n[d] + g, device=DEV) if d < dim else idx[d] for d in range(3)]
    u, w0c = F.velocity(idx), F.w0_cart(idx)
    base = {k: v.to(DEV) for k, v in F.base().items()}

    def col(name, edge):
        """A planar base-state row along the vertical direction."""
        i = torch.arange(-g, n[dim - 1] + g, device=DEV).clamp(0, n[dim - 1] - (not edge))
        shp = [1, 1, 1]
        shp[3 - dim] = len(i)
        return base[name][i].view(shp)

    vert = dim - 1
    if case["sph"]:
        w = w0 = [F.face(fidx, d, "w0mac")[0] for d in range(3)]
    else:
        w = [w0c[d] if d == vert else None for d in range(dim)]
        w0 = [col("w0", True) if d == vert else None for d in range(dim)]
    tr, um = G.velocities(u, u + w0c, F.vel_force(idx), w, w0)
    out = {}
    if not case["sph"]:
        out = dict(utrans=_ghost_faces(tr, g, boxes, n, dim, per),
                   umac=_ghost_faces(um, g, boxes, n, dim, per))
    del tr
    s, f = F.scalars(idx), F.scal_force(idx)
    nscal = s.shape[0]
    spec = list(range(4, nscal))
    zero = [[torch.zeros(nscal, *x.shape, dtype=F64, device=DEV)
             for x in _box_faces(um[0], g, boxes, d, 0, dim)] for d in range(dim)]
    out["sedge"] = zero
    out["sflux"] = [[torch.zeros_like(x) for x in z] for z in zero]
    eta = torch.zeros_like(um[0])

    def put(name, d, c, a):
        for dst, src in zip(out[name][d], _box_faces(a, g, boxes, d, 0, dim)):
            dst[c] = src

    se_rho = G.edge(s[0], f[0], um)
    for d in range(dim):
        put("sedge", d, 0, se_rho[d])
        if case["sph"]:
            r0 = F.face(fidx, d, "r0mac")[0]
            se_rho[d] = (0.5 * r0 + 0.5 * r0) + se_rho[d]
        else:
            se_rho[d] = col("rho0_edge" if d == vert else "rho0", d == vert) + se_rho[d]
    se = G.edge(s[1], f[1], um)
    for d in range(dim):
        put("sedge", d, 1, se[d])
        if case["sph"]:
            b0 = F.face(fidx, d, "r0mac")[0] * F.face(fidx, d, "h0mac")[0]
        else:
            b0 = col("rhoh0_edge" if d == vert else "rhoh0", d == vert)
        put("sflux", d, 1, um[d] * (b0 + se[d]))
    tot = [torch.zeros_like(um[0]) for _ in range(dim)]
    for c in spec:
        se = G.edge(s[c], f[c], um)
        for d in range(dim):
            put("sedge", d, c, se[d])
            fl = um[d] * se_rho[d] * se[d]
            put("sflux", d, c, fl)
            tot[d] += fl
            if d == vert and not case["sph"]:
                eta += fl
    if not case["sph"]:
        eta -= col("w0", True) * col("rho0_predicted_edge", True)
    for d in range(dim):
        put("sflux", d, 0, tot[d])
    out["etarhoflux"] = []
    for b, e in enumerate(_box_faces(eta, g, boxes, vert, 0, dim)):
        pad = [1, 1, 1, 1, 1, 1] if dim == 3 else [1, 1, 1, 1, 0, 0]
        out["etarhoflux"].append(torch.nn.functional.pad(e[None], pad))
    return {k: _pack(v) if k == "etarhoflux" else [_pack(x) for x in v] for k, v in out.items()}


def _exact_cons(case, seed):
    n = _edges(case)
    h = 1.0 / max(n)
    _, per = _geom(n, 3, False, h)
    F = Fields(n, 3, per, h, case["nspec"], False, seed)
    boxes = _boxes(case)
    G = Ref(n, 3, per, h, 0.5 * h / F.umax, 1e-8 * F.umax, case["ppm"])
    g = G.g
    idx = F.index([-g] * 3, [n[d] - 1 + g for d in range(3)])
    u, w0c = F.velocity(idx), F.w0_cart(idx)
    L, R = G.vel_states(u, u + w0c)
    um = []
    for d in range(3):
        l, r = G.outflow(d, L[d][d], R[d][d], normal=True)
        um.append(G.refill(G.riemann(l, r, w0c[d] if d == 2 else None), d))
    del L, R, u, w0c
    s, f = F.scalars(idx), F.scal_force(idx)
    out = [[torch.zeros(s.shape[0], *x.shape, dtype=F64, device=DEV)
            for x in _box_faces(um[0], g, boxes, d, 0, 3)] for d in range(3)]
    for c in range(4, s.shape[0]):
        se = G.edge(s[c], f[c], um, cons=True)
        for d in range(3):
            for dst, src in zip(out[d], _box_faces(se[d], g, boxes, d, 0, 3)):
                dst[c] = src
    return [_pack(x) for x in out]


def _exact_grad(n, per, nc, ppm, seed):
    """(snew, sbar, ubar) dense, one component at a time."""
    s, u, gb, dt, eps = _step_inputs(n, per, nc, seed)
    G = Ref(n, 3, per, [1.0 / q for q in n], dt, eps, ppm)
    g = G.g

    def pad(a, face=-1):
        if g == 0:
            return a
        for d in range(3):
            i = torch.arange(-g, n[d] + g, device=DEV)
            i = i % n[d] if per[d] else i.clamp(0, n[d] - 1 + (d == face))
            a = a.index_select(2 - d, i)
        return a

    u = [x.requires_grad_() for x in u]
    snew, sbar, ubar = torch.empty_like(s), torch.empty_like(s), [0.0] * 3
    inner = tuple(slice(g, g + n[d]) for d in (2, 1, 0))
    for c in range(nc):
        sc = s[c].clone().requires_grad_()
        um = [pad(u[d], d) for d in range(3)]
        sp = pad(sc)
        se = G.edge(sp, None, um)
        div = 0.0
        for d in range(3):
            fl = um[d] * se[d]
            div = div + (_sh(fl, d, 1) - fl) / G.h[d]
        new = (sp + dt * -div)[inner]
        gr = torch.autograd.grad(new, [sc, *u], gb[c])
        snew[c], sbar[c] = new.detach(), gr[0]
        ubar = [ubar[d] + gr[1 + d] for d in range(3)]
    return snew, sbar, ubar


def _exact_step(case, seed):
    snew, sbar, ubar = _exact_grad([case["n"]] * 3, [1, 1, 1], case["nc"], case["ppm"], seed)
    return [snew, sbar, *ubar]


def _exact_boxstep(case, seed):
    n, per = _edges(case), [1, 1, 0]
    boxes = _boxes(case)
    snew, sbar, ubar = _exact_grad(n, per, case["nc"], case["ppm"], seed)

    def cells(a):
        return [a[(slice(None),) + tuple(slice(lo[q], hi[q] + 1) for q in (2, 1, 0))]
                for lo, hi in boxes]

    faces = []
    for d in range(3):
        a = ubar[d]
        if per[d]:  # face n is face 0
            a = torch.cat([a, a.narrow(2 - d, 0, 1)], 2 - d)
        faces.append([x[None] for x in _box_faces(a, 0, boxes, d, 0, 3)])
    return [cells(snew), cells(sbar), faces]


def _exact_update(case, seed):
    n = _edges(case)
    h = 1.0 / max(n)
    dt, ns, cut = 0.05 * h, case["nspec"], 1e-3
    f = _update_fields(case, seed, _boxes(case), mx.device_backend(DEV))
    snew, unew = [], []

    def diff(a, d):
        m = a.shape[a.dim() - 1 - d] - 1
        return a.narrow(a.dim() - 1 - d, 1, m) - a.narrow(a.dim() - 1 - d, 0, m)

    for b in range(len(f["sold"].arrays)):
        so, fo = f["sold"].arrays[b], f["force"].arrays[b]
        div = sum(diff(f["sflux"][d].arrays[b], d) / h for d in range(3))
        upd = so + dt * (-div + fo)
        sn = torch.zeros_like(so)
        sn[1], sn[4:] = upd[1], upd[4:]
        rho = so[0].clone()
        for c in range(4, 4 + ns):
            rho += sn[c] - so[c]
        low = rho < 0.5 * cut
        sn[4:] *= torch.where(low, 0.5 * cut / rho, 1.0)
        sn[0] = torch.where(low, 0.5 * cut, rho)
        snew.append(sn)  # no partial density turns negative: |dt div| < 0.2
        uo, vf, w0 = f["uold"].arrays[b], f["vforce"].arrays[b], f["w0c"].arrays[b]
        grad = [diff(f["uedge"][d].arrays[b], d) / h for d in range(3)]
        bar = []
        for d in range(3):
            a = f["umac"][d].arrays[b]
            m = a.shape[3 - d] - 1
            bar.append(0.5 * (a.narrow(3 - d, 0, m) + a.narrow(3 - d, 1, m)))
        un = uo - dt * sum(bar[d] * grad[d] for d in range(3)) + dt * vf
        c = w0[2, :, 1:-1, 1:-1]
        unew.append(un - dt * (0.5 * (c[1:-1] + c[2:])) * grad[2])
    return [_pack(snew), _pack(unew)]


def _exact_fill(case, seed):
    n = _edges(case)
    _, per = _geom(n, 3, False, 1.0 / max(n))
    nc = 4 + case["nspec"]
    F = Fields(n, 3, per, 1.0 / max(n), nc, False, seed)
    out = []
    for lo, hi in _boxes(case):
        idx = F.index([lo[d] - NG for d in range(3)], [hi[d] + NG for d in range(3)])
        a = torch.stack([F.hash01(idx, c) for c in range(nc)])
        for side in ((slice(0, NG) if lo[2] == 0 else None),
                     (slice(-NG, None) if hi[2] == n[2] - 1 else None)):
            if side is not None:
                a[3, side] = 0.0  # Pi is zero beyond an outflow side
        out.append(a)
    return _pack(out)


def exact(case, seed):
    """`run`'s outputs in plain torch; None for the hierarchy, whose hundreds
    of coarse-fine ghost regions would take plain torch minutes."""
    fn = dict(cons=_exact_cons, step=_exact_step, boxstep=_exact_boxstep, update=_exact_update,
              fill=_exact_fill)
    if case["kind"] == "levels":
        return None
    with torch.no_grad() if case["kind"] not in ("step", "boxstep") else torch.enable_grad():
        return fn.get(case["kind"], _exact_pass)(case, seed)
