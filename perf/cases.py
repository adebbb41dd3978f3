"""Performance cases: the calls a program makes of this library, over the range of sizes it makes them with.

Four kinds of case:

- ``step``     one time step of a device-resident case (``DeviceCase.step``), the call a Python program or a
               serving loop repeats: bubbles (periodic x/y, walls in z), a walled box, THINC/QQ droplets;
- ``batch``    one time step of several same-shaped cases together (``CaseBatch.step``);
- ``routines`` one time step of a main program that calls the library routine by routine, as the Fortran
               modules' ``main.f90`` does (transport, boundary conditions, normals, momentum, projection, checks);
- ``poisson``  standalone pressure solves: one (``fz_solver``), several together (``fz_solver_batched``), or one in
               mixed precision with refinement (``fz_solver_mixed``).

``prepare`` makes what such a program holds before the call (a case in the middle of its run, a context with its
solver set up, the right-hand sides); ``run`` makes one call and returns the library's own device buffers as tensors.
"""
import ctypes as C
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cans-fizzy_amd"))

import fizzy_amd as F  # noqa: E402
from fizzy_amd import cases as fc  # noqa: E402
from fizzy_amd import serve  # noqa: E402

STEPS_BEFORE = 12  # steps taken in prepare: past the first step's Euler start and one check of the time step
FIELDS = ("u", "v", "w", "p", "psi")


def listed():
    return [
        # the smallest request of the serving mix: a 2-D bubble, where launches and latency are all there is
        dict(name="bubble2d_64", kind="step", flow="bubble2d", nx=64, ny=2, nz=64, precision="fp64", graphs=True),
        # an ensemble of small same-shaped requests, stepped together
        dict(name="ensemble_8x128x2x128", kind="batch", flow="bubble2d", nx=128, ny=2, nz=128, count=8,
             precision="fp64"),
        # the plain rising bubble at the size of the example that a user runs first
        dict(name="bubble_64x64x128", kind="step", flow="bubble", nx=64, ny=64, nz=128, precision="fp64",
             graphs=True),
        # the largest request of the serving mix, in mixed precision with one refinement
        dict(name="bubble_128x128x256_mixed", kind="step", flow="bubble", nx=128, ny=128, nz=256,
             precision="mixed", refine=1, graphs=True),
        # the flagship run: density ratio 1000 at 256x256x512, replayed from step graphs
        dict(name="bubble_256x256x512", kind="step", flow="bubble", nx=256, ny=256, nz=512, precision="fp64",
             graphs=True),
        # a box with walls in x and z whose sides are no powers of two, stepped without graphs
        dict(name="walls_90x75x130", kind="step", flow="walls", nx=90, ny=75, nz=130, precision="fp64",
             graphs=False),
        # THINC/QQ droplets in forced turbulence, triply periodic
        dict(name="droplets_256", kind="step", flow="droplets", nx=256, ny=256, nz=256, precision="fp64",
             graphs=False),
        # a main program over the drop-in routines, an ordinary production size
        dict(name="routines_128x128x256", kind="routines", nx=128, ny=128, nz=256),
        # the standalone pressure solve at its largest
        dict(name="poisson_512", kind="poisson", nx=512, ny=512, nz=512, cbc="PPPPNN", count=1, mode="fp64"),
        # small pressure solves of an ensemble, all in one call
        dict(name="poisson_16x64", kind="poisson", nx=64, ny=64, nz=64, cbc="PPPPNN", count=16, mode="batched"),
        # a solve with an outlet, in FP32 with FP64 refinement to 1e-12
        dict(name="poisson_256_mixed", kind="poisson", nx=256, ny=256, nz=256, cbc="PPPPND", count=1, mode="mixed"),
        # cosine transforms of lengths that are no powers of two, an outlet in z
        dict(name="poisson_150x98x126", kind="poisson", nx=150, ny=98, nz=126, cbc="NNNNND", count=1, mode="fp64"),
    ]


MOST_CELLS = {"step": 12e6, "batch": 2e6, "routines": 6e6, "poisson": 30e6}


def _length(rng, lo, hi):
    """A line length with no prime factor above 13, spread over the logarithm of [lo, hi]."""
    while True:
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        m = n
        for p in (2, 3, 5, 7, 11, 13):
            while m % p == 0:
                m //= p
        if m == 1:
            return n


def _any(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["step", "step", "step", "batch", "routines", "poisson", "poisson"])
        c = dict(kind=kind)
        if kind == "step":
            c["flow"] = rng.choice(["bubble2d", "bubble", "bubble", "walls", "droplets"])
            two_d = c["flow"] == "bubble2d"
            # power-of-two boxes are the ordinary choice; any other length is taken as often
            if rng.random() < 0.5:
                c["nx"] = 2 ** rng.randint(5, 8)
                c["ny"] = 2 if two_d else 2 ** rng.randint(5, 8)
            else:
                c["nx"] = _length(rng, 32, 320)
                c["ny"] = 2 if two_d else _length(rng, 24, 320)
            c["nz"] = _any(rng, 32, 512)
            mode = rng.choice(["fp64", "fp64", "fp64", "mixed", "mixed_fp64_projection"])
            c["precision"] = "fp64" if mode == "fp64" else "mixed"
            if mode != "fp64":
                c["refine"] = 1 if mode == "mixed" else -1
            c["graphs"] = rng.random() < 0.5
        elif kind == "batch":
            n = rng.choice([32, 48, 64, 96, 128, 160, 256])
            two_d = rng.random() < 0.7
            c.update(flow="bubble2d" if two_d else "bubble", nx=n, ny=2 if two_d else rng.choice([32, 40, 64]),
                     nz=_any(rng, 32, 160), count=rng.randint(2, 12), precision="fp64")
        elif kind == "routines":
            c.update(nx=_length(rng, 32, 256), ny=_length(rng, 32, 256), nz=_any(rng, 32, 384))
        else:
            c.update(nx=_length(rng, 16, 512), ny=_length(rng, 16, 512), nz=_any(rng, 16, 512),
                     cbc=rng.choice(["PPPPNN", "PPPPPP", "NNNNND", "NNPPNN", "PPNNDD", "DDPPND"]), count=1)
            c["mode"] = rng.choice(["fp64", "fp64", "mixed", "batched"])
            if c["mode"] == "batched":
                c["count"] = rng.randint(2, 16)
                if c["cbc"] == "PPPPPP":  # batched solves take no periodic z
                    c["cbc"] = "PPPPNN"
        if c["nx"] * c["ny"] * c["nz"] * c.get("count", 1) <= MOST_CELLS[kind]:
            return c


# ---------------------------------------------------------------------------
# device buffers as tensors
# ---------------------------------------------------------------------------
class _Buffer:
    """A buffer of the library for torch; keeps its owner alive as long as a tensor over it is."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(int(ptr), False), version=2)


def _tensor(owner, ptr, n, f32=False):
    """The halo'd field at ptr, indexed (z, y, x): the library's arrays run fastest in x."""
    shape = (n[2] + 2, n[1] + 2, n[0] + 2)
    return torch.as_tensor(_Buffer(owner, ptr, shape, "<f4" if f32 else "<f8"), device="cuda")


class _CaseFields:
    """The fields of a DeviceCase as tensors; the time step rotates some of them between two buffers."""

    def __init__(self, case):
        self.case, self.seen = case, {}

    def get(self, name):
        ptr, _ = self.case.field_ptr(name)
        t = self.seen.get((name, ptr))
        if t is None:
            f32 = self.case.field_dtype(name).__name__ == "float32"
            t = self.seen[(name, ptr)] = _tensor(self.case, ptr, self.case.n, f32)
        return t


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _spec(case, rng):
    """The case dictionary of one run: geometry and fluids from the seed."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    flow = case["flow"]
    ratio = rng.uniform(2.0, 1000.0)
    if flow == "bubble2d":
        spec = serve.bubble_case(nx, two_d=True, density_ratio=ratio)
        spec.update(ng=[nx, 2, nz], l=[1.0, 2.0 / nx, nz / nx],
                    spheres=[(rng.uniform(0.4, 0.6), 1.0 / nx, 0.5 * nz / nx, rng.uniform(0.15, 0.25) * min(1.0, nz / nx))])
    elif flow == "bubble":
        spec = fc.rising_bubble_3d(ng=(nx, ny, nz), rho12=(ratio, 1.0), mu12=(10.0, 1.0))
        spec["l"] = [1.0, ny / nx, nz / nx]
        small = min(spec["l"])
        spec["spheres"] = [(rng.uniform(0.4, 0.6), spec["l"][1] * rng.uniform(0.4, 0.6),
                            spec["l"][2] * rng.uniform(0.3, 0.5), small * rng.uniform(0.2, 0.3))]
    elif flow == "walls":
        spec = fc.rising_bubble_3d(ng=(nx, ny, nz), rho12=(ratio, 1.0), mu12=(10.0, 1.0))
        spec["l"] = [1.0, ny / nx, nz / nx]
        small = min(spec["l"])
        spec["spheres"] = [(rng.uniform(0.4, 0.6), 0.5 * spec["l"][1], spec["l"][2] * rng.uniform(0.35, 0.5),
                            small * rng.uniform(0.2, 0.3))]
        spec["cbcvel"] = fc.bc3("DD", "PP", "DD") + fc.bc3("NN", "PP", "DD") + fc.bc3("NN", "PP", "DD")
        spec["cbcpre"] = fc.bc3("NN", "PP", "NN")
        spec["cbcpsi"] = fc.bc3("NN", "PP", "NN")
        spec["cbcnor"] = fc.bc3("DD", "PP", "NN") + fc.bc3("NN", "PP", "NN") + fc.bc3("NN", "PP", "DD")
    else:
        lx = 2.0 * math.pi
        box = [lx, lx * ny / nx, lx * nz / nx]
        spec = fc.vof_droplets(ng=(nx, ny, nz), ndrop=1, r=0.3, sigma=0.12)
        r = 0.15 * min(box)
        count = 8
        spec.update(l=box, spheres=[(rng.uniform(0.0, box[0]), rng.uniform(0.0, box[1]), rng.uniform(0.0, box[2]), r)
                                    for _ in range(count)])
    spec["precision"] = case["precision"]
    if "refine" in case:
        spec["refine"] = case["refine"]
    return spec


def _set_flow(n, l, fields, rng, amplitude):
    """A smooth flow of a few modes in u, v, w (zero on the planes z = 0 and z = l[2])."""
    dev = fields[0].device
    x = [(torch.arange(n[d] + 2, device=dev, dtype=torch.float64) - 0.5) / n[d] for d in range(3)]
    z = torch.sin(2.0 * math.pi * x[2])[:, None, None]
    for d, f in enumerate(fields):
        f.zero_()
        for _ in range(3):
            kx, ky = rng.randint(1, 3), (0 if n[1] <= 2 else rng.randint(1, 3))
            a, px, py = rng.uniform(-1.0, 1.0), rng.uniform(0.0, 1.0), rng.uniform(0.0, 1.0)
            if d == 1 and n[1] <= 2:
                a = 0.0
            wave = torch.sin(2 * math.pi * (kx * x[0] + px))[None, None, :] * \
                torch.cos(2 * math.pi * (ky * x[1] + py))[None, :, None]
            f.add_(wave * z, alpha=amplitude * a)


def _bc(v):
    return (C.c_double * len(v))(*v)


def _started_case(case, seed):
    """A case in the middle of its run: a seeded bubble in a seeded flow, a few steps on."""
    rng = random.Random(seed)
    spec = _spec(case, rng)
    dc = F.DeviceCase(spec)
    dc.init()
    fields = _CaseFields(dc)
    uvw = [fields.get(q) for q in ("u", "v", "w")]
    _set_flow(dc.n, spec["l"], uvw, rng, 0.05 if spec["vof"] else 0.02)
    torch.cuda.synchronize()
    F.call("fz_bounduvw", dc.ctx, "".join(spec["cbcvel"]).encode(), _bc([0.0] * 18), 0, *[C.c_void_p(t.data_ptr())
                                                                                        for t in uvw])
    if case.get("graphs"):
        dc.set_graphs(True)
    dc.step(STEPS_BEFORE)
    dc.sync()
    return dc, fields


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        dc, fields = _started_case(case, seed)
        return dict(kind=kind, case=dc, fields=fields)
    if kind == "batch":
        made = [_started_case(case, 1000 * seed + q) for q in range(case["count"])]
        return dict(kind=kind, batch=F.cases.CaseBatch([dc for dc, _ in made]), fields=[f for _, f in made])
    if kind == "routines":
        prog = _Program(case, seed)
        for _ in range(STEPS_BEFORE):
            prog.step()
        prog.ctx.sync()
        return dict(kind=kind, prog=prog)
    n = [case["nx"], case["ny"], case["nz"]]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ctxs, rhs, sol = [], [], []
    for _ in range(case["count"]):
        ctx = F.Context(n, [1.0, 1.0, 1.0], case["cbc"])
        F.call("fz_initsolver", ctx.h, None, None, None, None, None, None, None, None, None)
        b, x = ctx.halo(), ctx.halo()
        tb, tx = _tensor(ctx, b.ptr.value, n), _tensor(ctx, x.ptr.value, n)
        tb.zero_()
        tx.zero_()
        tb[1:-1, 1:-1, 1:-1] = _rhs(n, case["cbc"], gen)
        ctxs.append(ctx)
        rhs.append(b)
        sol.append((x, tx))
    torch.cuda.synchronize()
    s = dict(kind=kind, mode=case["mode"], ctxs=ctxs, rhs=rhs, sol=sol)
    k = case["count"]
    s["handles"] = (C.c_void_p * k)(*[c.h.value for c in ctxs])
    s["ptrs"] = (C.c_void_p * k)(*[x.ptr.value for x, _ in sol])
    return s


def _rhs(n, cbc, gen):
    """A right-hand side uniform in [-1, 1], indexed (z, y, x); of a singular operator, with its mean taken out."""
    f = torch.rand((n[2], n[1], n[0]), generator=gen, device="cuda", dtype=torch.float64) * 2.0 - 1.0
    if "D" not in cbc:
        dz = _faces(n[2]).diff().to(f.device)[:, None, None]
        f -= (f * dz).sum() / (dz.sum() * n[0] * n[1])
    return f


def run(state):
    kind = state["kind"]
    if kind == "step":
        state["case"].step(1)
        return {q: state["fields"].get(q) for q in FIELDS}
    if kind == "batch":
        state["batch"].step(1)
        return [{q: f.get(q) for q in FIELDS} for f in state["fields"]]
    if kind == "routines":
        return state["prog"].step()
    for ctx, b, (x, _) in zip(state["ctxs"], state["rhs"], state["sol"]):
        F.call("fz_copy", ctx.h, x.ptr, b.ptr, C.c_size_t(b.nbytes))
    if state["mode"] == "batched":
        F.call("fz_solver_batched", state["handles"], state["ptrs"], len(state["ctxs"]))
    elif state["mode"] == "mixed":
        F.call("fz_solver_mixed", state["ctxs"][0].h, state["sol"][0][0].ptr, 1e-12, 10, C.byref(C.c_int()), None)
    else:
        F.call("fz_solver", state["ctxs"][0].h, state["sol"][0][0].ptr)
    return [t[1:-1, 1:-1, 1:-1] for _, t in state["sol"]]  # the solution; the halo is the next boundp's


class _Program:
    """A main program that holds the fields itself and calls the library routine by routine: the rising bubble
    (periodic x/y, no-slip walls in z), in the order and with the arguments of the reference's time loop
    (src/main.f90:414-562)."""

    def __init__(self, case, seed):
        rng = random.Random(seed)
        n = [case["nx"], case["ny"], case["nz"]]
        l = [1.0, n[1] / n[0], n[2] / n[0]]
        self.ctx = c = F.Context(n, l, "PPPPNN")
        F.call("fz_initsolver", c.h, _bc([0.0] * 6), None, None, None, None, None, None, None, None)
        self.cbcvel, self.cbcpre = b"PPPPDD" * 3, b"PPPPNN"
        self.cbcnor = (b"PPPPNN", b"PPPPNN", b"PPPPDD")
        self.zero6, self.zero18 = _bc([0.0] * 6), _bc([0.0] * 18)
        ratio = rng.uniform(2.0, 1000.0)
        self.rho12, self.mu12, self.beta12 = _bc([ratio, 1.0]), _bc([10.0, 1.0]), _bc([1.0, 1.0])
        self.rho0, self.sigma = 1.0, 24.5
        self.gacc, self.bforce, self.rho_av = _bc([0.0, 0.0, -0.98]), _bc([0.0] * 3), _bc([0.0] * 3)
        self.a, self.t = {}, {}
        for q in ("u", "v", "w", "p", "pp", "pn", "po", "psi", "psio", "phi", "kappa", "nx", "ny", "nz", "fx", "fy",
                  "fz"):
            self.a[q] = c.halo()
            self.t[q] = _tensor(c, self.a[q].ptr.value, n)
            self.t[q].zero_()
        self.nbytes = C.c_size_t(self.a["u"].nbytes)
        st = C.c_void_p()
        F.call("fz_rk_state_create", c.h, C.byref(st))
        self.rk = _Handle(st, c)
        seps = C.c_double()
        F.call("fz_acdi_set_epsilon", c.h, 1.0, C.byref(seps))
        self.seps = seps.value
        # psi of one sphere, as the initial condition gives it, and a seeded flow
        dev = self.t["u"].device
        x = [(torch.arange(n[d] + 2, device=dev, dtype=torch.float64) - 0.5) * (l[d] / n[d]) for d in range(3)]
        cen = [l[0] * rng.uniform(0.4, 0.6), l[1] * rng.uniform(0.4, 0.6), l[2] * rng.uniform(0.3, 0.5)]
        dist = torch.sqrt((x[0] - cen[0])[None, None, :] ** 2 + (x[1] - cen[1])[None, :, None] ** 2 +
                          (x[2] - cen[2])[:, None, None] ** 2) - min(l) * rng.uniform(0.2, 0.3)
        self.t["psi"].copy_(0.5 * (1.0 + torch.tanh(dist / (2.0 * self.seps))))
        _set_flow(n, l, [self.t[q] for q in "uvw"], rng, 0.02)
        torch.cuda.synchronize()
        self.bounduvw("u", "v", "w")
        self.boundp(self.cbcpre, "psi")
        self.geometry()
        self.gamma()
        self.istep = 0
        self.dt = self.dto = self.new_dt()

    def call(self, name, *args):
        F.call(name, self.ctx.h, *[self.a[x].ptr if isinstance(x, str) else x for x in args])

    def copy(self, dst, src):
        self.call("fz_copy", dst, src, self.nbytes)

    def boundp(self, cbc, f):
        self.call("fz_boundp", cbc, self.zero6, f)

    def bounduvw(self, u, v, w, is_correc=0):
        self.call("fz_bounduvw", self.cbcvel, self.zero18, is_correc, u, v, w)

    def geometry(self):
        self.call("fz_acdi_cmpt_phi", self.seps, "psi", "phi")
        self.call("fz_cmpt_norm_curv_youngs", "phi", "nx", "ny", "nz", "kappa")
        self.boundp(self.cbcpre, "kappa")
        for cbc, f in zip(self.cbcnor, ("nx", "ny", "nz")):
            self.boundp(cbc, f)

    def gamma(self):
        g = C.c_double()
        self.call("fz_acdi_set_gamma", 1.0, "u", "v", "w", C.byref(g))
        self.gam = max(g.value, 1e-12)

    def new_dt(self):
        d = C.c_double()
        self.call("fz_chkdt", 1, 1, 0, self.mu12, self.rho12, self.sigma, self.gacc, "u", "v", "w", self.gam,
                  self.seps, C.byref(d))
        return 0.25 * d.value

    def step(self):
        dt_r = self.dt / self.dto
        tm = _bc([1.0 + 0.5 * dt_r, -0.5 * dt_r])
        self.copy("psio", "psi")
        self.call("fz_rk_2fl", self.rk.h, tm, self.dt, self.gam, self.seps, 0.0, 0, "u", "v", "w", "nx", "ny", "nz",
                  "phi", "psi", "fx", "fy", "fz")
        self.bounduvw("fx", "fy", "fz")
        self.boundp(self.cbcpre, "psi")
        self.geometry()
        self.call("fz_rk", self.rk.h, tm, self.dt, dt_r, self.bforce, self.gacc, self.sigma, self.rho_av, self.rho12,
                  self.mu12, self.beta12, self.rho0, "psi", "kappa", "p", "pn", "po", "psio", "fx", "fy", "fz", "u",
                  "v", "w")
        self.bounduvw("u", "v", "w")
        self.copy("pp", "p")
        self.call("fz_fillps", 1.0 / self.dt, self.rho0, "u", "v", "w", "p")
        self.call("fz_updt_rhs_b", "p")
        self.call("fz_solver", "p")
        self.boundp(self.cbcpre, "p")
        self.call("fz_correc", self.rho0, self.rho12, self.dt, "p", "psi", "u", "v", "w")
        self.bounduvw("u", "v", "w", 1)
        self.call("fz_updatep", "pp", "p")
        self.boundp(self.cbcpre, "p")
        self.copy("po", "pn")
        self.copy("pn", "p")
        self.dto = self.dt
        self.gamma()
        self.istep += 1
        if self.istep % 10 == 0:
            self.dt = self.new_dt()
            tot, top = C.c_double(), C.c_double()
            self.call("fz_chkdiv", "u", "v", "w", C.byref(tot), C.byref(top))
        return {q: self.t[q] for q in FIELDS}


class _Handle:
    """An fz_rk_state, destroyed before its context."""

    def __init__(self, h, ctx):
        self.h, self.ctx = h, ctx

    def __del__(self):
        if self.ctx.h:
            F.lib().fz_rk_state_destroy(self.h)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its exact result
# ---------------------------------------------------------------------------
def work(case):
    cells = case["nx"] * case["ny"] * case["nz"] * case.get("count", 1)
    logs = math.log2(case["nx"]) + math.log2(case["ny"])
    # two real transforms each way per direction (2.5 n log2 n operations a line), about ten operations a row in z
    solve = 5.0 * logs + 10.0
    if case["kind"] == "poisson":
        return dict(bytes=16.0 * cells, flops=solve * cells)
    # in: u, v, w, p, the pressure before, psi and the four histories; out: all but the pressure before
    phase = 4.0 if case.get("precision") == "mixed" else 8.0
    return dict(bytes=(5 + 4) * 8.0 * cells + (5 + 5) * phase * cells, flops=(800.0 + solve) * cells)


def _faces(n):
    """The face coordinates of a uniform unit box, whose quotient the reference forms in single precision
    (src/initgrid.f90:38)."""
    return (torch.arange(n + 1, dtype=torch.float32) / float(n)).to(torch.float64)


def _second_difference(n, b):
    """The 3-point second difference in x or y on a unit box, its ghost cells by the boundary codes b."""
    m = torch.zeros((n, n), dtype=torch.float64)
    i = torch.arange(n)
    m[i, i] = -2.0
    m[i[:-1], i[1:]] += 1.0
    m[i[1:], i[:-1]] += 1.0
    if b == "PP":
        m[0, n - 1] += 1.0
        m[n - 1, 0] += 1.0
    else:
        for at, code in ((0, b[0]), (n - 1, b[1])):
            m[at, at] += 1.0 if code == "N" else -1.0
    return m * float(n) ** 2


def exact(case, seed):
    """Pressure solves whose operator has an inverse, by dense eigenvectors in x and y and elimination in z. A
    singular one's answer carries a constant that only the solver's own rounding sets, and a time step's carries
    phi = eps*log(psi/(1-psi)) of a psi within rounding of 0 and 1: neither has a value that 64 bits decide."""
    if case["kind"] != "poisson" or "D" not in case["cbc"]:
        return None
    n, cbc = [case["nx"], case["ny"], case["nz"]], case["cbc"]
    if cbc[4:] == "PP" or case["count"] * n[0] * n[1] * n[2] * (n[0] + n[1]) > 4e10:
        return None
    dev = torch.device("cuda")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lx, vx = torch.linalg.eigh(_second_difference(n[0], cbc[0:2]))
    ly, vy = torch.linalg.eigh(_second_difference(n[1], cbc[2:4]))
    lx, vx, ly, vy = lx.to(dev), vx.to(dev), ly.to(dev), vy.to(dev)
    zf = _faces(n[2])
    dzf = torch.cat([zf.diff()[:1], zf.diff(), zf.diff()[-1:]])
    dzc = 0.5 * (dzf[:-1] + dzf[1:])
    a, c = (1.0 / dzf[1:-1] / dzc[:-1]).tolist(), (1.0 / dzf[1:-1] / dzc[1:]).tolist()
    b = [-(p + q) for p, q in zip(a, c)]
    b[0] += a[0] if cbc[4] == "N" else -a[0]
    b[-1] += c[-1] if cbc[5] == "N" else -c[-1]
    lam = ly[:, None] + lx[None, :]
    out = []
    for _ in range(case["count"]):
        f = _rhs(n, cbc, gen)
        f = torch.matmul(vy.T.contiguous(), torch.matmul(f, vx))
        d = []
        for k in range(n[2]):
            z = 1.0 / (b[k] + lam - (a[k] * d[-1] if k else 0.0))
            d.append(c[k] * z)
            f[k] = (f[k] - (a[k] * f[k - 1] if k else 0.0)) * z
        for k in range(n[2] - 2, -1, -1):
            f[k] -= d[k] * f[k + 1]
        out.append(torch.matmul(vy, torch.matmul(f, vx.T.contiguous())))
    return out
