"""Launch shapes chosen from the grid give the fields of any other choice.

The z-marching kernels (momentum, phase-field step, normals) take their
planes per block from the grid; FZ_MARCH_PLANES, read when a context is made,
fixes the number. Every number gives the same fields bit for bit."""
import ctypes as C

import numpy as np
import pytest

import fizzy_amd as F
import oracle as O
from fizzy_amd import cases
from test_gpu_step import compare, load_oracle_from_device

pytestmark = pytest.mark.gpu

FIELDS = ["u", "v", "w", "p", "psi", "kappa"]
BUBBLE = cases.rising_bubble_3d(ng=(72, 20, 40))
SPECS = {"fp64": BUBBLE, "mixed": dict(BUBBLE, precision="mixed", refine=1),
         "two-d": cases.hysing_2d(ng=(32, 2, 33)), "droplets": cases.vof_droplets(ng=(32, 24, 18), ndrop=2, r=0.6)}


def run(spec, nsteps, planes, monkeypatch):
    if planes:
        monkeypatch.setenv("FZ_MARCH_PLANES", str(planes))
    else:
        monkeypatch.delenv("FZ_MARCH_PLANES", raising=False)
    dc = F.DeviceCase(spec)
    try:
        dc.init()
        dc.step(nsteps)
        return {k: dc.get(k) for k in FIELDS}, dc.scalars()
    finally:
        dc.close()


@pytest.mark.parametrize("planes", [1, 3, 16, 64])
@pytest.mark.parametrize("name", list(SPECS))
def test_planes_per_block_agree_bitwise(name, planes, monkeypatch):
    a, sa = run(SPECS[name], 8, 0, monkeypatch)
    b, sb = run(SPECS[name], 8, planes, monkeypatch)
    for k in FIELDS:
        assert np.array_equal(a[k], b[k]), k
    assert np.array_equal(sa, sb)


KINDS = {"R2HC": 0, "HC2R": 1, "REDFT01": 4, "REDFT10": 5, "REDFT11": 6, "RODFT01": 8, "RODFT10": 9, "RODFT11": 10}


@pytest.mark.parametrize("kind", list(KINDS))
def test_line_transforms_of_any_length_bitwise(kind, rng):
    """Every radix, the lengths on both sides of a block's capacity (2560
    complex points), odd line counts and several blocks, against the oracle."""
    ctx = F.Context([4, 4, 4], [1, 1, 1], "PPPPPP")
    try:
        for n, howmany in [(4, 131), (9, 1), (14, 257), (22, 70), (26, 65), (49, 33), (75, 64), (81, 67), (90, 300),
                           (121, 40), (160, 35), (162, 35), (169, 31), (225, 29), (343, 17), (500, 12), (637, 9),
                           (1001, 5), (1000, 3), (1287, 4), (1944, 3), (2002, 2), (2025, 3)]:
            if KINDS[kind] in (6, 10) and 2 * n > 2048:
                continue
            x = rng.standard_normal((howmany, n))
            d = F.DArray(ctx, (n * howmany,))
            d.upload(np.ascontiguousarray(x).reshape(-1))
            F.call("fz_r2r", ctx.h, KINDS[kind], n, howmany, d.ptr)
            got = d.download().reshape(howmany, n)
            d.free()
            assert np.array_equal(got, O.r2r(KINDS[kind], x)), (kind, n, howmany)
    finally:
        ctx.close()


RAGGED = {
    # the right-hand side evaluated in the load of a forward x transform whose length is no power of two
    "bubble_30x18x22": lambda: cases.rising_bubble_3d(ng=(30, 18, 22)),
    # the phase-field step whose waves own 62 cells of the halo'd plane: rows of one wave, rows across waves
    "droplets_60x6x7": lambda: cases.vof_droplets(ng=(60, 6, 7), ndrop=1, r=1.2),
    "droplets_26x9x21": lambda: cases.vof_droplets(ng=(26, 9, 21), ndrop=1, r=1.2),
    "walls_45x14x20": lambda: dict(cases.hysing_2d(ng=(45, 2, 20)), ng=[45, 14, 20], l=[1.0, 14 / 45, 20 / 45]),
}


@pytest.mark.parametrize("graphs", [False, True], ids=["direct", "graphs"])
@pytest.mark.parametrize("name", list(RAGGED))
def test_ragged_steps_match_the_oracle(name, graphs):
    """Steps of boxes whose sides are no powers of two against the oracle's
    from the same state, launched directly and (steps after the first)
    replayed from graphs."""
    spec = RAGGED[name]()
    dc, oc = F.DeviceCase(spec), O.Case(spec)
    try:
        dc.init()
        oc.init_fields()
        dc.set_graphs(graphs)
        for step in range(5):
            load_oracle_from_device(oc, dc)
            assert dc.step(1) == oc.step(1) == 0
            errs = compare(oc, dc)
            assert max(errs.values()) <= 1e-12, (step, errs)
    finally:
        dc.close()


def solve(n, cbc, f, mixed, count=1):
    ctxs = [F.Context(n, [1.0, 0.9, 1.7], cbc, gr=0.6 if cbc[4:] != "PP" else 0.0) for _ in range(count)]
    try:
        ds = []
        for c in ctxs:
            F.call("fz_initsolver", c.h, None, None, None, None, None, None, None, None, None)
            ds.append(c.halo(f))
        if count > 1:
            F.call("fz_solver_batched", (C.c_void_p * count)(*[c.h.value for c in ctxs]),
                   (C.c_void_p * count)(*[d.ptr.value for d in ds]), count)
        elif mixed:
            F.call("fz_solver_mixed", ctxs[0].h, ds[0].ptr, 0.0, 2, C.byref(C.c_int()), None)
        else:
            F.call("fz_solver", ctxs[0].h, ds[0].ptr)
        return ds[-1].download()[1:-1, 1:-1, 1:-1]
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("n3", [2, 3, 15, 16, 17, 32, 33, 64, 65, 127, 255, 256, 257, 258, 511, 512, 513, 1024, 1025])
@pytest.mark.parametrize("cbc", ["PPPPNN", "NNPPDD", "PPPPPP"])
def test_columns_in_registers_match_the_chunked_kernels(n3, cbc, rng, monkeypatch):
    """Both sides of a thread's, a wave's and a block's rows, and column
    counts that are no multiple of a block's, in FP64, mixed precision and
    (non-periodic z) as a batch, against the chunked kernels bit for bit."""
    for n in ([6, 5, n3], [16, 4, n3]):
        f = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n]))
        kinds = [(False, 1), (True, 1)] + ([(False, 3)] if cbc != "PPPPPP" else [])
        for mixed, count in kinds:
            monkeypatch.delenv("FZ_THOMAS_ROWS64", raising=False)
            got = solve(n, cbc, f, mixed, count)
            monkeypatch.setenv("FZ_THOMAS_ROWS64", "16")
            assert np.array_equal(got, solve(n, cbc, f, mixed, count), equal_nan=True), (n, mixed, count)


@pytest.mark.parametrize("n", [[5, 3, 2], [33, 7, 9], [64, 8, 17], [70, 13, 40]], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("vof", [0, 1], ids=["acdi", "thinc"])
def test_integrators_match_their_parts(n, vof, rng):
    """rk and rk_2fl (one pass each and a copy back) against transport,
    momentum terms and clip called by themselves with the AB2 updates of
    src/rk.f90:86-130 and :232-252 between them, over three calls."""
    ctx = F.Context(n, [1.0, 0.9, 1.7], "PPPPNN", gr=0.5)
    try:
        rand = lambda lo=-1.0, hi=1.0: np.asfortranarray(rng.uniform(lo, hi, [x + 2 for x in n]))  # noqa: E731
        h = {q: ctx.halo(rand()) for q in ("u", "v", "w", "nx", "ny", "nz", "phi", "p", "pn", "po", "kappa")}
        h.update(psi=ctx.halo(rand(-0.2, 1.2)), fx=ctx.halo(rand()), fy=ctx.halo(rand()), fz=ctx.halo(rand()))
        h["psio"] = ctx.halo(rand(0.0, 1.0))
        part = {q: ctx.interior() for q in ("r", "du", "dv", "dw", "au", "av", "aw")}
        st = C.c_void_p()
        F.call("fz_rk_state_create", ctx.h, C.byref(st))
        rho12, mu12 = (C.c_double * 2)(50.0, 1.0), (C.c_double * 2)(0.3, 0.02)
        three = [(C.c_double * 3)(*v) for v in ([0.1, 0.0, -0.2], [0.0, 0.3, -0.98], [0.0, 0.5, 3.0])]
        gam, seps, beta, dt, dt_r = 0.7, 0.02, 40.0, 1e-3, 1.2
        tm = (C.c_double * 2)(1.0 + 0.5 * dt_r, -0.5 * dt_r)
        f1, f2 = tm[0] * dt, tm[1] * dt
        inner = (slice(1, -1),) * 3
        hist, vel_hist = None, None
        P = {q: a.ptr for q, a in h.items()}
        for _ in range(3):
            psi = h["psi"].download()
            args = [P[q] for q in ("u", "v", "w", "nx", "ny", "nz", "phi", "psi")]
            name, par = ("fz_vof_thinc_transport_psi", [beta]) if vof else ("fz_acdi_transport_pf", [gam, seps])
            F.call(name, ctx.h, *par, *args, part["r"].ptr, P["fx"], P["fy"], P["fz"])
            flux = [h[q].download() for q in ("fx", "fy", "fz")]
            r = part["r"].download()
            hist = r if hist is None else hist
            ref = psi.copy(order="F")
            ref[inner] = psi[inner] + f1 * r + f2 * hist
            ref = np.minimum(np.maximum(0.0, ref), 1.0)
            hist = r
            F.call("fz_rk_2fl", ctx.h, st, tm, dt, gam, seps, beta, vof, *args, P["fx"], P["fy"], P["fz"])
            assert np.array_equal(h["psi"].download(), ref)
            for q, f in zip(("fx", "fy", "fz"), flux):
                assert np.array_equal(h[q].download()[inner], f[inner]), q
            # momentum
            F.call("fz_mom_xyz_ad", ctx.h, rho12, mu12, P["fx"], P["fy"], P["fz"], P["u"], P["v"], P["w"], P["psi"],
                   part["du"].ptr, part["dv"].ptr, part["dw"].ptr)
            F.call("fz_mom_xyz_oth", ctx.h, dt_r, rho12, rho12, three[0], three[1], 24.5, 1.0, three[2], P["p"],
                   P["psi"], P["kappa"], P["pn"], P["po"], part["au"].ptr, part["av"].ptr, part["aw"].ptr)
            now = [part[q].download() for q in ("du", "dv", "dw")]
            vel_hist = now if vel_hist is None else vel_hist
            pn_, po_ = h["psi"].download(), h["psio"].download()
            refs = []
            for d, q in enumerate("uvw"):
                up = [slice(1, -1)] * 3
                up[d] = slice(2, None)
                up = tuple(up)
                rn = 1.0 + 49.0 * 0.5 * (po_[inner] + po_[up])
                rp = 1.0 + 49.0 * 0.5 * (pn_[inner] + pn_[up])
                a = h[q].download()
                b = a[inner] * rn / rp + (f1 * now[d] + f2 * vel_hist[d]) / rp
                a[inner] = b + (f1 + f2) * part["a" + q].download() / rp
                refs.append(a)
            vel_hist = now
            F.call("fz_rk", ctx.h, st, tm, dt, dt_r, three[0], three[1], 24.5, three[2], rho12, mu12, rho12, 1.0,
                   P["psi"], P["kappa"], P["p"], P["pn"], P["po"], P["psio"], P["fx"], P["fy"], P["fz"], P["u"],
                   P["v"], P["w"])
            for q, a in zip("uvw", refs):
                assert np.array_equal(h[q].download(), a), q
        F.lib().fz_rk_state_destroy(st)
    finally:
        ctx.close()


@pytest.mark.parametrize("n,cbc", [([6, 256, 3], "PPPPDD"), ([70, 512, 2], "PPPPND"), ([33, 1024, 2], "NNNNDD"),
                                   ([20, 2048, 2], "PPDDNN"), ([9, 512, 3], "DDNNDD")],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else v)
def test_long_strided_lines_bitwise(n, cbc, rng):
    """y lines of the sixteen-point transform kernel, every kind it takes and
    line counts that are no multiple of a block's, against the oracle; FP32
    ones against the FP64 solve to the accuracy of their refinement."""
    ctx = F.Context(n, [1.0, 0.9, 1.7], cbc)
    try:
        F.call("fz_initsolver", ctx.h, None, None, None, None, None, None, None, None, None)
        sol = O.Solver(n, ctx.dli, ctx.dzci, ctx.dzfi, list(cbc))
        f = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n]))
        d, m = ctx.halo(f), ctx.halo(f)
        F.call("fz_solver", ctx.h, d.ptr)
        ref = f.copy(order="F")
        sol.solve(ref)
        assert np.array_equal(d.download(), ref)
        rel = C.c_double()
        F.call("fz_solver_mixed", ctx.h, m.ptr, 1e-12, 10, C.byref(C.c_int()), C.byref(rel))
        assert rel.value <= 1e-11
    finally:
        ctx.close()


def test_cases_move_between_batches(monkeypatch):
    """A batch takes its cases onto one stream; cases of an older batch join a
    newer one, the older one goes first or last, a member is destroyed while
    in a batch, and every case's fields stay those of its own steps."""
    specs = [cases.rising_bubble_3d(ng=(16, 8, 12), rho12=(r, 1.0)) for r in (10.0, 50.0, 200.0, 900.0)]

    def start():
        out = []
        for s in specs:
            dc = F.DeviceCase(s)
            dc.init()
            dc.step(1)
            out.append(dc)
        return out

    alone, batched = start(), start()
    try:
        a = cases.CaseBatch(batched[:3])
        a.step(2)
        mid = batched[1].get("psi")  # on the batch's stream, between its steps
        b = cases.CaseBatch(batched[1:])  # led by a member of the first batch
        a.close()
        b.step(3)
        c = cases.CaseBatch([batched[3], batched[0]])
        c.step(2)
        b.close()
        batched[0].step(1)
        c.close()
        steps = [2 + 2 + 1, 2 + 3, 2 + 3, 3 + 2]
        alone[1].step(2)
        assert np.array_equal(mid, alone[1].get("psi"))
        alone[1].step(3)
        for q in (0, 2, 3):
            alone[q].step(steps[q])
        for x, y in zip(alone, batched):
            for k in FIELDS:
                assert np.array_equal(x.get(k), y.get(k)), k
        d = cases.CaseBatch(batched[:2])
        d.step(1)
        d.close()
        e = cases.CaseBatch(batched[1:3])
        batched[2].close()  # a member goes before its batch
        e.close()
        batched[1].step(1)
        batched[1].sync()
    finally:
        for x in alone + batched:
            x.close()


def cavity(n):
    return dict(cases.lid_driven_cavity(), ng=n, l=[x / 10.0 for x in n])


PAIRS = {
    # n1 + 2 cells a row in pairs: rows per wave below and above one, ends of rows at the ends of waves
    "one pair a row": lambda: cases.rising_bubble_3d(ng=(2, 6, 8)),
    "periodic 60": lambda: cases.rising_bubble_3d(ng=(60, 5, 9)),
    "periodic 126": lambda: cases.rising_bubble_3d(ng=(126, 9, 8)),
    "periodic 130": lambda: cases.rising_bubble_3d(ng=(130, 3, 6)),
    "walls 40": lambda: dict(cases.hysing_2d(ng=(40, 2, 12)), ng=[40, 7, 12], l=[1.0, 7 / 40, 12 / 40]),
    "cavity 14": lambda: cavity([14, 9, 11]),
    "droplets 28": lambda: cases.vof_droplets(ng=(28, 24, 18), ndrop=2, r=0.6),
    "mixed 78": lambda: dict(cases.rising_bubble_3d(ng=(78, 6, 10)), precision="mixed", refine=1),
}


@pytest.mark.parametrize("name", list(PAIRS))
def test_correction_in_pairs_matches_the_tiled_kernel(name, rng, monkeypatch):
    """The correction of rows of even length, pairs of cells a lane, against
    the LDS kernel's on whole fields, halos included, from a pressure whose
    halo is not its boundary condition's; alone, and for some as a batch."""
    out = []
    spec = PAIRS[name]()
    n = spec["ng"]
    dp = rng.uniform(-1e-3, 1e-3, [x + 2 for x in n])
    for tiled in (False, True):
        monkeypatch.delenv("FZ_CORREC_MY", raising=False)
        if tiled:
            monkeypatch.setenv("FZ_CORREC_MY", "4")
        dcs = [F.DeviceCase(spec) for _ in range(3)]
        try:
            for q, dc in enumerate(dcs):
                dc.init()
                dc.step(1)
                dc.set("p", dc.get("p") + (q + 1) * dp)
            dcs[0].step(3)
            if name.startswith(("periodic", "walls")):
                b = cases.CaseBatch(dcs[1:])
                b.step(3)
                b.close()
            out.append([(dc.get(k), k) for dc in dcs for k in ("u", "v", "w", "p", "psi")] + [(dcs[0].scalars(), "s")])
        finally:
            for dc in dcs:
                dc.close()
    for (a, k), (b, _) in zip(*out):
        assert np.array_equal(a, b, equal_nan=True), k


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [[33, 1, 9], [40, 2, 33], [130, 2, 20], [65, 3, 12]],
                         ids=lambda n: "x".join(map(str, n)))
def test_tiles_of_thin_boxes_match_the_plain_kernels(n, precision, monkeypatch):
    """Boxes of one and two rows take momentum and ACDI tiles of two rows (three
    rows do not): the plain kernels' fields bit for bit, and a batch's as its
    cases' alone."""
    spec = dict(cases.hysing_2d(ng=tuple(n)), precision=precision, refine=-1)

    def start(count):
        out = [F.DeviceCase(dict(spec, sigma=24.5 * (q + 1))) for q in range(count)]
        for dc in out:
            dc.init()
            dc.step(1)
        return out

    tiled, batched = start(2), start(2)
    monkeypatch.setenv("FZ_MOM_WPE", "2")
    monkeypatch.setenv("FZ_ACDI_VARIANT", "2")
    plain = start(2)
    try:
        b = cases.CaseBatch(batched)
        b.step(5)
        b.close()
        for t, p, q in zip(tiled, plain, batched):
            t.step(5)
            p.step(5)
            for k in FIELDS:
                assert np.array_equal(t.get(k), p.get(k)), k
                assert np.array_equal(t.get(k), q.get(k)), k
    finally:
        for dc in tiled + batched + plain:
            dc.close()


@pytest.mark.parametrize("n", [[5, 3, 2], [33, 7, 9], [60, 5, 6], [65, 4, 33], [96, 6, 7]],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("walls", [False, True], ids=["bubble", "walls"])
def test_phase_steps_over_rows_match_the_tiles(n, walls, monkeypatch):
    """The ACDI step whose waves own 62 cells of the halo'd plane (taken where
    tiles would idle) against the tiled kernel bit for bit: rows shorter than
    a wave, of one wave's cells, and across waves; one block and several in z."""
    spec = cases.rising_bubble_3d(ng=tuple(n))
    if walls:
        spec = dict(cases.hysing_2d(ng=(n[0], 2, n[2])), ng=n, l=[1.0, n[1] / n[0], n[2] / n[0]])
    out = []
    for variant in ("3", "4"):
        monkeypatch.setenv("FZ_ACDI_VARIANT", variant)
        dc = F.DeviceCase(spec)
        try:
            dc.init()
            dc.step(4)
            out.append({k: dc.get(k) for k in FIELDS})
        finally:
            dc.close()
    for k in FIELDS:
        assert np.array_equal(out[0][k], out[1][k], equal_nan=True), k


@pytest.mark.parametrize("n", [[256, 192, 257], [245, 225, 257]], ids=["even columns", "odd columns"])
def test_many_long_fp32_columns(n, rng, monkeypatch):
    """FP32 columns of more than 256 rows go two to a lane where an even number
    of at least 49152 fill the device, an odd number in registers: as the
    chunked kernel's bit for bit."""
    f = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n]))
    monkeypatch.delenv("FZ_THOMAS_ROWS32", raising=False)
    got = solve(n, "PPPPNN", f, True)
    monkeypatch.setenv("FZ_THOMAS_ROWS32", "16")
    assert np.array_equal(got, solve(n, "PPPPNN", f, True))


@pytest.mark.parametrize("n", [[1, 1, 2], [5, 3, 2], [33, 7, 9], [64, 8, 17], [70, 13, 40]],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("vof", [0, 1], ids=["acdi", "thinc"])
def test_rk_2fl_writes_the_faces_of_its_transport(n, vof, rng):
    """The flux arrays after rk_2fl are the transport routine's in every
    element, halo included: THINC/QQ has the faces at index 0 (src/
    vof_thinc_qq.f90:66-121), and what neither writes keeps its value."""
    ctx = F.Context(n, [1.0, 0.9, 1.7], "PPPPNN", gr=0.5)
    try:
        rand = lambda lo=-1.0, hi=1.0: np.asfortranarray(rng.uniform(lo, hi, [x + 2 for x in n]))  # noqa: E731
        h = {q: ctx.halo(rand()) for q in ("u", "v", "w", "nx", "ny", "nz", "phi")}
        h["psi"] = ctx.halo(rand(0.0, 1.0))
        before = [rand() for _ in range(3)]
        one, two = [ctx.halo(f) for f in before], [ctx.halo(f) for f in before]
        args = [h[q].ptr for q in ("u", "v", "w", "nx", "ny", "nz", "phi", "psi")]
        name, par = ("fz_vof_thinc_transport_psi", [40.0]) if vof else ("fz_acdi_transport_pf", [0.7, 0.02])
        F.call(name, ctx.h, *par, *args, ctx.interior().ptr, *[d.ptr for d in one])
        st = C.c_void_p()
        F.call("fz_rk_state_create", ctx.h, C.byref(st))
        F.call("fz_rk_2fl", ctx.h, st, (C.c_double * 2)(1.5, -0.5), 1e-3, 0.7, 0.02, 40.0, vof, *args,
               *[d.ptr for d in two])
        for a, b, f in zip(one, two, before):
            a = a.download()
            assert np.array_equal(b.download(), a)
            assert not np.array_equal(a, f)
        F.lib().fz_rk_state_destroy(st)
    finally:
        ctx.close()


def test_batched_solves_follow_the_default_stream(rng):
    """Right-hand sides written on the default stream, behind copies that take
    milliseconds, are there when fz_solver_batched reads them."""
    hip, n, k = F.lib(), [32, 24, 16], 3  # (the library's own HIP runtime)
    ctxs = [F.Context(n, [1.0, 0.9, 1.7], "PPPPNN") for _ in range(k)]
    try:
        for c in ctxs:
            F.call("fz_initsolver", c.h, None, None, None, None, None, None, None, None, None)
        f, zero = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n])), np.zeros([x + 2 for x in n])
        src, ref = ctxs[0].halo(f), ctxs[0].halo(f)
        F.call("fz_solver", ctxs[0].h, ref.ptr)
        ref = ref.download()
        ds = [c.halo(zero) for c in ctxs]
        big = [F.DArray(ctxs[0], (1 << 27,)) for _ in range(2)]  # 1 GiB each
        copy = lambda dst, s: hip.hipMemcpyAsync(dst.ptr, s.ptr, C.c_size_t(s.nbytes), 3, None)  # noqa: E731
        for _ in range(3):
            for d in ds:
                d.upload(zero)
            assert all(copy(*big) == 0 for _ in range(20))
            assert all(copy(d, src) == 0 for d in ds)
            F.call("fz_solver_batched", (C.c_void_p * k)(*[c.h.value for c in ctxs]),
                   (C.c_void_p * k)(*[d.ptr.value for d in ds]), k)
            for d in ds:
                assert np.array_equal(d.download()[1:-1, 1:-1, 1:-1], ref[1:-1, 1:-1, 1:-1])
        for d in big:
            d.free()
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("n", [[16, 15, 16], [16, 15, 17], [128, 126, 23], [128, 128, 23], [128, 128, 24]],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("cbc", ["NNPPDD", "PPPPPP"])
def test_short_columns_match_the_chunked_kernels(n, cbc, rng, monkeypatch):
    """Both sides of the lines from which columns are held in registers (17
    rows; 24 for 16384 FP64 columns, which the cases of a batch have together)."""
    f = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n]))
    for mixed, count in [(False, 1), (True, 1)] + ([(False, 2)] if cbc != "PPPPPP" else []):
        monkeypatch.delenv("FZ_THOMAS_ROWS64", raising=False)
        got = solve(n, cbc, f, mixed, count)
        monkeypatch.setenv("FZ_THOMAS_ROWS64", "16")
        assert np.array_equal(got, solve(n, cbc, f, mixed, count), equal_nan=True), (mixed, count)


def solve_unrefined(n, cbc, f):
    ctx = F.Context(n, [1.0, 0.9, 1.7], cbc)
    try:
        F.call("fz_initsolver", ctx.h, None, None, None, None, None, None, None, None, None)
        d = ctx.halo(f)
        F.call("fz_solver_mixed", ctx.h, d.ptr, 0.0, 0, C.byref(C.c_int()), None)
        return d.download()[1:-1, 1:-1, 1:-1]
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [[33, 256, 3], [35, 512, 2], [18, 1024, 2], [10, 2048, 2]],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("y", ["PP", "NN", "DD"])
def test_sixteen_points_a_thread_match_four(n, y, rng, monkeypatch):
    """Long y lines of every kind in FP32, without refinement, and of the
    periodic one in FP64, alone and as a batch, line counts that are no
    multiple of a block's: bit for bit as four points a thread."""
    f = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n]))
    cbc = "PP" + y + "DD"
    for mixed, count in [(True, 1), (False, 1), (False, 2)]:
        out = []
        for p16 in ("1", "0"):
            monkeypatch.setenv("FZ_P16", p16)
            out.append(solve_unrefined(n, cbc, f) if mixed else solve(n, cbc, f, False, count))
        assert np.array_equal(*out), (mixed, count)
        assert np.abs(out[0]).max() > 0.0


@pytest.mark.parametrize("n,y", [([64, 256, 256], "PP"), ([64, 256, 255], "PP"), ([16, 1024, 256], "NN"),
                                 ([256, 512, 64], "DD"), ([256, 512, 63], "DD")],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else v)
def test_long_fp32_lines_at_the_rule(n, y, rng, monkeypatch):
    """Both sides of the launch sizes from which FP32 lines take sixteen points
    a thread (8 waves a CU; 16 for cosine and sine lines below 1024)."""
    f = np.asfortranarray(rng.uniform(-1.0, 1.0, [x + 2 for x in n]))
    out = []
    for p16 in (None, "0"):
        monkeypatch.delenv("FZ_P16", raising=False)
        if p16:
            monkeypatch.setenv("FZ_P16", p16)
        out.append(solve_unrefined(n, "PP" + y + "DD", f))
    assert np.array_equal(*out)


@pytest.mark.parametrize("n", [[33, 1, 9], [40, 2, 33], [1, 12, 20], [20, 14, 6], [20, 15, 6], [64, 16, 5], [60, 16, 5],
                               [59, 16, 5], [65, 33, 4], [130, 4, 40]], ids=lambda n: "x".join(map(str, n)))
def test_integrators_at_the_rules_of_their_tiles(n, rng):
    """rk and rk_2fl (ACDI) against their parts on both sides of the fill of
    their tiles' rows and lanes that picks another form."""
    test_integrators_match_their_parts(n, 0, rng)
