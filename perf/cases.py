"""The work that is measured: what users of this OP2 backend have it do.

  app       a whole airfoil program through op2amd.airfoil.run: from a mesh in host memory through the declarations, plan
            builds and all time steps to the final q and the per-iteration reductions back on the host
  step      one eager time step (nine op_par_loops through the C API) on data that stays on the device
  ensemble  many meshes advanced in lock step through op2amd.ensemble.run
  train     training of the plan-selection cost model, predict: its forward pass at a loop's first call
  update    the update loop on caller-owned device arrays (op2h_update_noalloc)
"""
import ctypes as C
import functools
import math
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "op2-common_amd"))
import op2amd  # noqa: E402
from op2amd import api, costmodel  # noqa: E402

FEATURES, HIDDEN = 22, 64  # the cost model's


def listed():
    app = dict(kind="app", ordering="rcm", mode="graphed", plan="owner", block=128, mixed=False, soa=False, renumber=False)
    return [
        # a small program, steps replayed from graphs: launches and gaps between them, set-up and tear-down
        dict(app, name="app 120x60 graphed", I=120, J=60, niter=1000),
        # the benchmark's mesh and plans over a real run's length, FP64
        dict(app, name="app 1200x600 graphed", I=1200, J=600, niter=2000),
        # a mesh whose data stays in HBM, FP32 fluxes under FP64 state
        dict(app, name="app 2400x1200 mixed graphed", I=2400, J=1200, niter=1000, block=256, mixed=True),
        # an odd mesh as a mesher numbers it, SoA dats, renumbered on the device only
        dict(app, name="app 613x287 random soa", I=613, J=287, ordering="random", soa=True, renumber=True, niter=500),
        # tuned plans without graphs: a host that looks at rms after every update
        dict(app, name="app 333x177 tuned", I=333, J=177, mode="tuned", plan="gather", niter=500),
        # a translated program with nothing set, its mesh as generated: staged, coloured plans and a sync after every loop
        dict(app, name="app 400x200 plain", I=400, J=200, ordering="structured", mode="plain", plan="auto", block=0, niter=200),
        # one eager step of the largest mesh, on resident data
        dict(name="step 4800x2400", kind="step", I=4800, J=2400, ordering="structured", block=256, soa=False),
        # a parameter study on small meshes: many members, little work each
        dict(name="ensemble 64 small", kind="ensemble", nmesh=64, max_I=160, max_J=80, niter=500, autotune=False),
        # a study on uneven meshes up to 640x320, workgroup sizes picked at run time
        dict(name="ensemble 16 uneven", kind="ensemble", nmesh=16, max_I=640, max_J=320, niter=1000, autotune=True),
        # a chunk of epochs on the rows of about a hundred timed loops
        dict(name="train 2371x100", kind="train", n=2371, epochs=100),
        # the variants of one loop ranked at its first call
        dict(name="predict 23", kind="predict", n=23),
        # the update alone, on arrays that the caller owns
        dict(name="update 720001", kind="update", n=720001, soa=False, block=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["app", "app", "app", "app", "app", "step", "ensemble", "ensemble", "train", "predict", "update"])
    if kind == "app":
        mode = rng.choice(["graphed", "graphed", "graphed", "graphed", "tuned", "plain"])
        ordering = rng.choice(["rcm", "structured", "hilbert"] + ["random"] * (mode != "plain"))
        renumber = ordering == "random"
        cells = _log(rng, 1200, 2.5e5 if renumber else 1.5e6)
        J = max(8, int(math.sqrt(cells / rng.uniform(1.2, 3.5))))
        I = max(8, cells // J)
        mixed = mode == "graphed" and rng.random() < 0.35
        plan = "auto" if mode == "plain" else "owner" if mode == "graphed" else rng.choice(["owner", "gather", "atomic"])
        return dict(kind="app", I=I, J=J, ordering=ordering, mode=mode, plan=plan, block=0 if mode == "plain" else rng.choice([128, 256]), mixed=mixed,
                    soa=rng.random() < 0.25, renumber=renumber, niter=max(100, min(_log(rng, 200, 1500), int(1.2e9 / cells), 400 if mode == "plain" else 1500)))
    if kind == "step":
        J = _log(rng, 200, 2300)
        return dict(kind="step", I=int(J * rng.uniform(1.1, 2.0)), J=J, ordering="structured", block=rng.choice([128, 256]), soa=rng.random() < 0.25)
    if kind == "ensemble":
        nmesh = _log(rng, 4, 64)
        max_J = min(320, int(80 * math.sqrt(64 / nmesh) * rng.uniform(0.6, 1.6)))
        return dict(kind="ensemble", nmesh=nmesh, max_I=2 * max_J, max_J=max_J, niter=_log(rng, 200, 1000), autotune=rng.random() < 0.5)
    if kind == "train":
        return dict(kind="train", n=_log(rng, 200, 4000), epochs=_log(rng, 20, 120))
    if kind == "predict":
        return dict(kind="predict", n=_log(rng, 5, 8000))
    return dict(kind="update", n=_log(rng, 5000, 1.1e7), soa=rng.random() < 0.3, block=rng.choice([128, 256, 512]))


# ---- inputs ----


@functools.lru_cache(maxsize=1)
def _numbered(I, J, ordering):
    m = op2amd.mesh.generate(I, J, 0, ordering)
    inner = np.ones(m.nnode)
    inner[m.bedge.reshape(-1)] = 0.0
    return m, inner


def _mesh(case, seed):
    """The case's mesh with its inner nodes moved by up to 4 % of a cell's sides, as the seed says."""
    m, inner = _numbered(case["I"], case["J"], case["ordering"])
    step = np.random.default_rng(seed).uniform(-0.04, 0.04, (m.nnode, 2)) * (2.0 / case["I"], 1.0 / case["J"])
    return op2amd.mesh.Mesh(m.nnode, m.ncell, m.nedge, m.nbedge, x=m.x + step * inner[:, None], cell=m.cell, edge=m.edge, ecell=m.ecell, bedge=m.bedge,
                            becell=m.becell, bound=m.bound)


def _constants():
    """The program's constants, float literals as the airfoil application has them (rotated free stream)."""
    f = np.float32
    gam, cfl, eps, mach = float(f(1.4)), float(f(0.9)), float(f(0.05)), float(f(0.4))
    gm1 = gam - 1.0
    alpha = float(f(3.0) * np.arctan(f(1.0)) / f(45.0))
    u = math.sqrt(gam) * mach
    e = 1.0 / gm1 + 0.5 * u * u
    return dict(gam=[gam], gm1=[gm1], cfl=[cfl], eps=[eps], mach=[mach], alpha=[alpha], qinf=[1.0, u * math.cos(alpha), u * math.sin(alpha), e])


def _start_q(ncell, seed):
    return np.array(_constants()["qinf"]) * (1 + 0.01 * np.random.default_rng(seed + 77).standard_normal((ncell, 4)))


class _Array:
    """A dat's device rows, for torch to look at without a copy; keeps its program alive."""

    def __init__(self, program, dat, rows):
        self.program, d = program, dat.contents
        shape = (rows, d.dim) if d.dim > 1 else (rows,)
        if api.lib.op2h_dat_soa_stride(dat):
            shape = (d.dim, d.set.contents.stride)
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f8", data=(d.data_d, False), version=3)


class _Program:
    """An airfoil program on the C API, its data on the device; the library is left when the last one goes."""

    live = weakref.WeakSet()

    def __init__(self, case, seed):
        m = _mesh(case, seed)
        if not _Program.live:
            api.init(*(["OP_AUTO_SOA"] if case["soa"] else []))
            api.op2h_set_sync_mode(api.SYNC_GBL_ONLY)
            api.op2h_set_loop_plan(b"res_calc", api.PLAN_OWNER, case["block"])
            api.op2h_set_loop_plan(b"bres_calc", api.PLAN_GATHER, 128)
            for name, v in _constants().items():
                a = np.array(v)
                api.op_decl_const_char(len(v), b"double", 8, a.ctypes.data_as(C.c_void_p), name.encode())
        _Program.live.add(self)
        nodes, self.edges, self.bedges, self.cells = (api.op_decl_set(n, s) for n, s in ((m.nnode, b"nodes"), (m.nedge, b"edges"), (m.nbedge, b"bedges"), (m.ncell, b"cells")))
        pedge = api.decl_map(self.edges, nodes, 2, m.edge, "pedge")
        pecell = api.decl_map(self.edges, self.cells, 2, m.ecell, "pecell")
        pbedge = api.decl_map(self.bedges, nodes, 2, m.bedge, "pbedge")
        pbecell = api.decl_map(self.bedges, self.cells, 1, m.becell, "pbecell")
        pcell = api.decl_map(self.cells, nodes, 4, m.cell, "pcell")
        bound = api.decl_dat(self.bedges, 1, "int", m.bound, "p_bound")
        x = api.decl_dat(nodes, 2, "double", m.x, "p_x")
        q0 = _start_q(m.ncell, seed)
        q, qold, adt, res = (api.decl_dat(self.cells, d, "double", v, n) for d, v, n in (
            (4, q0, "p_q"), (4, q0, "p_qold"), (1, np.zeros(m.ncell), "p_adt"), (4, np.zeros((m.ncell, 4)), "p_res")))
        self.dats, self.ncell = dict(q=q, qold=qold, adt=adt, res=res), m.ncell
        self.rms, self.maxerr, self.errloc = C.c_double(), C.c_double(), C.c_int()
        R, W, RW, INC, MAX = api.OP_READ, api.OP_WRITE, api.OP_RW, api.OP_INC, api.OP_MAX

        def d(dat, idx, mp, dim, acc, typ="double"):
            return api.arg_dat(dat, idx, mp, dim, typ, acc)

        def gbl(v, typ, size, acc):
            return api.op_arg_gbl_char(C.cast(C.pointer(v), C.c_void_p), 1, typ, size, acc)

        self.loops = (
            (api.loops["op_par_loop_airfoil_1_save_soln"], b"save_soln", self.cells, (d(q, -1, None, 4, R), d(qold, -1, None, 4, W))),
            (api.loops["op_par_loop_airfoil_2_adt_calc"], b"adt_calc", self.cells, (*(d(x, k, pcell, 2, R) for k in range(4)), d(q, -1, None, 4, R), d(adt, -1, None, 1, W))),
            (api.loops["op_par_loop_airfoil_3_res_calc"], b"res_calc", self.edges, (
                d(x, 0, pedge, 2, R), d(x, 1, pedge, 2, R), d(q, 0, pecell, 4, R), d(q, 1, pecell, 4, R), d(adt, 0, pecell, 1, R), d(adt, 1, pecell, 1, R),
                d(res, 0, pecell, 4, INC), d(res, 1, pecell, 4, INC))),
            (api.loops["op_par_loop_airfoil_4_bres_calc"], b"bres_calc", self.bedges, (
                d(x, 0, pbedge, 2, R), d(x, 1, pbedge, 2, R), d(q, 0, pbecell, 4, R), d(adt, 0, pbecell, 1, R), d(res, 0, pbecell, 4, INC), d(bound, -1, None, 1, R, "int"))),
            (api.loops["op_par_loop_airfoil_5_update"], b"update", self.cells, (
                d(qold, -1, None, 4, R), d(q, -1, None, 4, W), d(res, -1, None, 4, RW), d(adt, -1, None, 1, R), gbl(self.rms, b"double", 8, INC),
                gbl(self.maxerr, b"double", 8, MAX), api.op_arg_idx(-1, api.OP_ID), api.op_arg_info_char(C.cast(C.pointer(self.errloc), C.c_void_p), 1, b"int", 4, 5))))

    def __del__(self):
        if _Program is not None:  # (None in a process's own end)
            _Program.live.discard(self)
            if not _Program.live:
                api.op_exit()

    def step(self):
        save, rest = self.loops[0], self.loops[1:]
        save[0](save[1], save[2], *save[3])
        for _ in range(2):
            self.rms.value, self.maxerr.value, self.errloc.value = 0.0, 0.0, 0
            for fn, name, over, args in rest:
                fn(name, over, *args)

    def outputs(self):
        out = {k: torch.as_tensor(_Array(self, v, self.ncell), device="cuda") for k, v in self.dats.items()}
        return dict(out, rms=self.rms.value, maxerr=self.maxerr.value, errloc=self.errloc.value)


def _spec(case, seed):
    """The meshes are the case's own; the seed sets the study's range of Mach numbers and angles."""
    r = np.random.default_rng(seed)
    lo, al = r.uniform(0.28, 0.34), r.uniform(0.0, 1.0)
    return op2amd.ensemble.spec(nmesh=case["nmesh"], max_IJ=(case["max_I"], case["max_J"]), seed=7, mach=(lo, lo + 0.25), alpha_deg=(al, al + 4.0))


def _rows(case, seed):
    """Standardised feature rows and targets that depend on them, as the timed loops' log times do."""
    r = np.random.default_rng(seed)
    x = r.standard_normal((case["n"], FEATURES)).astype(np.float32)
    w = r.standard_normal((FEATURES, 3)) / math.sqrt(FEATURES)
    h = x @ w
    return x, (0.5 * np.tanh(h[:, 0]) + 0.3 * np.abs(h[:, 1]) - 0.2 * h[:, 2] + 0.05 * r.standard_normal(case["n"])).astype(np.float32)


def _arrays(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = case["n"]
    stride = (n + 63) // 64 * 64 if case["soa"] else 0
    shape = (4, stride) if stride else (n, 4)
    qinf = torch.tensor(_constants()["qinf"], dtype=torch.float64, device="cuda")
    qold = (qinf[:, None] if stride else qinf) * (1 + 0.02 * torch.randn(shape, dtype=torch.float64, device="cuda", generator=g))
    res = 1e-3 * torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
    adt = 0.5 + torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
    return stride, qold, res, adt


def prepare(case, seed):
    kind = case["kind"]
    # OP_AUTO_SOA holds for the whole process, as a program's command line gives it: each case sets its own
    C.c_int.in_dll(api.lib, "OP_auto_soa").value = int(case.get("soa", False))
    if kind == "app":
        return case, _mesh(case, seed)
    if kind == "step":
        p = _Program(case, seed)
        p.step()  # builds the plans
        return case, p
    if kind == "ensemble":
        return case, _spec(case, seed)
    if kind in ("train", "predict"):
        net = costmodel.MLP(FEATURES, HIDDEN, seed=seed)
        net.set_weight_decay(1e-4)
        return case, net, *_rows(case, seed)
    stride, qold, res, adt = _arrays(case, seed)
    return case, stride, qold, torch.zeros_like(qold), res, adt, torch.zeros(3, dtype=torch.float64, device="cuda")


def run(state):
    case = state[0]
    kind = case["kind"]
    if kind == "app":
        plans = {} if case["plan"] == "auto" else dict(plan_res=case["plan"], block_res=case["block"], plan_bres="atomic" if case["plan"] == "atomic" else "gather")
        r = op2amd.airfoil.run(state[1], case["niter"], mode=case["mode"], mixed=case["mixed"], soa=case["soa"], graph_steps=10,
                               renumber="transparent" if case["renumber"] else False, **plans)
        return {k: r[k] for k in ("q", "rms", "rms_k0", "maxerr", "errloc")}
    if kind == "step":
        state[1].step()
        return state[1].outputs()
    if kind == "ensemble":
        r = op2amd.ensemble.run(state[1], case["niter"], want_q=True, autotune=case["autotune"])
        return {k: r[k] for k in ("q", "rms", "maxerr", "errloc")}
    if kind == "train":
        _, net, x, t = state
        return dict(loss=net.train(x, t, case["epochs"], 3e-3), params=net.params())
    if kind == "predict":
        return state[1].forward(state[2])
    _, stride, qold, q, res, adt, result = state
    if api.lib.op2h_update_noalloc(case["n"], stride, case["block"], *(C.c_void_p(t.data_ptr()) for t in (qold, q, res, adt, result)),
                                   C.c_void_p(torch.cuda.current_stream().cuda_stream)):
        raise RuntimeError("op2h_update_noalloc failed")
    return dict(q=q, res=res, result=result[:2], errloc=result.view(torch.int32)[4])


# ---- work, tolerances ----


def _step_work(ncell, nnode, nedge, real=8):
    """A time step of two half steps: the maps and x, q and adt read and written in each, the step's first q in the second."""
    half = 16 * ncell + 16 * nedge + 16 * nnode + 2 * (32 + real) * ncell
    return dict(bytes=2.0 * half + 32.0 * ncell, flops=2.0 * (75 * nedge + 80 * ncell))


def work(case):
    kind = case["kind"]
    if kind in ("app", "step", "ensemble"):
        sizes = [(case["I"], case["J"])] if kind != "ensemble" else [(m["I"], m["J"]) for m in op2amd.ensemble.describe(_spec(case, 0))]
        nc, nn = sum(i * j for i, j in sizes), sum((i + 1) * (j + 1) for i, j in sizes)
        ne = sum((i - 1) * j + i * (j - 1) for i, j in sizes)
        w = _step_work(nc, nn, ne, 4 if case.get("mixed") else 8)
        steps = case.get("niter", 1)
        return {k: v * steps for k, v in w.items()}
    params = (FEATURES + 1) * HIDDEN + (HIDDEN + 1) * HIDDEN + HIDDEN + 1
    if kind == "train":
        return dict(bytes=4.0 * (case["n"] * (FEATURES + 1) + 4 * params), flops=6.0 * params * case["n"] * case["epochs"])
    if kind == "predict":
        return dict(bytes=4.0 * (case["n"] * (FEATURES + 1) + params), flops=2.0 * params * case["n"])
    return dict(bytes=136.0 * case["n"], flops=20.0 * case["n"])


def tolerance(case):
    kind = case["kind"]
    if kind == "app" and case["mixed"]:
        return dict(rel=5e-5, max=2e-3, differ=0.01)
    if kind in ("app", "ensemble"):
        return dict(rel=3e-13, max=1e-11, differ=0.01)
    if kind in ("step", "update"):
        return dict(rel=1e-13, max=1e-11)
    if kind == "train":
        return dict(rel=2e-2, max=0.8)
    return dict(rel=8e-7, max=8e-6)


# ---- the same in 64 bits, in plain torch ----


class _Exact:
    """Airfoil time steps in float64 torch; `member` gives each cell's mesh, for reductions of its own."""

    def __init__(self, x, cell, edge, ecell, bedge, becell, bound, qinf_b, q, member=None, sizes=None):
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
        self.c = {k: v[0] for k, v in _constants().items()}
        x = t(x)
        corner = [x[t(cell[:, k]).long()] for k in range(4)]
        self.sides = [corner[(k + 1) % 4] - corner[k] for k in range(4)]
        self.e0, self.e1 = t(ecell[:, 0]).long(), t(ecell[:, 1]).long()
        self.de = x[t(edge[:, 0]).long()] - x[t(edge[:, 1]).long()]
        self.b = t(becell).long()
        self.db = x[t(bedge[:, 0]).long()] - x[t(bedge[:, 1]).long()]
        self.wall = (t(bound) == 1)[:, None]
        self.qb, self.q = t(qinf_b), t(q)
        n = len(cell)
        sizes = sizes or [n]
        self.M = len(sizes)
        self.member = torch.repeat_interleave(torch.arange(self.M, device="cuda"), torch.tensor(sizes, device="cuda"))
        self.local = torch.cat([torch.arange(s, device="cuda") for s in sizes])
        self.cells = torch.tensor(sizes, dtype=torch.float64, device="cuda")

    def _adt(self, q):
        ri = 1.0 / q[:, 0]
        u, v = ri * q[:, 1], ri * q[:, 2]
        c = torch.sqrt(self.c["gam"] * self.c["gm1"] * (ri * q[:, 3] - 0.5 * (u * u + v * v)))
        return sum((u * d[:, 1] - v * d[:, 0]).abs() + c * torch.sqrt(d[:, 0] ** 2 + d[:, 1] ** 2) for d in self.sides) / self.c["cfl"]

    def _flux(self, q1, q2, d, a):
        def side(q):
            ri = 1.0 / q[:, 0]
            p = self.c["gm1"] * (q[:, 3] - 0.5 * ri * (q[:, 1] ** 2 + q[:, 2] ** 2))
            vol = ri * (q[:, 1] * d[:, 1] - q[:, 2] * d[:, 0])
            zero = torch.zeros_like(p)
            return torch.stack([vol * q[:, 0], vol * q[:, 1] + p * d[:, 1], vol * q[:, 2] - p * d[:, 0], vol * (q[:, 3] + p)], 1), torch.stack([zero, p * d[:, 1], -p * d[:, 0], zero], 1)
        (f1, w1), (f2, _) = side(q1), side(q2)
        return 0.5 * (f1 + f2) + (a * self.c["eps"])[:, None] * (q1 - q2), w1

    def step(self):
        self.qold, self.raw = self.q, []
        for _ in range(2):
            q = self.q
            self.adt = self._adt(q)
            f, _ = self._flux(q[self.e0], q[self.e1], self.de, 0.5 * (self.adt[self.e0] + self.adt[self.e1]))
            res = torch.zeros_like(q).index_add_(0, self.e0, f).index_add_(0, self.e1, f, alpha=-1)
            far, wall = self._flux(q[self.b], self.qb, self.db, self.adt[self.b])
            res.index_add_(0, self.b, torch.where(self.wall, wall, far))
            d = res / self.adt[:, None]
            self.q = self.qold - d
            s = d * d
            self.raw.append(torch.zeros(self.M, dtype=torch.float64, device="cuda").index_add_(0, self.member, s.sum(1)) if self.M > 1 else s.sum()[None])
        top = s.amax(1)
        self.maxerr = torch.zeros(self.M, dtype=torch.float64, device="cuda").index_reduce_(0, self.member, top, "amax") if self.M > 1 else top.amax()[None]
        at = torch.where(top == self.maxerr[self.member], self.local, 1 << 30)
        self.errloc = torch.full((self.M,), 1 << 30, device="cuda").index_reduce_(0, self.member, at, "amin") if self.M > 1 else at.amin()[None]
        self.rms = torch.sqrt(self.raw[1] / self.cells)

    def steps(self, n):
        log = []
        for _ in range(n):
            self.step()
            log.append((self.rms, self.raw[0], self.maxerr, self.errloc.to(torch.int32)))
        return [torch.stack(v) for v in zip(*log)]


def _soa(t, stride):
    out = torch.zeros((t.shape[1], stride), dtype=t.dtype, device=t.device)
    out[:, : t.shape[0]] = t.T
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("app", "step"):
        m = _mesh(case, seed)
        qinf = np.array(_constants()["qinf"])
        q0 = np.tile(qinf, (m.ncell, 1)) if kind == "app" else _start_q(m.ncell, seed)
        e = _Exact(m.x, m.cell, m.edge, m.ecell, m.bedge, m.becell, m.bound, np.tile(qinf, (m.nbedge, 1)), q0)
        if kind == "app":
            rms, k0, maxerr, errloc = (v[:, 0] for v in e.steps(case["niter"]))
            return dict(q=e.q, rms=rms, rms_k0=k0, maxerr=maxerr, errloc=errloc)
        e.steps(2)
        q, qold = (_soa(v, (m.ncell + 63) // 64 * 64) if case["soa"] else v for v in (e.q, e.qold))
        return dict(q=q, qold=qold, adt=e.adt, res=torch.zeros_like(q), rms=float(e.raw[1]), maxerr=float(e.maxerr), errloc=int(e.errloc))
    if kind == "ensemble":
        parts, members = [], op2amd.ensemble.describe(_spec(case, seed))
        for k, mb in enumerate(members):  # a member's mesh: the spec's seed + 1 + its number
            parts.append(op2amd.mesh.generate(mb["I"], mb["J"], 7 + 1 + k, "rcm"))
        no = np.cumsum([0] + [p.nnode for p in parts])
        co = np.cumsum([0] + [p.ncell for p in parts])
        cat = lambda f: np.concatenate([f(p, k) for k, p in enumerate(parts)])  # noqa: E731
        qi = [np.array(mb["qinf"]) for mb in members]
        e = _Exact(cat(lambda p, k: p.x), cat(lambda p, k: p.cell + no[k]), cat(lambda p, k: p.edge + no[k]), cat(lambda p, k: p.ecell + co[k]),
                   cat(lambda p, k: p.bedge + no[k]), cat(lambda p, k: p.becell + co[k]), cat(lambda p, k: p.bound), cat(lambda p, k: np.tile(qi[k], (p.nbedge, 1))),
                   cat(lambda p, k: np.tile(qi[k], (p.ncell, 1))), sizes=[p.ncell for p in parts])
        rms, _, maxerr, errloc = e.steps(case["niter"])
        return dict(q=e.q, rms=rms, maxerr=maxerr, errloc=errloc)
    if kind in ("train", "predict"):
        _, net, x, t = prepare(case, seed)
        return _exact_train(case, net.params(), x, t) if kind == "train" else _layers(_weights(torch.as_tensor(net.params()).double()), torch.as_tensor(x).double())[0]
    _, stride, qold, _, res, adt, _ = prepare(case, seed)
    n = case["n"]
    rows = (lambda v: v[:, :n].T) if stride else (lambda v: v)
    d = rows(res) / adt[:, None]
    q = rows(qold) - d
    top = (d * d).amax(1)
    maxerr = top.amax()
    return dict(q=None if stride else q, res=torch.zeros_like(res) if not stride else None, result=torch.stack([(d * d).sum(), maxerr]), errloc=int((top == maxerr).nonzero()[0]))


def _weights(p):
    out, o = [], 0
    for a, b in ((FEATURES, HIDDEN), (HIDDEN, HIDDEN), (HIDDEN, 1)):
        out += [p[o:o + a * b].reshape(a, b), p[o + a * b:o + a * b + b]]
        o += a * b + b
    return out


def _layers(w, x):
    a1 = (x @ w[0] + w[1]).clamp_min(0)
    a2 = (a1 @ w[2] + w[3]).clamp_min(0)
    return (a2 @ w[4] + w[5])[:, 0], a1, a2


def _exact_train(case, params, x, t):
    p, x, t = (torch.as_tensor(v).double() for v in (params, x, t))
    n = case["n"]
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for k in range(1, case["epochs"] + 1):
        w = _weights(p)
        y, a1, a2 = _layers(w, x)
        dy = (2 * (y - t) / n)[:, None]
        d2 = (dy @ w[4].T) * (a2 > 0)
        d1 = (d2 @ w[2].T) * (a1 > 0)
        g = torch.cat([v2.reshape(-1) for a, d in ((x, d1), (a1, d2), (a2, dy)) for v2 in (a.T @ d, d.sum(0))])
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        p = p - 3e-3 * (m / (1 - 0.9 ** k)) / ((v / (1 - 0.999 ** k)).sqrt() + 1e-8) - 3e-3 * 1e-4 * p
    return dict(loss=float(((_layers(_weights(p), x)[0] - t) ** 2).mean()), params=p)
