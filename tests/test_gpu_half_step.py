"""Captured airfoil steps as fused half steps (one launch per half step over
the owner plan's patches): bit for bit the unfused loops, at the edges of the
patches (fewer cells than one, partly filled last ones, more staged cells or
nodes than two per thread), on every ordering, layout and precision, where the
patches do not fit their 16-bit lists and the loops run unfused, and for
captured sequences that are not whole time steps."""
import ctypes as C

import numpy as np
import pytest

import op2amd
import op2amd.api as api
from oracle import oracle
from test_gpu_loops import App, inputs

pytestmark = pytest.mark.gpu
KEYS = ("rms", "rms_k0", "maxerr", "errloc", "q")


def fused_and_not(mesh, niter, **kw):
    """The runs with and without fusion, and how many half steps the first
    one's graph holds."""
    kw = dict(dict(mode="graphed", plan_res="owner", plan_bres="gather", graph_steps=4), **kw)
    n0 = api.op2h_half_step_count()
    fused = op2amd.airfoil.run(mesh, niter, **kw)
    n1 = api.op2h_half_step_count()
    api.op2h_set_fusion(0)
    try:
        plain = op2amd.airfoil.run(mesh, niter, **kw)
    finally:
        api.op2h_set_fusion(1)
    assert api.op2h_half_step_count() == n1
    return fused, plain, n1 - n0


@pytest.mark.parametrize("I,J,ordering,block", [
    (2, 2, "structured", 64), (9, 7, "structured", 64), (16, 8, "random", 128),
    (33, 31, "rcm", 64), (61, 47, "random", 192), (90, 90, "hilbert", 256),
    (100, 83, "structured", 1024), (64, 64, "rcm", 512), (640, 450, "rcm", 64)])
@pytest.mark.parametrize("kw", [dict(), dict(soa=True), dict(mixed=True)],
                         ids=["fp64", "soa", "mixed"])
def test_half_steps_equal_unfused_loops(I, J, ordering, block, kw):
    """640x450 in patches of 64: more of them than one launch has workgroups
    (at most 4096), so each walks two.  Of 1024 cells and the rows around them
    one patch at a time fits in the LDS of a CU."""
    mesh = op2amd.mesh.generate(I, J, 3, ordering)
    fused, plain, halves = fused_and_not(mesh, 29, block_res=block, **kw)
    assert fused["graph_steps"] == 4 and halves == 8
    for k in KEYS:
        assert np.array_equal(fused[k], plain[k]), k
    if not kw:
        ref = oracle.airfoil_run(mesh, 29, 1, "seq")
        assert np.array_equal(fused["q"], ref["q"])


@pytest.mark.parametrize("renumber", [False, "transparent"])
def test_wide_patches_run_unfused(renumber):
    """75,000 randomly numbered cells: a patch's cells span more than 16 bits
    unless the device renumbers them."""
    mesh = op2amd.mesh.generate(300, 250, 5, "random")
    fused, plain, halves = fused_and_not(mesh, 13, block_res=128, renumber=renumber)
    assert fused["graph_steps"] == 4 and halves == (8 if renumber else 0)
    for k in KEYS:
        assert np.array_equal(fused[k], plain[k]), k


@pytest.mark.parametrize("limit", [0, 30_000, 100_000])
def test_without_room_the_loops_run_unfused(limit):
    """Half steps need memory of their own: none of it is there, too little for
    the scratch of the boundary records (69 kB), or all but the other copies of
    q and adt (115 kB)."""
    mesh = op2amd.mesh.generate(61, 47, 3, "rcm")
    api.op2h_set_extra_memory(limit)
    try:
        fused, plain, halves = fused_and_not(mesh, 29, block_res=128)
    finally:
        api.op2h_set_extra_memory(2 ** 64 - 1)
    assert halves == 0
    for k in KEYS:
        assert np.array_equal(fused[k], plain[k]), k
    assert fused_and_not(mesh, 29, block_res=128)[2] == 8


STEP = ["save_soln"] + 2 * ["adt_calc", "res_calc", "bres_calc", "update"]
# the captured loops, and how many half steps they hold
SEQUENCES = {
    "step": (STEP, 2),
    "three steps": (3 * STEP, 6),
    "step, then one stage": (STEP + ["save_soln", "adt_calc", "res_calc", "bres_calc", "update"], 2),
    "one stage, twice": (2 * ["save_soln", "adt_calc", "res_calc", "bres_calc", "update"], 0),
    "ends on save_soln": (STEP + ["save_soln"], 2),
    "ends on adt_calc": (2 * STEP + ["save_soln", "adt_calc"], 4),
    "ends on res_calc": (STEP + ["save_soln", "adt_calc", "res_calc"], 2),
    "ends on bres_calc": (STEP + STEP[:-1], 2),
    "starts inside a step": (STEP[1:] + STEP, 2),
    "no save_soln": (STEP[1:] + STEP[1:], 0),
    "a second adt_calc": (STEP[:2] + ["adt_calc"] + STEP[2:] + STEP, 2),
}


class Program(App):
    def save_soln(self):
        api.loops["op_par_loop_airfoil_1_save_soln"](
            b"save_soln", self.cells, self.d(self.q, -1, None, 4, "double", api.OP_READ),
            self.d(self.qold, -1, None, 4, "double", api.OP_WRITE))

    def play(self, names):
        g = (C.c_double(0.0), C.c_double(0.0), C.c_int(0))
        for n in names:
            getattr(self, n)(*(g if n == "update" else ()))

    def state(self):
        n = self.m.ncell
        for d in (self.q, self.qold, self.adt, self.res):
            api.lib.op_download_dat(d)  # (a replayed graph marks no dat as newer on the device)
        return [self.fetch(d, s) for d, s in ((self.q, (n, 4)), (self.qold, (n, 4)),
                                              (self.adt, (n,)), (self.res, (n, 4)))]


@pytest.mark.parametrize("soa", [False, True], ids=["aos", "soa"])
@pytest.mark.parametrize("name", SEQUENCES)
def test_captured_sequences_leave_every_dat_as_eager_loops_do(name, soa):
    """Three replays of a captured sequence, each followed by a fetch of q,
    qold, adt and res, against the same loops run eagerly."""
    mesh = op2amd.mesh.generate(70, 41, 2, "rcm")
    q, res = inputs(mesh, 4)
    loops, halves = SEQUENCES[name]

    def run(captured):
        app = Program(mesh, q, res, soa=soa)
        try:
            api.op2h_set_sync_mode(api.SYNC_GBL_ONLY)
            api.op2h_set_loop_plan(b"res_calc", api.PLAN_OWNER, 128)
            api.op2h_set_loop_plan(b"bres_calc", api.PLAN_GATHER, 128)
            app.play(STEP)  # builds the plans
            out = []
            if captured:
                n0 = api.op2h_half_step_count()
                assert api.lib.op2h_graph_begin() == 0
                app.play(loops)
                assert api.lib.op2h_graph_end() == 0
                assert api.op2h_half_step_count() - n0 == halves
            for _ in range(3):
                if captured:
                    assert api.lib.op2h_graph_launch(1) == 0
                    api.op2h_device_sync()
                else:
                    app.play(loops)
                out.append(app.state())
            return out
        finally:
            app.close()

    for eager, graph in zip(run(False), run(True)):
        for a, b in zip(eager, graph):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("names", ["two steps", "an update, then a step"])
def test_steps_on_another_res_read_and_zero_it(names):
    """Captured steps that increment a second res dat, which holds values: the
    update before them zeroed the first one, so its zeros say nothing here."""
    mesh = op2amd.mesh.generate(70, 41, 2, "rcm")
    q, res = inputs(mesh, 4)

    def run(captured):
        app = Program(mesh, q, res)
        try:
            first, second = app.res, api.decl_dat(app.cells, 4, "double", 2 * res, "p_res2")

            def play():
                app.res = first
                app.play(STEP if names == "two steps" else ["update"])
                app.res = second
                app.play(STEP)
            api.op2h_set_sync_mode(api.SYNC_GBL_ONLY)
            api.op2h_set_loop_plan(b"res_calc", api.PLAN_OWNER, 128)
            api.op2h_set_loop_plan(b"bres_calc", api.PLAN_GATHER, 128)
            for app.res in (second, first):  # builds the plans; both hold values again
                app.play(STEP[:-1])
            if captured:
                n0 = api.op2h_half_step_count()
                assert api.lib.op2h_graph_begin() == 0
                play()
                assert api.lib.op2h_graph_end() == 0
                assert api.op2h_half_step_count() - n0 == (4 if names == "two steps" else 2)
                assert api.lib.op2h_graph_launch(1) == 0
                api.op2h_device_sync()
            else:
                play()
            app.res = first
            out = app.state()
            app.res = second
            return out + app.state()
        finally:
            app.close()

    for a, b in zip(run(False), run(True)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("names", [["update"], ["update", "save_soln", "adt_calc"], STEP],
                         ids=["eager update", "direct chain", "half steps"])
def test_equal_maxima_keep_the_lowest_application_index(names):
    """288,000 renumbered cells (two and more per thread of every form of the
    update) of which all from one on have exactly the same change: at rest on a
    uniform mesh with sides that are powers of two every flux of mass is zero
    and pressures cancel exactly, so their res is what they start with."""
    mesh = op2amd.mesh.generate(640, 450, 5, "random")  # (the nodes stay in rows)
    mesh.x[:] = np.stack(np.divmod(np.arange(mesh.nnode), 641)[::-1], 1) * 2.0 ** -9
    mesh.bound[:] = 1
    q = np.tile([1.0, 0.0, 0.0, 2.5], (mesh.ncell, 1))
    captured = len(names) > 1
    for first in (0, 1, 2, 3, 5, 8, 20):
        res = np.zeros((mesh.ncell, 4))
        res[first:, 0] = 2.0 ** -10
        app = Program(mesh, q, res, tokens=("OP_HIP_RENUMBER=pecell",))
        try:
            api.op2h_set_sync_mode(api.SYNC_GBL_ONLY)
            api.op2h_set_loop_plan(b"res_calc", api.PLAN_OWNER, 64)
            api.op2h_set_loop_plan(b"bres_calc", api.PLAN_GATHER, 128)
            app.play(["adt_calc", "res_calc", "bres_calc"])  # builds the plans
            if captured:
                n0 = api.op2h_half_step_count()
                assert api.lib.op2h_graph_begin() == 0
                app.play(names)
                assert api.lib.op2h_graph_end() == 0
                assert api.op2h_half_step_count() - n0 == (2 if names == STEP else 0)
                assert api.lib.op2h_graph_launch(1) == 0
                record, n = np.zeros(6), C.c_int()
                api.lib.op2h_graph_history(1, record.ctypes.data_as(C.c_void_p), C.byref(n))
                assert record[1] > 0
                at = int(record.view(np.int32)[4])
            else:
                rms, maxerr, errloc = C.c_double(), C.c_double(), C.c_int(-1)
                app.update(rms, maxerr, errloc)
                at = errloc.value
            assert at == first
        finally:
            app.close()


def test_update_reductions_do_not_depend_on_the_grouping():
    """rms is a sum of unevaluated pairs rounded once: the same bits for every
    workgroup size and launch shape, within 2^-52 of the exactly rounded sum
    (each cell's own four squares are summed in double first: 3 roundings of
    positive terms, 1.5 * 2^-52), also with infinities and NaN."""
    import math
    from test_zz_no_alloc import inputs as arrays, stub_update
    n = 70_001
    qold, q, res, adt = arrays(n, 9)
    got = set()
    for block in (64, 256, 1024):
        api.init()
        try:
            api.op2h_set_loop_plan(b"update", 0, block)
        finally:
            api.op_exit()
        for mode in (0, 1):
            api.op2h_set_streaming(mode)
            try:
                got.add(stub_update(qold, q, res, adt, False)[2])
            finally:
                api.op2h_set_streaming(-1)
    assert len(got) == 1
    exact = math.fsum(((res / adt[:, None]) ** 2).ravel())
    # adti * res rounds twice where res / adt rounds once: another 2 * 2^-53 per
    # square, doubled by squaring
    assert abs(got.pop() - exact) <= 5 * 2.0 ** -52 * exact
    res[123, 2] = np.inf
    assert stub_update(qold, q, res, adt, False)[2] == np.inf
    res[60_000, 1] = np.nan
    assert np.isnan(stub_update(qold, q, res, adt, False)[2])
