"""The update's launch shapes: one cell per thread on small meshes, chunks of three beyond, and the lines between them.

The increments are computed as the kernel computes them (adt divides, the squares are added in component order), so q, the
maximum and its first cell are equal; a cell's own sum of four squares has at most four roundings, the sum over the cells one.
"""
import ctypes as C
import math

import numpy as np
import pytest

from op2amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 128, 256, 512])
@pytest.mark.parametrize("n", [1, 255, 257, 65536, 65537, 131072, 131073, 200001])
def test_update_shapes(n, block):
    rng = np.random.default_rng(n + block)
    qold, res = 1 + rng.standard_normal((n, 4)), 1e-3 * rng.standard_normal((n, 4))
    adt = 0.5 + rng.random(n)
    res[n // 2] = res[n // 3] = 7.0  # the maximum twice: its first cell counts
    adt[n // 2] = adt[n // 3] = 0.25
    d = (1.0 / adt)[:, None] * res
    api.init()
    try:
        api.op2h_set_loop_plan(b"update", api.PLAN_AUTO, block)
        cells = api.op_decl_set(n, b"cells")
        dats = [api.decl_dat(cells, a.shape[1], "double", a, name)
                for a, name in ((qold, "qold"), (np.zeros((n, 4)), "q"), (res.copy(), "res"), (adt[:, None].copy(), "adt"))]
        args = [api.arg_dat(v, -1, None, v.contents.dim, "double", acc)
                for v, acc in zip(dats, (api.OP_READ, api.OP_WRITE, api.OP_RW, api.OP_READ))]
        rms, maxerr, errloc = C.c_double(), C.c_double(), C.c_int(-1)
        api.loops["op_par_loop_airfoil_5_update"](
            b"update", cells, *args, api.op_arg_gbl_char(C.cast(C.pointer(rms), C.c_void_p), 1, b"double", 8, api.OP_INC),
            api.op_arg_gbl_char(C.cast(C.pointer(maxerr), C.c_void_p), 1, b"double", 8, api.OP_MAX), api.op_arg_idx(-1, api.OP_ID),
            api.op_arg_info_char(C.cast(C.pointer(errloc), C.c_void_p), 1, b"int", 4, 5))
        assert np.array_equal(api.fetch(dats[1], (n, 4), np.float64), qold - d)
        assert not api.fetch(dats[2], (n, 4), np.float64).any()
    finally:
        api.op2h_set_loop_plan(b"update", api.PLAN_AUTO, 0)
        api.op_exit()
    assert maxerr.value == 28.0**2 and errloc.value == n // 3
    assert abs(rms.value - math.fsum((d * d).ravel())) <= 5 * 2.0**-53 * rms.value
