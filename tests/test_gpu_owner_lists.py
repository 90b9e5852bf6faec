"""Owner plans whose lists are built on the device (20,000 elements and more):
the patches are the host partition's, and every list passes the host checks of
OP_diags (each increment once, in the sequential order, under the block owning
its target), on local and random numberings, with every block size, under
transparent renumbering, and for a map with hundreds of increments per target,
which falls back to the host's lists."""
import ctypes as C

import numpy as np
import pytest

import op2amd
import op2amd.api as api

pytestmark = pytest.mark.gpu


def plan_of(mesh, block, tokens=()):
    """res_calc's owner plan over pecell, built with OP_diags 1 (checked)."""
    api.init(*tokens, diags=1)
    edges = api.op_decl_set(mesh.nedge, b"edges")
    cells = api.op_decl_set(mesh.ncell, b"cells")
    m = api.decl_map(edges, cells, 2, mesh.ecell, "pecell")
    d = api.decl_dat(cells, 1, "double", np.zeros(mesh.ncell), "res")
    args = (api.op_arg * 2)(*[api.arg_dat(d, k, m, 1, "double", api.OP_INC) for k in range(2)])
    p = api.op2h_plan_owner_for(b"res_calc", edges, block, 2, args)
    assert p
    return p.contents


def lists(p, nel):
    ip = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    oo, ow = np.empty(p.nblocks + 1, np.int32), np.empty(p.n_owned, np.int32)
    eo, el = np.empty(p.nblocks + 1, np.int32), np.empty(p.total, np.int32)
    co, cs = np.empty(p.n_owned + 1, np.int32), np.empty(2 * nel, np.uint16)
    assert api.op2h_owner_plan_download(C.byref(p), *map(ip, (oo, ow, eo, el, co, cs))) == 0
    return oo, ow, eo, el, co, cs


@pytest.mark.parametrize("block", [1, 64, 128, 1000, 1024, 4096])
@pytest.mark.parametrize("ordering", ["rcm", "random", "structured"])
def test_device_lists_are_the_host_partitions(ordering, block):
    mesh = op2amd.mesh.generate(147, 93, 4, ordering)
    assert mesh.nedge >= 20000
    p = plan_of(mesh, block)
    try:
        oo, ow, eo, el, co, cs = lists(p, mesh.nedge)
    finally:
        api.op_exit()
    nb, block_of = api.owner_partition(mesh.ncell, mesh.ecell, [0, 1], block)
    assert p.nblocks == nb and p.n_owned == mesh.ncell
    got = np.empty(mesh.ncell, np.int32)
    got[ow] = np.repeat(np.arange(nb), np.diff(oo))
    assert np.array_equal(got, block_of)
    for b in range(0, nb, max(1, nb // 50)):  # ascending within a block
        assert np.all(np.diff(ow[oo[b]:oo[b + 1]]) > 0) and np.all(np.diff(el[eo[b]:eo[b + 1]]) > 0)
    # each cell's increments in element order, by brute force
    bl = np.repeat(np.arange(nb), np.diff(oo))
    want = [[] for _ in range(mesh.ncell)]
    for e, (a, c) in enumerate(mesh.ecell):
        want[a].append((e, 0))
        want[c].append((e, 1))
    for i in range(0, len(ow), 7):
        have = [(int(el[eo[bl[i]] + x // 2]), int(x) % 2) for x in cs[co[i]:co[i + 1]]]
        assert have == want[ow[i]], i


@pytest.mark.parametrize("block", [64, 256])
def test_device_lists_follow_the_applications_order(block):
    """Transparent renumbering: the checks follow the application's element
    order (both forms of a block's instances)."""
    mesh = op2amd.mesh.generate(160, 100, 6, "random")
    kw = dict(mode="graphed", plan_res="owner", block_res=block, plan_bres="gather", graph_steps=4)
    ref = op2amd.airfoil.run(mesh, 9, **kw)
    got = op2amd.airfoil.run(mesh, 9, renumber="transparent", **kw)
    for k in ("maxerr", "errloc", "q"):
        assert np.array_equal(ref[k], got[k]), k
    p = plan_of(mesh, block, ("OP_HIP_RENUMBER",))
    assert p.n_owned == mesh.ncell
    api.op_exit()


def test_targets_with_hundreds_of_increments_use_the_host_lists():
    rng = np.random.default_rng(0)
    hub = rng.integers(0, 100, (30000, 2)).astype(np.int32)

    class Star:
        nedge, ncell, ecell = 30000, 100, hub
    p = plan_of(Star, 10)
    assert p.max_incs > 64 and p.n_owned == 100
    api.op_exit()


@pytest.mark.parametrize("hub", [64, 65, 25000])
def test_a_target_that_many_elements_name(hub):
    """30,000 elements of which `hub` name target 0: up to 64 of them the lists
    are built on the device, beyond on the host, where a target's list costs
    what it is long.  (In one thread's insertion sort 25,000 neighbours would
    be about 10^8 dependent moves in memory, seconds; the host takes
    milliseconds.)"""
    n = 30000
    ecell = np.stack([np.where(np.arange(n) % (n // hub) == 0, 0, 1 + np.arange(n)), 1 + n + np.arange(n)], 1).astype(np.int32)
    ecell[np.flatnonzero(ecell[:, 0] == 0)[hub:], 0] = 1

    class Star:
        nedge, ncell = n, 2 * n + 1
    Star.ecell = ecell
    p = plan_of(Star, 64)
    try:
        assert p.max_incs == hub and p.build_ms < 1000
        oo, ow, eo, el, co, cs = lists(p, n)
    finally:
        api.op_exit()
    nb, block_of = api.owner_partition(Star.ncell, ecell, [0, 1], 64)
    got = np.full(Star.ncell, -1, np.int32)
    got[ow] = np.repeat(np.arange(nb), np.diff(oo))
    assert p.nblocks == nb and np.array_equal(got, block_of)


@pytest.mark.parametrize("limit", [0, 100_000, 400_000, 2 ** 50])
def test_without_room_for_scratch_the_host_builds_the_lists(limit):
    """27,000 edges: scratch of at most so many bytes at a time, from none at
    all to the graph's neighbours (430 kB), and no limit."""
    mesh = op2amd.mesh.generate(147, 93, 4, "random")
    want = plan_of(mesh, 128)
    want = lists(want, mesh.nedge)
    api.op_exit()
    api.op2h_set_extra_memory(limit)
    try:
        got = lists(plan_of(mesh, 128), mesh.nedge)
    finally:
        api.op2h_set_extra_memory(2 ** 64 - 1)
        api.op_exit()
    n = want[4][-1]
    for k, (a, b) in enumerate(zip(want, got)):
        assert np.array_equal(a[:n], b[:n]) if k == 5 else np.array_equal(a, b)


def test_more_than_the_device_holds_is_refused_without_an_error():
    api.init()
    try:
        p = api.lib.op2h_extra_alloc
        p.restype, p.argtypes = C.c_void_p, [C.c_size_t]
        assert p(1 << 50) is None
        cells = api.op_decl_set(1000, b"cells")
        d = api.decl_dat(cells, 1, "double", np.arange(1000.0), "d")
        assert np.array_equal(api.fetch(d, (1000,), np.float64), np.arange(1000.0))
    finally:
        api.op_exit()
