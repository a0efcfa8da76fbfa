"""Edges of the engine's entry points: CFL numbers of either sign, engines of many cases and of finished
ones, meshes beyond the 32-bit offsets, what an Euler engine holds, what creation costs and
what the kernel times count."""
import resource
import time

import numpy as np
import pytest

import pyoracle as po
from horses3d_amd import mesh, specmesh

pytestmark = pytest.mark.gpu
TOL = 1e-12   # the parity bar: normwise per variable
KW = dict(mach=0.3, reynolds=700.0, riemann="roe")


def one_step_matches(eng, ora, Q0, cfl, dcfl):
    """advance() by one step takes max_dt's limit, whatever its sign, and ends where the oracle ends"""
    dt = eng.max_dt(cfl, dcfl)
    assert dt == pytest.approx(ora.max_dt(Q0, cfl, dcfl), rel=1e-13) and dt < 0.0
    assert eng.advance(1, cfl, dcfl, t=0.0) == dt
    Q, G = Q0.copy(), np.zeros_like(Q0)
    ora.rk3_step(Q, G, 0.0, dt)
    dq = np.abs(Q - Q0).max(axis=0)
    floor = 4.0 * np.finfo(float).eps * np.abs(Q).max(axis=0)   # four ulp of the state the increment is added to
    assert np.all(np.abs(eng.get_state() - Q).max(axis=0) <= TOL * dq + floor)


def gauss_box(n, N, tmp_path):
    """An n^3 curvilinear box from the front end on Gauss nodes, with the oracle's face tables."""
    from horses3d_amd.engine import read_specmesh
    path = str(tmp_path / "box.mesh")
    specmesh.write_specmesh(path, n, 0.1, mesh.box_phases(5), bface_order=N + 1)
    case = read_specmesh(path, N=N, periodic=dict(specmesh.PERIODIC_PAIRS), nodes="gauss")
    case["fNf"] = np.full((case["F"], 2), N, np.int32)
    case["foff"] = np.arange(case["F"] + 1, dtype=np.int64) * (N + 1) ** 2
    return case


@pytest.mark.parametrize("kind,cfl,dcfl", [(k, c, d) for k in ("gauss-lobatto", "euler", "gauss", "mixed")
                                           for c, d in ((-0.1, -0.1), (0.1, -0.1), (-0.1, 0.1))
                                           if c < 0.0 or k != "euler"])   # Euler: no viscous limit
def test_negative_cfl_numbers(kind, cfl, dcfl, tmp_path):
    """A negative CFL number steps backwards with the limit of the smallest value, as max_dt gives it: the
    minima of the blocks order like the numbers, not like their bits."""
    from horses3d_amd.engine import Engine
    N, euler = 3, kind == "euler"
    if kind == "gauss":
        case = gauss_box(3, N, tmp_path)
    elif kind == "mixed":
        case = mesh.periodic_box_mixed(3, mesh.random_orders(27, 2, 4, 5))
    else:
        case = mesh.periodic_box(3, N, amplitude=0.1, phase_seed=5)
    nodes = "gauss" if kind == "gauss" else "gauss-lobatto"
    Q0 = mesh.taylor_green(case, 0.3, noise=1e-3, seed=3)
    ora = po.Oracle(case, po.make_params(0.3, 700.0, riemann="roe", euler=euler, nodes=nodes))
    eng = Engine(case, euler=euler, nodes=nodes, **KW)
    eng.set_state(Q0)
    one_step_matches(eng, ora, Q0, cfl, dcfl)
    # a zero of either sign is the smallest of these limits: the time stands still
    eng.set_state(Q0)
    assert eng.advance(1, -0.0, 0.4, t=0.0) == 0.0
    # and the next step forwards takes its own limit
    eng.set_state(Q0)
    assert eng.advance(1, 0.4, 0.4, t=0.0) == eng_dt(case, Q0, euler, nodes)
    eng.close()


def eng_dt(case, Q0, euler, nodes):
    from horses3d_amd.engine import Engine
    e = Engine(case, euler=euler, nodes=nodes, **KW)
    e.set_state(Q0)
    dt = e.max_dt(0.4, 0.4)
    e.close()
    return dt


def test_times_of_many_cases_start_at_zero():
    """An engine of more than 256 cases, created where one that had advanced was before."""
    from horses3d_amd.engine import MultiEngine
    box, n = mesh.straight_box(2, 3), 600
    Q0 = [mesh.taylor_green(box, 0.3)] * n
    for _ in range(4):
        eng = MultiEngine([box] * n, KW)
        times, bad = eng.status()
        assert not times.any() and not bad.any()
        eng.set_states(Q0)
        eng.advance(1, 0.4, 0.4)
        times, _ = eng.status()
        assert times[0] > 0.0 and np.all(times == times[0])
        eng.close()


@pytest.mark.parametrize("n,N,ncases", [(1, 1, 64), (1, 2, 300), (2, 1, 70)])
def test_many_small_cases_match_cases_alone(n, N, ncases):
    """More cases than their face nodes fill blocks of 256 with: each ends where it ends alone."""
    from horses3d_amd.engine import Engine, MultiEngine
    box = mesh.periodic_box(n, N, amplitude=0.1, phase_seed=4)
    assert box["F"] * (N + 1) ** 2 * ncases // 256 + 1 < ncases
    Q0 = [mesh.taylor_green(box, 0.3, noise=1e-2, seed=c) for c in range(ncases)]
    phys = [dict(KW, reynolds=200.0 + c) for c in range(ncases)]
    m = MultiEngine([box] * ncases, phys)
    m.set_states(Q0)
    m.advance(3, 0.4, 0.4)
    times, bad = m.status()
    got = m.get_states()
    assert not bad.any()
    for c in {0, 1, ncases // 2, ncases - 1}:
        e = Engine(box, **phys[c])
        e.set_state(Q0[c])
        assert e.advance(3, 0.4, 0.4, t=0.0) == times[c], c
        assert np.array_equal(e.get_state(), got[c]), c
        e.close()
    m.close()


@pytest.mark.parametrize("graph", [False, True])
def test_finished_cases_keep_their_state(graph):
    """Cases switched off and on again after odd and even numbers of stages, with states set while one is
    off: each ends where it ends alone, and a finished one reads back the same after every step."""
    from horses3d_amd.engine import Engine, MultiEngine
    boxes = [mesh.periodic_box(n, 3, amplitude=0.1, phase_seed=n) for n in (2, 1, 3)]
    phys = [dict(KW, reynolds=300.0 + 100.0 * c) for c in range(3)]
    Q0 = [mesh.taylor_green(b, 0.3, noise=1e-2, seed=c) for c, b in enumerate(boxes)]
    alone = [Engine(b, **p) for b, p in zip(boxes, phys)]
    m = MultiEngine(boxes, phys)
    m.set_step_graph(graph)
    on = [True] * 3

    def states(qs):
        m.set_states(qs)
        for e, q in zip(alone, qs):
            e.set_state(q)

    def switch(c, to):
        m.set_active(c, to)
        on[c] = to

    def steps(n):
        m.advance(n, 0.4, 0.4)
        for c, e in enumerate(alone):
            if on[c]:
                e.advance(n, 0.4, 0.4)
        got = m.get_states()
        for c, e in enumerate(alone):
            assert np.array_equal(got[c], e.get_state()), c

    states(Q0)
    steps(1)
    switch(1, False)
    steps(1)
    steps(2)
    switch(0, False)
    switch(0, False)                 # again: nothing changes
    steps(5)
    switch(1, True)
    steps(1)
    states([q[::-1].copy() for q in Q0])   # while case 0 is off
    steps(3)
    switch(0, True)
    steps(2)
    switch(0, False)
    switch(2, False)
    m.rk3_step(0.0, 1e-4)
    alone[1].rk3_step(0.0, 1e-4)
    steps(0)
    m.close()
    for e in alone:
        e.close()


def test_finished_cases_cost_no_memory_traffic():
    """Sixteen cases of 12^3 elements of order 4: a step with all of them finished takes what its launches
    take (33 us, 0.026 of a step with all of them on); carrying the states along from copy to copy took 241
    us (0.19)."""
    from horses3d_amd.engine import MultiEngine
    box = mesh.straight_box(12, 4)
    m = MultiEngine([box] * 16, KW)
    m.set_states([mesh.taylor_green(box, 0.3)] * 16)

    def per_step():
        best = np.inf
        for _ in range(7):
            m.synchronize()
            t0 = time.perf_counter()
            m.advance(20, 0.4, 0.4)
            m.synchronize()
            best = min(best, (time.perf_counter() - t0) / 20)
        return best

    on = per_step()
    for c in range(16):
        m.set_active(c, False)
    off = per_step()
    print("step with all on %.1f us, with all finished %.1f us" % (1e6 * on, 1e6 * off), flush=True)
    assert off < 0.06 * on
    m.close()


def test_mesh_beyond_the_offsets_is_refused_by_its_size():
    """2^29 element face nodes and more: refused as too large before any table is built, whose 32-bit
    entries would wrap (the tables and geometry here are untouched zeros)."""
    from horses3d_amd.engine import Engine
    K = 2 ** 29 // 24 + 1   # order 1
    case = dict(K=K, F=3 * K, N=np.ones((K, 3), np.int32), J=np.zeros(8 * K), Ja=np.zeros((8 * K, 9)))
    for name, shape in (("faceID", (K, 6)), ("faceSide", (K, 6)), ("fElem", (3 * K, 2)), ("fESide", (3 * K, 2)), ("fRot", 3 * K)):
        case[name] = np.zeros(shape, np.int32)
    with pytest.raises(Exception, match="mesh too large"):
        Engine(case, **KW)


@pytest.mark.parametrize("nodes", ["gauss-lobatto", "gauss"])
def test_euler_engine_holds_no_viscous_arrays(nodes, tmp_path):
    """An Euler engine's memory is that of a Navier-Stokes one without nine viscous values and |curl u|^2 a
    node (Gauss nodes: and nine values an element face node); every call works on it."""
    from horses3d_amd.engine import Engine
    n, N = 4, 3
    case = gauss_box(n, N, tmp_path) if nodes == "gauss" else mesh.periodic_box(n, N, amplitude=0.1, phase_seed=5)
    ns, eu = (Engine(case, euler=e, nodes=nodes, **KW) for e in (False, True))
    held = 10 * n ** 3 * (N + 1) ** 3 + (9 * 6 * n ** 3 * (N + 1) ** 2 if nodes == "gauss" else 0)
    assert ns.device_bytes() - eu.device_bytes() == 8 * held
    Q0 = mesh.taylor_green(case, 0.3)
    eu.set_state(Q0)
    eu.advance(2, 0.4, 0.4, t=0.0)
    for kind in ("kinetic energy", "kinetic energy rate", "mean velocity", "internal energy", "entropy", "math entropy"):
        assert np.isfinite(eu.volume_monitor(kind)), kind
    with pytest.raises(Exception, match="enstrophy"):
        eu.volume_monitor("enstrophy")
    assert np.all(np.isfinite(eu.residuals())) and np.all(np.isfinite(eu.qdot()))
    ora = po.Oracle(case, po.make_params(0.3, 700.0, riemann="roe", euler=True, nodes=nodes))
    eu.set_state(Q0)
    assert po.normwise_error(eu.qdot(), ora.qdot(Q0)).max() <= TOL
    ns.close()
    eu.close()


def test_repeated_creation_reuses_its_host_pages():
    """16^3 elements of order 4: the face tangents of a Lax-Friedrichs engine (15 MB) cost no page faults of
    their own when engines are created one after another (in one array with the normals, past the size of
    which the allocator keeps pages, they cost 8400 on top of 9000)."""
    from horses3d_amd.engine import Engine
    case = mesh.periodic_box(16, 4, amplitude=0.1, phase_seed=1)
    faults = {}
    for _ in range(4):
        for riemann in ("roe", "lxf"):
            before = resource.getrusage(resource.RUSAGE_SELF).ru_minflt
            e = Engine(case, mach=0.3, reynolds=700.0, riemann=riemann)
            faults[riemann] = resource.getrusage(resource.RUSAGE_SELF).ru_minflt - before
            e.close()
    print(faults, flush=True)
    assert faults["lxf"] < 1.3 * faults["roe"] + 500


@pytest.mark.parametrize("kind", ["gauss-lobatto", "gauss", "mixed"])
def test_kernel_times_count_launches(kind, tmp_path):
    """A case of one order has no face kernel, and none is timed (two events with nothing between them are
    4 us apart); mixed orders have one."""
    from horses3d_amd.engine import Engine
    case = {"gauss": lambda: gauss_box(3, 3, tmp_path), "mixed": lambda: mesh.periodic_box_mixed(3, mesh.random_orders(27, 2, 4, 5)),
            "gauss-lobatto": lambda: mesh.periodic_box(3, 3, amplitude=0.1, phase_seed=5)}[kind]()
    eng = Engine(case, nodes="gauss" if kind == "gauss" else "gauss-lobatto", **KW)
    eng.set_state(mesh.taylor_green(case, 0.3))
    eng.set_timing(True)
    eng.advance(3, 0.4, 0.4, t=0.0)
    grad, face, volume, stage = eng.kernel_times()
    assert grad > 0.0 and volume > 0.0 and stage == grad + face + volume
    assert (face > 0.0) == (kind == "mixed")
    eng.close()
