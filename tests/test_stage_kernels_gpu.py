"""The two-launch stage of cases of one order: every pairing of Riemann solver and LES model (the
volume kernel's template flags) at orders with whole and remainder element blocks, and Gauss nodes
with Lax-Friedrichs, against the oracle; and the two copies of the state through odd and even step
counts."""
import numpy as np
import pytest

import pyoracle as po
from horses3d_amd import mesh, specmesh

pytestmark = pytest.mark.gpu
TOL = 1e-12   # the parity bar: normwise per variable


@pytest.mark.parametrize("riemann,les", [("roe", None), ("roe", "smagorinsky"), ("lxf", None), ("lxf", "wale")])
@pytest.mark.parametrize("N,inviscid,averaging", [(1, "standard", "kennedy-gruber"), (2, "split-form", "ducros"),
                                                  (3, "standard", "pirozzoli"), (4, "split-form", "morinishi"),
                                                  (5, "standard", "standard"), (6, "split-form", "standard")])
def test_volume_kernel_variants_match_oracle(N, inviscid, averaging, riemann, les):
    from horses3d_amd.engine import Engine
    case = mesh.periodic_box(3, N, amplitude=0.1, phase_seed=20 + N)   # 27 elements
    Q0 = mesh.taylor_green(case, 0.3, noise=1e-3, seed=N)
    kw = dict(mach=0.3, reynolds=700.0, riemann=riemann, inviscid=inviscid, averaging=averaging, les=les)
    ora = po.Oracle(case, po.make_params(kw["mach"], kw["reynolds"], riemann=riemann, inviscid=inviscid,
                                         averaging=averaging, les=les))
    eng = Engine(case, **kw)
    eng.set_state(Q0)
    err = po.normwise_error(eng.qdot(), ora.qdot(Q0))
    print(N, inviscid, averaging, riemann, les, err, flush=True)
    assert err.max() <= TOL
    # one step: the increment to the bar, plus four ulp of the state it is added to
    dt = ora.max_dt(Q0, 0.4, 0.4)
    assert eng.advance(1, 0.4, 0.4, t=0.0) == pytest.approx(dt, rel=1e-13)
    Q, G = Q0.copy(), np.zeros_like(Q0)
    ora.rk3_step(Q, G, 0.0, dt)
    dq = np.abs(Q - Q0).max(axis=0)
    floor = 4.0 * np.finfo(float).eps * np.abs(Q).max(axis=0)
    assert np.all(np.abs(eng.get_state() - Q).max(axis=0) <= TOL * dq + floor)
    eng.close()


def gauss_box(n, N, tmp_path):
    """An n^3 curvilinear box from the front end on Gauss nodes, with the oracle's face tables."""
    path = str(tmp_path / "box.mesh")
    specmesh.write_specmesh(path, n, 0.1, mesh.box_phases(30 + N), bface_order=max(4, N))
    from horses3d_amd.engine import read_specmesh
    case = read_specmesh(path, N=N, periodic=dict(specmesh.PERIODIC_PAIRS), nodes="gauss")
    case["fNf"] = np.full((case["F"], 2), N, np.int32)
    case["foff"] = np.arange(case["F"] + 1, dtype=np.int64) * (N + 1) ** 2
    return case


@pytest.mark.parametrize("tangents", ["cross product", "turned"])
@pytest.mark.parametrize("N,les", [(1, None), (3, "wale"), (4, None), (6, "smagorinsky")])
def test_gauss_lax_friedrichs_matches_oracle(N, les, tangents, tmp_path):
    """Gauss nodes with Lax-Friedrichs face fluxes (one to three rounds of face nodes per thread),
    the second tangent formed in the kernel or, where it is not n x t1, read."""
    from horses3d_amd.engine import Engine
    case = gauss_box(2, N, tmp_path)
    if tangents == "turned":   # the opposite second tangent: another frame, the same flux
        case["t2"] = -case["t2"]
    kw = dict(mach=0.3, reynolds=700.0, riemann="lxf", les=les, nodes="gauss")
    Q0 = mesh.taylor_green(case, 0.3, noise=1e-2, seed=N)
    ora = po.Oracle(case, po.make_params(0.3, 700.0, riemann="lxf", les=les, nodes="gauss"))
    eng = Engine(case, **kw)
    eng.set_state(Q0)
    err = po.normwise_error(eng.qdot(), ora.qdot(Q0))
    print(N, les, tangents, err, flush=True)
    assert err.max() <= TOL
    eng.close()


@pytest.mark.parametrize("kind", ["gauss-lobatto", "euler", "gauss"])
def test_state_copies_through_odd_and_even_steps(kind, tmp_path):
    """A step of three stages ends in the other copy of the state (Gauss nodes: of its traces): any
    split of the steps, with host reads, derivatives and captured steps between, gives the same
    bits."""
    from horses3d_amd.engine import Engine
    case = gauss_box(3, 3, tmp_path) if kind == "gauss" else mesh.periodic_box(3, 3, amplitude=0.1, phase_seed=4)
    Q0 = mesh.taylor_green(case, 0.2, noise=1e-3, seed=9)
    kw = dict(mach=0.2, reynolds=800.0, riemann="roe", euler=kind == "euler",
              nodes="gauss" if kind == "gauss" else "gauss-lobatto")
    ref = Engine(case, **kw)
    ref.set_state(Q0)
    t = ref.advance(17, 0.4, 0.4, t=0.0)
    eng = Engine(case, **kw)
    for graph in (False, True):
        eng.set_step_graph(graph)
        eng.set_state(Q0)
        eng.t = 0.0
        for n in (1, 6, 2, 5, 3):
            eng.advance(n, 0.4, 0.4)
            eng.qdot()
            eng.kinetic_energy()
        assert eng.t == t
        assert np.array_equal(eng.get_state(), ref.get_state()), graph
    eng.close()
    ref.close()


@pytest.mark.parametrize("nodes", ["gauss-lobatto", "gauss"])
@pytest.mark.parametrize("orders,les", [("cubes", None), ("bricks", "smagorinsky")])
def test_rotated_mortar_faces_match_oracle(orders, les, nodes, tmp_path):
    """Every rotation of the right side on faces between elements of unlike orders 1..7: elements of
    equal orders along their axes with all eight rotations, anisotropic ones with the four that keep
    the face axes.  The rotations are drawn, so neighbouring nodes do not meet: a face flux is as well
    defined for the engine and the oracle as on a mesh that turns its elements."""
    from horses3d_amd.engine import Engine, read_specmesh
    rng = np.random.default_rng(5)
    K = 27
    N3 = np.repeat(rng.integers(1, 8, (K, 1)), 3, axis=1) if orders == "cubes" else rng.integers(1, 8, (K, 3))
    if nodes == "gauss":
        path = str(tmp_path / "box.mesh")
        specmesh.write_specmesh(path, 3, 0.1, mesh.box_phases(8), bface_order=7)
        case = read_specmesh(path, N=4, orders=N3.astype(np.int32), periodic=dict(specmesh.PERIODIC_PAIRS), nodes="gauss")
        uv = {1: (0, 2), 2: (0, 2), 3: (0, 1), 4: (1, 2), 5: (0, 1), 6: (1, 2)}
        case["fNf"] = np.array([[max(N3[e][uv[s][d]] for e, s in zip(case["fElem"][f], case["fESide"][f]))
                                 for d in range(2)] for f in range(case["F"])], np.int32)
        case["foff"] = np.concatenate([[0], np.cumsum(np.prod(case["fNf"] + 1, axis=1))]).astype(np.int64)
    else:
        case = mesh.periodic_box_mixed(3, N3.astype(np.int32))
    assert not np.any(case["fRot"])   # the box turns no element
    case["fRot"] = rng.choice(np.arange(8) if orders == "cubes" else [0, 2, 5, 7], case["F"]).astype(np.int32)
    Q0 = mesh.taylor_green(case, 0.3, noise=1e-3, seed=9)
    kw = dict(mach=0.3, reynolds=700.0, riemann="roe", inviscid="standard", averaging="standard", les=les)
    ora = po.Oracle(case, po.make_params(kw["mach"], kw["reynolds"], riemann="roe", les=les, nodes=nodes))
    eng = Engine(case, nodes=nodes, **kw)
    eng.set_state(Q0)
    err = po.normwise_error(eng.qdot(), ora.qdot(Q0))
    print(orders, les, nodes, err, flush=True)
    assert err.max() <= TOL
    eng.close()


@pytest.mark.parametrize("riemann", ["roe", "lxf"])
@pytest.mark.parametrize("orders", [1, 3, 4, 6, "mixed"])
def test_constant_metrics_read_once_give_the_same_bits(orders, riemann):
    """Straight elements: metrics and face frames are read once per element and face.  A zero of other
    sign at one node (which no sum sees) makes them differ, and the kernels read them by node: the
    derivative and two steps are equal, and the derivative agrees with the oracle."""
    from horses3d_amd.engine import Engine
    mixed = orders == "mixed"
    case = mesh.periodic_box_mixed(3, mesh.random_orders(27, 1, 7, 4)) if mixed else mesh.straight_box(3, orders)
    Q0 = mesh.taylor_green(case, 0.3, noise=1e-3, seed=6)
    kw = dict(mach=0.3, reynolds=700.0, riemann=riemann, les="smagorinsky")
    out = []
    for signed in (False, True):
        c = dict(case)
        if signed:
            for name in ("Ja", "normal"):
                c[name] = np.array(case[name])
                c[name][0, np.argwhere(c[name][0] == 0.0)[0, 0]] = -0.0
        eng = Engine(c, **kw)
        eng.set_state(Q0)
        qd = eng.qdot()
        t = eng.advance(2, 0.4, 0.4, t=0.0)
        out.append((qd, eng.get_state(), t))
        eng.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1]) and out[0][2] == out[1][2]
    ora = po.Oracle(case, po.make_params(0.3, 700.0, riemann=riemann, les="smagorinsky"))
    err = po.normwise_error(out[0][0], ora.qdot(Q0))
    print(orders, riemann, err, flush=True)
    assert err.max() <= TOL


@pytest.mark.parametrize("n,N", [(4, 1), (13, 4), (15, 4)])
def test_host_transfers_through_chunks_are_exact(n, N):
    """A state smaller than a staging chunk, one of several chunks that reuse the slots (11 MB) and one with a
    short last chunk (16.9 MB): set, get, a part of it, and the derivative against a copy of it; pageable
    arrays and the caller's pinned ones."""
    import ctypes as C
    from horses3d_amd.engine import Engine
    case = mesh.straight_box(n, N)
    eng = Engine(case, mach=0.2, reynolds=800.0)
    base = mesh.taylor_green(case, 0.2)
    hip, p = C.CDLL("libamdhip64.so.7"), C.c_void_p()
    assert hip.hipHostMalloc(C.byref(p), C.c_size_t(base.nbytes), C.c_uint(0)) == 0
    pinned = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), shape=base.shape)
    for k, Q in enumerate((base, mesh.taylor_green(case, 0.2, noise=1e-3, seed=2))):
        eng.set_state(Q)
        assert np.array_equal(eng.get_state(), Q)
        qd = eng.qdot()
        assert np.array_equal(eng.get_qdot(), qd)
        pinned[:] = Q
        eng.set_state(pinned)
        assert np.array_equal(eng.get_state(), Q) and np.array_equal(eng.qdot(), qd)
    eng.close()
    assert hip.hipHostFree(p) == 0


@pytest.mark.parametrize("riemann", ["roe", "lxf"])
@pytest.mark.parametrize("N,averaging", [(1, "pirozzoli"), (3, "standard"), (4, "kennedy-gruber"), (5, "ducros"), (6, "morinishi"),
                                         (7, "pirozzoli"), (2, None), (6, None)])
def test_euler_volume_kernel_matches_oracle(N, averaging, riemann):
    """The volume kernel without viscous values, split (with the pair table and, at N = 5, by rows) and
    standard form: the derivative and a step against the oracle."""
    from horses3d_amd.engine import Engine
    case = mesh.periodic_box(3, N, amplitude=0.1, phase_seed=40 + N)
    Q0 = mesh.taylor_green(case, 0.3, noise=1e-3, seed=N)
    kw = dict(riemann=riemann, euler=True, inviscid="split-form" if averaging else "standard", averaging=averaging or "standard")
    ora = po.Oracle(case, po.make_params(0.3, 700.0, **kw))
    eng = Engine(case, mach=0.3, reynolds=700.0, **kw)
    eng.set_state(Q0)
    err = po.normwise_error(eng.qdot(), ora.qdot(Q0))
    print(N, averaging, riemann, err, flush=True)
    assert err.max() <= TOL
    # one step: the increment to the bar, plus four ulp of the state it is added to
    dt = ora.max_dt(Q0, 0.4, 0.4)
    assert eng.advance(1, 0.4, 0.4, t=0.0) == pytest.approx(dt, rel=1e-13)
    Q, G = Q0.copy(), np.zeros_like(Q0)
    ora.rk3_step(Q, G, 0.0, dt)
    dq = np.abs(Q - Q0).max(axis=0)
    floor = 4.0 * np.finfo(float).eps * np.abs(Q).max(axis=0)
    assert np.all(np.abs(eng.get_state() - Q).max(axis=0) <= TOL * dq + floor)
    eng.close()
