"""The two-launch stage of Gauss-Lobatto cases of one order: every pairing of Riemann solver and
LES model (the volume kernel's template flags) at orders with whole and remainder element blocks,
against the oracle; and the two copies of the state through odd and even step counts."""
import numpy as np
import pytest

import pyoracle as po
from horses3d_amd import mesh

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


@pytest.mark.parametrize("euler", [False, True])
def test_state_copies_through_odd_and_even_steps(euler):
    """A step of three stages ends in the other copy of the state: any split of the steps, with
    host reads, derivatives and captured steps between, gives the same bits."""
    from horses3d_amd.engine import Engine
    case = mesh.periodic_box(3, 3, amplitude=0.1, phase_seed=4)
    Q0 = mesh.taylor_green(case, 0.2, noise=1e-3, seed=9)
    kw = dict(mach=0.2, reynolds=800.0, riemann="roe", euler=euler)
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
