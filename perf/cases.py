"""The workloads this engine is timed on: explicit Navier-Stokes DGSEM runs through its public
entry points (`horses3d_amd.engine`), from the reference's smallest CPU case to a case that no
cache holds, over node types, volume forms, Riemann solvers, LES models, element orders, one and
several cases per engine, resident and host-held states.

A case is a dict of plain values:
  call       how the program drives the engine: "advance" (device-resident state, CFL dt),
             "monitors" (the same, then the residuals and volume monitors of an output
             interval), "batch" (several cases in one engine), "host" (the drop-in of the
             reference's TakeRK3Step: host state in, one step, host state and derivative out)
  n          elements per side of the periodic box [-pi, pi]^3
  lo, hi     element orders: one order if equal, else (Nx, Ny, Nz) drawn per element on {lo..hi}
  nodes      "gauss-lobatto" or "gauss"
  amplitude  of the box's curvilinear deformation (0: straight elements)
  riemann, inviscid, averaging, les, euler, mach, reynolds: the physics and discretisation
  steps      RK3 steps a pass takes
  count      cases in the engine ("batch")
"""
import functools
import math
import os
import tempfile

import numpy as np
import torch

from horses3d_amd import engine as E
from horses3d_amd import mesh, specmesh

CFL = 0.4
RK_A, RK_C = (0.0, -5.0 / 9.0, -153.0 / 128.0), (1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0)
MONITORS = ("kinetic energy", "kinetic energy rate", "enstrophy", "internal energy", "entropy")

_BASE = dict(call="advance", nodes="gauss-lobatto", amplitude=0.0, riemann="roe", inviscid="standard",
             averaging="standard", les="none", euler=False, mach=0.1, reynolds=1600.0, count=1)


def _case(n, lo, hi, steps, **kw):
    return dict(_BASE, n=n, lo=lo, hi=hi, steps=steps, **kw)


def listed():
    return [
        # the reference's own CPU test size: 4,096 nodes, nothing but launches and latency
        dict(_case(4, 3, 3, 20), name="box4_n3_roe"),
        # low order on an odd box, the setting of a coarse first run
        dict(_case(15, 2, 2, 8, amplitude=0.1, riemann="lxf", averaging="morinishi", mach=0.3), name="box15_n2_lxf"),
        # one case of a parameter sweep: straight boxes of 8..24 elements, N = 3..6, Smagorinsky
        dict(_case(9, 6, 6, 4, les="smagorinsky", mach=0.7, reynolds=4000.0), name="box9_n6_smagorinsky"),
        # the single-GPU benchmark: kinetic-energy-preserving split form on a curvilinear box
        dict(_case(16, 4, 4, 5, amplitude=0.1, riemann="lxf", inviscid="split-form", averaging="pirozzoli"),
             name="box16_n4_split"),
        # an inviscid run (no gradient sweep)
        dict(_case(11, 5, 5, 4, amplitude=0.1, euler=True, inviscid="split-form", averaging="ducros", riemann="lxf",
                   mach=0.3), name="box11_n5_euler"),
        # the largest: 3.0 M nodes, split form, Roe, WALE on a strongly curvilinear box
        dict(_case(24, 5, 5, 2, amplitude=0.15, inviscid="split-form", averaging="kennedy-gruber", les="wale"),
             name="box24_n5_wale"),
        # the reference's default node type
        dict(_case(16, 4, 4, 5, nodes="gauss", amplitude=0.1), name="box16_n4_gauss"),
        # p-anisotropic elements with mortar faces, on both node types
        dict(_case(20, 2, 7, 2, mach=0.2), name="box20_p2to7"),
        dict(_case(10, 2, 5, 4, nodes="gauss", mach=0.3), name="box10_p2to5_gauss"),
        # many small cases in one engine, each with its own Mach and Reynolds numbers and dt
        dict(_case(4, 3, 3, 10, call="batch", count=64), name="batch64_box4_n3"),
        # a run with monitors every few steps, the time derivative taken at the new state
        dict(_case(12, 4, 4, 4, call="monitors", amplitude=0.1, inviscid="split-form", averaging="kennedy-gruber",
                   les="smagorinsky", mach=0.2), name="monitors_box12_n4"),
        # the drop-in inside the reference's time loop: its state in, one step, state and derivative back
        dict(_case(14, 4, 4, 1, call="host", amplitude=0.1, riemann="lxf", inviscid="split-form", averaging="pirozzoli"),
             name="host_box14_n4"),
    ]


def _nodes(case):
    """Nodes of one case (for drawn orders, their expected number)."""
    mean = np.mean([m + 1 for m in range(case["lo"], case["hi"] + 1)])
    return case["n"] ** 3 * mean ** 3


def draw(rng):
    """A case of the ranges the listed ones stand for."""
    call = rng.choices(("advance", "monitors", "batch", "host"), (14, 2, 2, 1))[0]
    kw = dict(call=call, mach=round(rng.uniform(0.1, 0.8), 3), reynolds=round(math.exp(rng.uniform(math.log(400.0), math.log(5000.0))), 1))
    kw["riemann"] = rng.choice(("roe", "lxf"))
    kw["les"] = rng.choice(("none", "none", "smagorinsky", "wale"))
    kw["amplitude"] = rng.choice((0.0, 0.1, 0.15))
    lo = hi = rng.choice((1, 2, 3, 3, 4, 4, 5, 5, 6, 7))
    if call != "batch":
        kw["nodes"] = rng.choice(("gauss-lobatto", "gauss-lobatto", "gauss-lobatto", "gauss"))
        if rng.random() < 0.2:
            lo, hi = rng.choice(((2, 4), (2, 5), (3, 6), (2, 7)))
            kw["amplitude"] = 0.0
    if kw.get("nodes") != "gauss" and rng.random() < 0.6:
        kw["inviscid"] = "split-form"
        kw["averaging"] = rng.choice(("standard", "ducros", "kennedy-gruber", "pirozzoli", "morinishi"))
    if call == "advance" and rng.random() < 0.15:
        kw.update(euler=True, les="none")
    if call == "batch":
        kw["count"] = rng.randint(5, 64)
    side = (lo + hi + 2) / 2
    top = {"batch": 2.0e5, "host": 5.0e5}.get(call, 1.5e6 if lo == hi else 8.0e5) / kw.get("count", 1)
    if kw.get("nodes") == "gauss":
        top = min(top, 6.0e5)   # the mesh reader's set-up time
    n = int(round(math.exp(rng.uniform(math.log(3.0), math.log(max(3.5, top ** (1.0 / 3.0) / side))))))
    n = max(min(n, 24 if kw.get("nodes") == "gauss" else 64), 3 if call == "batch" else 4)
    c = _case(n, lo, hi, 1, **kw)
    total = _nodes(c) * c["count"]
    c["steps"] = 1 if call == "host" else rng.randint(2, 12 if total < 2.0e5 else 4)
    return c


# ---------------------------------------------------------------------------------------
# what the program holds before the call
# ---------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=3)
def _box(n, lo, hi, nodes, amplitude):
    """The mesh, metrics and connectivity of a periodic box (the same for every state)."""
    orders = None if lo == hi else mesh.random_orders(n ** 3, lo, hi, 3)
    if nodes == "gauss" or (orders is not None and amplitude):
        fd, path = tempfile.mkstemp(suffix=".mesh")
        os.close(fd)
        try:
            specmesh.write_specmesh(path, n, amplitude, mesh.box_phases(2), bface_order=min(lo, 4))
            return E.read_specmesh(path, N=lo, orders=orders, periodic=dict(specmesh.PERIODIC_PAIRS), nodes=nodes)
        finally:
            os.remove(path)
    if orders is not None:
        return mesh.periodic_box_mixed(n, orders)
    return mesh.periodic_box(n, lo, amplitude=amplitude, phase_seed=2) if amplitude else mesh.straight_box(n, lo)


def _mesh_of(case):
    return _box(case["n"], case["lo"], case["hi"], case["nodes"], case["amplitude"])


def _physics(case, mach=None, reynolds=None):
    return dict(mach=mach or case["mach"], reynolds=reynolds or case["reynolds"], riemann=case["riemann"],
                inviscid=case["inviscid"], averaging=case["averaging"], les=case["les"], euler=case["euler"],
                nodes=case["nodes"])


def _members(case, seed):
    """(mach, reynolds) of each case of the engine."""
    if case["call"] != "batch":
        return [(case["mach"], case["reynolds"])]
    r = np.random.default_rng([seed, 1])
    return [(float(r.uniform(0.1, 0.8)), float(np.exp(r.uniform(np.log(400.0), np.log(5000.0)))))
            for _ in range(case["count"])]


def _states(case, seed):
    """The initial states: Taylor-Green vortices of random phase with a small velocity noise."""
    r = np.random.default_rng([seed, 2])
    box = _mesh_of(case)
    return [mesh.taylor_green(box, m, phase=tuple(r.uniform(0.0, 2.0 * np.pi, 3)), noise=1e-3, seed=int(r.integers(1 << 30)))
            for m, _ in _members(case, seed)]


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, box, who = case, _mesh_of(case), _members(case, seed)
    Q = np.concatenate(_states(case, seed))
    if case["call"] == "batch":
        s.eng = E.MultiEngine([box] * len(who), [_physics(case, m, re) for m, re in who])
    else:
        s.eng = E.Engine(box, **_physics(case))
    if case["call"] == "host":
        s.eng.set_state(Q)
        s.Q, s.dt = Q, 0.5 * s.eng.max_dt(CFL, CFL)
        return s
    s.Q = torch.from_numpy(Q).cuda()
    s.out = torch.empty_like(s.Q)
    if case["call"] == "monitors":
        s.eng.set_ctd_after_steps(True)
    if case["lo"] != case["hi"]:
        s.eng.set_state(Q)
        s.eng.set_tiling(1)
    torch.cuda.synchronize()
    return s


def run(s):
    eng, case, lib = s.eng, s.case, E.load_library()
    if case["call"] == "host":
        eng.set_state(s.Q)
        eng.rk3_step(0.0, s.dt)
        return {"Q": eng.get_state(), "QDot": eng.get_qdot()}
    out = {"Q": s.out}
    lib.hx3d_set_state_device(eng.h, s.Q.data_ptr())
    if case["call"] == "batch":
        eng.advance(case["steps"], CFL, CFL)
        lib.hx3d_get_state_device(eng.h, s.out.data_ptr())
        eng.synchronize()
        return out
    out["t"] = np.float64(eng.advance(case["steps"], CFL, CFL, t=0.0))
    lib.hx3d_get_state_device(eng.h, s.out.data_ptr())
    if case["call"] == "monitors":
        out["residuals"] = eng.residuals()
        out["monitors"] = np.array([eng.volume_monitor(m) for m in MONITORS])
    return out


def work(case):
    """Bytes and operations of one pass.  Bytes: what each stage reads and writes of arrays that
    outlive it: the state and the RK register in and out, the metrics and the Jacobian, and the
    faces' normals and surface Jacobians (10 + 10 + 10 doubles a node, 4 a face node), with the
    exchange between elements (both traces of the state and of the four viscous fluxes, 18
    doubles a face node).  Operations: the derivative and flux sums along the lines, the
    two-point fluxes of the split form and the point-wise fluxes."""
    n1 = np.mean([m + 1 for m in range(case["lo"], case["hi"] + 1)])
    nodes = _nodes(case) * case["count"]
    fnodes = 3.0 * nodes / n1
    split = case["inviscid"] == "split-form"
    stage_bytes = 8.0 * (30.0 * nodes + 22.0 * fnodes)
    grad = 0.0 if case["euler"] else 30.0 * n1 + 75.0 + 100.0
    pairs = 1.5 * (n1 - 1.0) * 52.0 + 3.0 * n1 * 18.0 if split else 30.0 * n1 + 90.0
    stage_flops = nodes * (grad + pairs + 120.0) + fnodes * 250.0
    io = 8.0 * nodes * (10.0 + (5.0 if case["call"] == "host" else 0.0))
    return {"bytes": 3.0 * case["steps"] * stage_bytes + 2.0 * io, "flops": 3.0 * case["steps"] * stage_flops}


# ---------------------------------------------------------------------------------------
# the same passes in plain torch, 64 bits
# ---------------------------------------------------------------------------------------
def _rule(gauss, N):
    """Nodes and weights of the Gauss or Gauss-Lobatto rule of order N."""
    if gauss:
        return np.polynomial.legendre.leggauss(N + 1)
    c = np.zeros(N + 1)
    c[N] = 1.0
    L = np.polynomial.Legendre(c)
    x = np.concatenate([[-1.0], np.sort(L.deriv().roots().real), [1.0]])
    for _ in range(3):   # polish the interior nodes
        x[1:-1] -= L.deriv()(x[1:-1]) / L.deriv(2)(x[1:-1])
    return x, 2.0 / (N * (N + 1) * L(x) ** 2)


def _lagrange(x, y):
    """T[i, j]: the Lagrange polynomial of node x[j] at y[i]."""
    T = np.ones((len(y), len(x)))
    for j in range(len(x)):
        for m in range(len(x)):
            if m != j:
                T[:, j] *= (y - x[m]) / (x[j] - x[m])
    return T


def _derivative(x):
    n = len(x)
    D = np.zeros((n, n))
    for i in range(n):
        for j in range(n):
            if i != j:
                D[i, j] = np.prod([(x[i] - x[m]) / (x[j] - x[m]) for m in range(n) if m not in (i, j)]) / (x[j] - x[i])
        D[i, i] = -D[i].sum()
    return D


class _Reference:
    """The time derivative, MaxTimeStep and monitors of one case.  Node arrays are (component,
    element, k, j, i), face arrays (component, face, b, a), both padded to the largest order;
    padded nodes hold a state of rest and are masked out of every result."""

    AXIS, PLUS = (1, 1, 2, 0, 2, 0), (0, 1, 0, 1, 1, 0)   # of the slots front, back, bottom, right, top, left
    UV = ((0, 2), (0, 2), (0, 1), (1, 2), (0, 1), (1, 2))

    def __init__(self, box, case, mach, reynolds):
        dev = self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.c = case
        N = np.asarray(box["N"])
        K, F = int(box["K"]), int(box["F"])
        P = self.P = int(N.max()) + 1
        gauss = case["nodes"] == "gauss"
        put = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)
        rules = {m: _rule(gauss, m) for m in range(1, P)}

        def padded(f, shape):
            t = np.zeros((P,) + shape)
            for m in range(1, P):
                a = f(m)
                t[m][tuple(slice(0, z) for z in np.shape(a))] = a
            return t
        D = padded(lambda m: _derivative(rules[m][0]), (P, P))
        w = padded(lambda m: rules[m][1], (P,))
        hat = padded(lambda m: _derivative(rules[m][0]).T * rules[m][1][None, :] / rules[m][1][:, None], (P, P))
        v = [padded(lambda m: _lagrange(rules[m][0], np.array([s]))[0], (P,)) for s in (-1.0, 1.0)]
        self.one = bool((N == N[0, 0]).all())
        sel = (lambda t, d: put(t[N[:1, d]])) if self.one else (lambda t, d: put(t[N[:, d]]))
        self.D, self.hat = [sel(D, d) for d in range(3)], [sel(hat, d) for d in range(3)]
        sharp = 2.0 * D
        for m in range(1, P):
            sharp[m, 0, 0] += 1.0 / w[m, 0]
            sharp[m, m, m] -= 1.0 / w[m, m]
        self.sharp = [sel(sharp, d) for d in range(3)]
        self.v = [[sel(v[s], d) for d in range(3)] for s in range(2)]
        wi = np.where(w > 0, 1.0 / np.where(w > 0, w, 1.0), 0.0)
        self.b = [[sel(v[s] * wi, d) for d in range(3)] for s in range(2)]
        self.dxi = [put(np.array([0.0] + [1.0 / (rules[m][0][1] - rules[m][0][0]) for m in range(1, P)])[N[:, d]])[:, None, None, None]
                    for d in range(3)]
        # where node g = off[e] + i + nx (j + ny k) sits in the padded arrays
        ids = np.full((K, P, P, P), -1, np.int64)
        off = np.asarray(box["off"])
        for nx, ny, nz in np.unique(N, axis=0):
            e = np.nonzero((N == (nx, ny, nz)).all(1))[0]
            loc = np.arange((nx + 1) * (ny + 1) * (nz + 1)).reshape(nz + 1, ny + 1, nx + 1)
            ids[e, :nz + 1, :ny + 1, :nx + 1] = off[e][:, None, None, None] + loc
        self.valid = put(ids >= 0)
        self.ids = put(np.maximum(ids, 0))
        self.where = put(np.nonzero(ids.reshape(-1) >= 0)[0])
        self.order = put(ids.reshape(-1)[ids.reshape(-1) >= 0])
        self.Ja = self._spread(put(box["Ja"]), 0.0).reshape(3, 3, K, P, P, P)
        self.J = self._spread(put(box["J"])[:, None], 1.0)[0]
        wn = [put(w[N[:, d]]) for d in range(3)]
        self.w = wn[2][:, :, None, None] * wn[1][:, None, :, None] * wn[0][:, None, None, :] * self.valid
        nn = put(np.prod(N + 1, axis=1))
        self.delta = (((self.w * self.J).sum((1, 2, 3)) / nn) ** (1.0 / 3.0))[:, None, None, None]
        # faces (all of rotation 0): element and slot of each side, face order, interpolation both ways
        assert not np.any(box["fRot"])
        el, sl = np.asarray(box["fElem"]), np.asarray(box["fESide"]) - 1
        self.side = [(put(el[:, s]), put(sl[:, s])) for s in range(2)]
        uv = np.array(self.UV)
        Ns = [np.stack([N[el[:, s], uv[sl[:, s], d]] for d in range(2)], 1) for s in range(2)]
        Nf = np.maximum(Ns[0], Ns[1])
        self.To = self.Back = None
        if not self.one:
            T, B = np.zeros((P, P, P, P)), np.zeros((P, P, P, P))
            for m in range(1, P):
                for k in range(m, P):
                    t = np.eye(m + 1) if k == m else _lagrange(rules[m][0], rules[k][0])
                    T[m, k, :k + 1, :m + 1] = t
                    B[m, k, :m + 1, :k + 1] = t.T * rules[k][1][None, :] / rules[m][1][:, None]
            self.To = [[put(T[Ns[s][:, d], Nf[:, d]]) for d in range(2)] for s in range(2)]
            self.Back = [[put(B[Ns[s][:, d], Nf[:, d]]) for d in range(2)] for s in range(2)]
        q = np.arange(P)
        fv = (q[None, None, :] <= Nf[:, 0][:, None, None]) & (q[None, :, None] <= Nf[:, 1][:, None, None])
        foff = np.concatenate([[0], np.cumsum(np.prod(Nf + 1, axis=1))])
        fid = foff[:F, None, None] + q[None, None, :] + (Nf[:, 0] + 1)[:, None, None] * q[None, :, None]
        fid = put(np.where(fv, fid, 0))
        self.fvalid = put(fv)
        self.n = torch.where(self.fvalid, put(box["normal"]).T[:, fid], 0.0)
        self.sj = torch.where(self.fvalid, put(box["fjac"])[fid], 0.0)
        wf = [put(w[Nf[:, d]]) for d in range(2)]
        self.fdelta = torch.sqrt((self.sj * wf[1][:, :, None] * wf[0][:, None, :]).sum((1, 2)) / put(np.prod(Nf + 1, axis=1)))[:, None, None]
        # constants
        self.g, self.gM2 = 1.4, 1.4 * mach * mach
        self.mu0 = 0.0 if case["euler"] else 1.0 / reynolds
        self.to_kappa = 0.0 if case["euler"] else 1.0 / (0.4 * mach * mach * 0.72)
        self.les_c = {"none": 0.0, "smagorinsky": 0.2, "wale": 0.325}[case["les"]]

    def _spread(self, x, pad):
        return torch.where(self.valid, x.T[:, self.ids], pad)

    def state(self, Q):
        rest = torch.tensor([1.0, 0.0, 0.0, 0.0, 2.5 / self.gM2], dtype=torch.float64, device=self.dev)
        return torch.where(self.valid, torch.as_tensor(Q, device=self.dev).T[:, self.ids], rest[:, None, None, None, None])

    def packed(self, Q):
        out = torch.empty((len(self.order), Q.shape[0]), dtype=torch.float64, device=self.dev)
        out[self.order] = Q.reshape(Q.shape[0], -1).T[self.where]
        return out

    # -- lines and traces
    @staticmethod
    def _line(M, A, d):
        """sum_l M[e, i, l] A[..., l, ...] along reference direction d."""
        A = A.movedim(-1 - d, -1)
        out = 0.0
        for l in range(M.shape[-1]):
            out = out + A[..., l:l + 1] * M[:, None, None, :, l]
        return out.movedim(-1, -1 - d)

    def _traces(self, A):
        """The values on both sides of every face, at the face's order: two (C, F, P, P)."""
        ends = []
        for s in range(6):
            B, v = A.movedim(-1 - self.AXIS[s], -1), self.v[self.PLUS[s]][self.AXIS[s]]
            ends.append(sum(B[..., l] * v[:, None, None, l] for l in range(self.P)))
        ends = torch.stack(ends, 2)
        out = []
        for s in range(2):
            t = ends[:, self.side[s][0], self.side[s][1]]
            if self.To:
                t = self._face(self.To[s], t)
            out.append(t)
        return out

    @staticmethod
    def _face(T, A):
        n = A.shape[-1]
        B = sum(A[..., l:l + 1] * T[0][:, None, :, l] for l in range(n))
        return sum(B[..., l:l + 1, :] * T[1][:, :, l, None] for l in range(n))

    def _surface(self, left, right):
        """The surface integral of face values (C, F, P, P), each side's given, at every node."""
        C, K = left.shape[0], self.J.shape[0]
        slots = torch.zeros((C, K, 6, self.P, self.P), dtype=torch.float64, device=self.dev)
        for s, f in enumerate((left, right)):
            slots[:, self.side[s][0], self.side[s][1]] = self._face(self.Back[s], f) if self.Back else f
        out = 0.0
        for s in range(6):
            d = self.AXIS[s]
            b = self.b[self.PLUS[s]][d]
            t = slots[:, :, s].unsqueeze(-1) * b[:, None, None, :]
            out = out + t.movedim(-1, -1 - d)
        return out

    # -- physics
    def _prim(self, q):
        u = q[1:4] / q[0]
        p = (self.g - 1.0) * (q[4] - 0.5 * (q[1:4] * u).sum(0))
        return q[0], u, p, q[4]

    def _euler(self, q, n):
        r, u, p, rE = self._prim(q)
        un = (u * n).sum(0)
        return torch.cat([(r * un)[None], q[1:4] * un + p * n, ((rE + p) * un)[None]])

    def _average(self, a, b, n):
        """The two-point flux of the case's averaging along n."""
        kind = self.c["averaging"]
        if kind == "standard":
            return 0.5 * (self._euler(a, n) + self._euler(b, n))
        ra, ua, pa, Ea = self._prim(a)
        rb, ub, pb, Eb = self._prim(b)
        u, p = 0.5 * (ua + ub), 0.5 * (pa + pb)
        un = (u * n).sum(0)
        if kind == "ducros":
            m = 0.5 * (a + b)
            return torch.cat([(m[0] * un)[None], m[1:4] * un + p * n, ((m[4] + p) * un)[None]])
        if kind == "morinishi":
            ma, mb = a[1:4], b[1:4]
            m = 0.5 * ((ma + mb) * n).sum(0)
            na, nb = (ma * n).sum(0), (mb * n).sum(0)
            cp = self.g / (self.g - 1.0)
            e = 0.5 * cp * ((ua * n).sum(0) * pa + (ub * n).sum(0) * pb)
            e = e + (0.25 * (na * ua + nb * ub) * (ua + ub) - 0.25 * (na * ua * ua + nb * ub * ub)).sum(0)
            return torch.cat([m[None], m * u + p * n, e[None]])
        r = 0.5 * (ra + rb)
        if kind == "kennedy-gruber":
            e = r * un * 0.5 * (Ea / ra + Eb / rb) + p * un
        else:
            e = r * un * 0.5 * ((Ea + pa) / ra + (Eb + pb) / rb)
        return torch.cat([(r * un)[None], (r * un) * u + p * n, e[None]])

    def _riemann(self, L, R):
        n, g = self.n, self.g
        rL, uL, pL, EL = self._prim(L)
        rR, uR, pR, ER = self._prim(R)
        nL, nR = (uL * n).sum(0), (uR * n).sum(0)
        if self.c["riemann"] == "lxf":
            lam = torch.maximum(nL.abs() + torch.sqrt(g * pL / rL), nR.abs() + torch.sqrt(g * pR / rR))
            return self._average(L, R, n) - 0.5 * lam * (R - L)
        HL, HR = (EL + pL) / rL, (ER + pR) / rR
        s = torch.sqrt(rL * rR)
        wL = rL / (rL + s)
        u, H = wL * uL + (1.0 - wL) * uR, wL * HL + (1.0 - wL) * HR
        c2 = (g - 1.0) * (H - 0.5 * (u * u).sum(0))
        c, un = torch.sqrt(c2), (u * n).sum(0)
        sg = torch.where(un >= 0.0, 1.0, -1.0)   # the wave facing the flow: u - c, or u + c
        amp = 0.5 * ((pR - pL) / c2 - sg * (nR - nL) * s / c)
        lam = sg * un - c
        eps = torch.clamp(-lam.abs() - sg * (g + 1.0) / 4.0 * c / s * amp, min=0.0)
        k = amp * (torch.clamp(lam, max=0.0) - 0.5 * eps)
        side = torch.where(un >= 0.0, self._euler(L, n), self._euler(R, n))
        return side + torch.cat([k[None], k * (u - sg * c * n), (k * (H - sg * un * c))[None]])

    def _velocity_gradient(self, q, U):
        """dv[c][d] = d u_c / d x_d from the state's gradients U[d][v]."""
        return [[(U[d][1 + c] - q[1 + c] / q[0] * U[d][0]) / q[0] for d in range(3)] for c in range(3)]

    def _viscous(self, q, U, delta):
        """Viscous fluxes [5][3] of the state and its gradients."""
        r, u, p, rE = self._prim(q)
        dv = self._velocity_gradient(q, U)
        T = self.gM2 * p / r
        S = 198.6 / 520.0
        mu = self.mu0 * (1.0 + S) / (T + S) * T * torch.sqrt(T)
        les = self.c["les"]
        if les != "none":
            G = dv
            sym = [[0.5 * (G[a][b] + G[b][a]) for b in range(3)] for a in range(3)]
            ss = sum(sym[a][b] ** 2 for a in range(3) for b in range(3))
            if les == "smagorinsky":
                X = torch.sqrt(2.0 * ss)
            else:
                G2 = [[sum(G[a][m] * G[m][b] for m in range(3)) for b in range(3)] for a in range(3)]
                tr = (G2[0][0] + G2[1][1] + G2[2][2]) / 3.0
                sd = sum((0.5 * (G2[a][b] + G2[b][a]) - (tr if a == b else 0.0)) ** 2 for a in range(3) for b in range(3))
                X = torch.where((ss < 1e-8) & (sd < 1e-8), 0.0, sd ** 1.5 / torch.clamp(ss ** 2.5 + sd ** 1.25, min=1e-300))
            mt = r * (self.les_c * delta) ** 2 * X
        else:
            mt = 0.0
        kappa = (mu + mt) * self.to_kappa
        mu = mu + mt
        div = dv[0][0] + dv[1][1] + dv[2][2]
        F = [[torch.zeros_like(r)] * 3]
        for c in range(3):
            F.append([mu * (dv[c][d] + dv[d][c] - (2.0 / 3.0 * div if c == d else 0.0)) for d in range(3)])
        heat = []
        for d in range(3):
            # T = (gamma - 1) gamma M^2 (E - |u|^2 / 2)
            dT = (self.g - 1.0) * self.gM2 * ((U[d][4] - rE / r * U[d][0]) / r - sum(u[c] * dv[c][d] for c in range(3)))
            heat.append(sum(F[1 + c][d] * u[c] for c in range(3)) + kappa * dT)
        F.append(heat)
        return F

    def gradients(self, q):
        L, R = self._traces(q)
        jump = 0.5 * (R - L) * self.sj
        d = [self._line(self.D[m], q, m) for m in range(3)]
        out = []
        for c in range(3):
            lift = jump * self.n[c]
            out.append((sum(d[m] * self.Ja[m, c] for m in range(3)) + self._surface(lift, lift)) / self.J)
        return torch.stack(out)

    def qdot(self, q):
        K = self.J.shape[0]
        L, R = self._traces(q)
        rest = torch.tensor([1.0, 0.0, 0.0, 0.0, 2.5 / self.gM2], dtype=torch.float64, device=self.dev)[:, None, None, None]
        L, R = torch.where(self.fvalid, L, rest), torch.where(self.fvalid, R, rest)
        face = self._riemann(L, R)
        Fv = None
        if not self.c["euler"]:
            U = self.gradients(q)
            UL, UR = self._traces(U.reshape(15, K, self.P, self.P, self.P))
            a = self._viscous(L, UL.reshape(3, 5, *UL.shape[1:]), self.fdelta)
            b = self._viscous(R, UR.reshape(3, 5, *UR.shape[1:]), self.fdelta)
            face = face - torch.stack([sum(0.5 * (a[v][d] + b[v][d]) * self.n[d] for d in range(3)) for v in range(5)])
            del UL, UR, a, b
            Fv = self._viscous(q, U, self.delta)
        face = torch.where(self.fvalid, face * self.sj, 0.0)
        out = self._surface(face, -face)
        del face
        acc = 0.0
        for d in range(3):
            Ja = self.Ja[d]
            visc = 0.0 if Fv is None else torch.stack([sum(Fv[v][c] * Ja[c] for c in range(3)) for v in range(5)])
            if self.c["inviscid"] == "standard":
                acc = acc + self._line(self.hat[d], self._euler(q, Ja) - visc, d)
                continue
            if Fv is not None:
                acc = acc - self._line(self.hat[d], visc, d)
            qm, Jm = q.movedim(-1 - d, -1), Ja.movedim(-1 - d, -1)
            S = self.sharp[d]
            split = 0.0
            for l in range(self.P):
                f = self._average(qm, qm[..., l:l + 1], 0.5 * (Jm + Jm[..., l:l + 1]))
                split = split + f * S[:, None, None, :, l]
            acc = acc - split.movedim(-1, -1 - d)
        return torch.where(self.valid, (acc - out) / self.J, 0.0)

    def max_dt(self, q):
        r, u, p, _ = self._prim(q)
        lam = u.abs() + torch.sqrt(self.g * p / r)
        conv = sum((self.Ja[d] * lam).sum(0).abs() * self.dxi[d] for d in range(3))
        lim = [torch.where(self.valid, CFL * self.J.abs() / conv, math.inf).min()]
        if not self.c["euler"]:
            T, S = self.gM2 * p / r, 198.6 / 520.0
            mu = (1.0 + S) / (T + S) * T * torch.sqrt(T)
            visc = mu * sum(self.dxi[d] ** 2 * self.Ja[d].sum(0).abs() for d in range(3))
            lim.append(torch.where(self.valid, CFL * self.J.abs() / visc, math.inf).min())
        return torch.stack(lim).min()

    def step(self, q, dt):
        """One RK3 step; also the last stage's derivative."""
        G = torch.zeros_like(q)
        for a, c in zip(RK_A, RK_C):
            qd = self.qdot(q)
            G = a * G + qd
            q = q + c * dt * G
        return q, qd

    def advance(self, Q, steps):
        q, t = self.state(Q), 0.0
        for _ in range(steps):
            dt = self.max_dt(q)
            q, _ = self.step(q, dt)
            t = t + float(dt)
        return q, t

    def monitors(self, q):
        qd, U = self.qdot(q), self.gradients(q)
        r, u, p, rE = self._prim(q)
        dv = self._velocity_gradient(q, U)
        curl2 = (dv[2][1] - dv[1][2]) ** 2 + (dv[0][2] - dv[2][0]) ** 2 + (dv[1][0] - dv[0][1]) ** 2
        mean = lambda f: float((self.w * self.J * f).sum() / (self.w * self.J).sum())
        vals = [mean(0.5 * r * (u * u).sum(0)), mean((u * qd[1:4]).sum(0) - 0.5 * (u * u).sum(0) * qd[0]), 0.5 * mean(curl2),
                mean(rE), mean(torch.log(p) - self.g * torch.log(r))]
        return qd.abs().amax((1, 2, 3, 4)).cpu().numpy(), np.array(vals)


def exact(case, seed):
    if case["call"] == "batch":   # independent cases, one after the other
        box, outs = _mesh_of(case), []
        for (m, re), Q in zip(_members(case, seed), _states(case, seed)):
            ref = _Reference(box, case, m, re)
            outs.append(ref.packed(ref.advance(Q, case["steps"])[0]))
        return {"Q": torch.cat(outs)}
    ref = _Reference(_mesh_of(case), case, case["mach"], case["reynolds"])
    Q = _states(case, seed)[0]
    if case["call"] == "host":
        q = ref.state(Q)
        q, qd = ref.step(q, 0.5 * ref.max_dt(q))
        return {"Q": ref.packed(q).cpu().numpy(), "QDot": ref.packed(qd).cpu().numpy()}
    q, t = ref.advance(Q, case["steps"])
    out = {"Q": ref.packed(q), "t": np.float64(t)}
    if case["call"] == "monitors":
        out["residuals"], out["monitors"] = ref.monitors(q)
    return out
