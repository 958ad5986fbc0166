"""Performance cases of the engine: the work its users have it do, through the public entry points.

Every case is one call sequence of a user's program:
  rhs     fx_rhs_noalloc on device arrays (a harness or a host code that keeps its state on the GPU)
  dropin  Engine.upload + Engine.rhs: the host-side Runge-Kutta form, one RHS per stage with U going up
          and Ut coming back (DeviceResident=F of the driver)
  run     Engine.upload + Engine.run + Engine.download: a simulation segment between two outputs, or one
          per-request solve
  serve   Server.submit of a burst of mixed requests and Server.wait
The meshes are the periodic box meshes of the Fortran host (Cartesian, or warped with curved elements).
Initial states are those of the configurations in bench.py and fluxo_amd.workloads, moved by a seeded
random shift of the origin (density wave, Taylor-Green), a seeded centre (blast) or carrying the seeded
random perturbation (Orszag-Tang).
"""
import ctypes as C
import functools
import math
import random

import numpy as np
import torch

from fluxo_amd import native as NT
from fluxo_amd import workloads as W
from fluxo_amd.mesh import box_mesh

MU0 = 1.0 / 1600  # Re = 1600


def _run(name, flow, N, K, steps, warp, **kw):
    K = [K] * 3 if isinstance(K, int) else list(K)
    d = dict(name=name, kind="run", flow=flow, N=N, Kx=K[0], Ky=K[1], Kz=K[2], steps=steps, warp=warp,
             parabolic=False, lifting=1, fp32=False, cfl=0.9)
    d.update(kw)
    return d


def listed():
    return [
        # the smallest call: one Euler right-hand side on device arrays, 8^3 elements; latency and launches
        dict(_run("rhs_euler_n3_8", "wave", 3, 8, 1, False), kind="rhs"),
        # the drop-in form of the reference's host loop: one Navier-Stokes RHS with U up and Ut down
        dict(_run("dropin_ns_n3_16", "tgv", 3, 16, 1, True, parabolic=True), kind="dropin"),
        # Euler density wave, 8^3, N=3, 100 steps: a small solve, bound by launches and gaps
        _run("wave_euler_n3_8", "wave", 3, 8, 100, False),
        # one inviscid request of the serving mix alone: highest degree, an odd medium mesh
        _run("tgv_euler_n5_13", "tgv", 5, 13, 50, False, cfl=0.5),
        # the headline: Navier-Stokes Taylor-Green vortex, 32^3 warped elements, N=3, BR1
        _run("tgv_ns_n3_32", "tgv", 3, 32, 40, True, parabolic=True),
        # the same workload with FP32 flux differencing
        _run("tgv_ns_n3_32_fp32", "tgv", 3, 32, 40, True, parabolic=True, fp32=True),
        # Navier-Stokes at N=4 on a ragged box
        _run("tgv_ns_n4_15x14x13", "tgv", 4, (15, 14, 13), 50, True, parabolic=True, cfl=0.5),
        # BR2 lifting at the lowest degree
        _run("tgv_ns_br2_n2_24", "tgv", 2, 24, 40, True, parabolic=True, lifting=2),
        # resistive GLM-MHD Orszag-Tang, 24^3 warped elements, N=4
        _run("ot_mhd_n4_24", "ot", 4, 24, 30, True, parabolic=True, cfl=0.5),
        # the same equations with FP32 flux differencing on a medium mesh
        _run("ot_mhd_n4_15_fp32", "ot", 4, 15, 40, True, parabolic=True, cfl=0.5, fp32=True),
        # Sedov blast with sub-cell shock capturing, 40^3 elements, N=3: its first 20 steps, in which
        # rounding differences are not yet amplified by the corners near vacuum
        _run("sedov_n3_40", "sedov", 3, 40, 20, False, cfl=0.5),
        # a burst of 16 requests of the serving stream (N 2..5, Euler and Navier-Stokes)
        dict(name="serve_mix_16", kind="serve", requests=16, steps=50, Kmax=16),
    ]


def _nodes(c):
    return c["Kx"] * c["Ky"] * c["Kz"] * (c["N"] + 1) ** 3


# most node-stages of a drawn segment, below the work of the largest listed one (tgv_ns_n3_32)
_MAX_NODE_STEPS = 70e6


def draw(rng):
    """One more case: the same calls over their ranges of degree, mesh size and options."""
    kind = rng.choice(["rhs", "dropin", "run", "run", "run", "run", "run", "run", "serve"])
    if kind == "serve":
        return dict(kind="serve", requests=rng.randint(2, 20), steps=rng.choice([10, 20, 50]),
                    Kmax=rng.randint(6, 16))
    flow = rng.choice(["wave", "tgv", "tgv", "ot", "sedov"]) if kind == "run" else rng.choice(["wave", "tgv"])
    N = 3 if flow == "sedov" else rng.choice([2, 3, 4, 5])
    top = {"rhs": 2.0e5, "dropin": 5e5}.get(kind, 2.2e6 if flow != "ot" else 1.7e6)
    low = 3.0e5 if flow == "sedov" else 2.0e4  # the blast's pulse needs a mesh that resolves it
    nodes = math.exp(rng.uniform(math.log(low), math.log(top)))
    k = (nodes / (N + 1) ** 3) ** (1.0 / 3.0)
    K = [max(4, int(round(k * math.exp(rng.uniform(-0.15, 0.15))))) for _ in range(3)]
    c = _run("", flow, N, K, 1, flow == "ot" or (flow != "sedov" and rng.random() < 0.5))
    del c["name"]
    c["kind"] = kind
    c["parabolic"] = flow in ("tgv", "ot") and rng.random() < 0.75
    if c["parabolic"] and flow == "tgv" and N <= 4 and rng.random() < 0.25:
        c["lifting"] = 2
    c["fp32"] = kind == "run" and flow in ("tgv", "ot") and rng.random() < 0.3
    c["cfl"] = 0.5 if (flow in ("ot", "sedov") or N >= 4) else 0.9
    if kind == "run":
        weight = 2.0 if flow == "ot" else 1.0
        c["steps"] = int(max(5, min(rng.choice([10, 20] if flow == "sedov" else [10, 20, 40]), _MAX_NODE_STEPS / (weight * _nodes(c)))))
    return c


# ---------------------------------------------------------------------------------------
# what a user's program holds before the call

_DOMAIN = {"wave": ((0.0,) * 3, (2.0,) * 3), "tgv": ((-math.pi,) * 3, (2.0 * math.pi,) * 3),
           "ot": ((0.0,) * 3, (1.0,) * 3), "sedov": ((-1.5,) * 3, (3.0,) * 3)}


@functools.lru_cache(maxsize=64)
def _box(K, N, flow, warp):
    x0, L = _DOMAIN[flow]
    return box_mesh(K, N, x0=x0, length=L, Ngeo=3 if warp else 1, warp=warp)


def _mesh(c):
    # the mesh is a simulation's configuration, built once and shared by its runs (as workloads.MeshCache does)
    return _box((c["Kx"], c["Ky"], c["Kz"]), c["N"], c["flow"], c["warp"])


def _state(c, mesh, seed):
    rng = np.random.default_rng([seed, 11])
    x = mesh["Elem_xGP"]
    if c["flow"] == "ot":
        return W.perturbed_orszag_tang(x, seed)
    shift = rng.uniform(-1.0, 1.0, 3)
    if c["flow"] == "wave":
        return W.density_wave(x + shift, amp=0.1 * rng.uniform(0.8, 1.2))
    if c["flow"] == "sedov":
        return W.sedov_blast(x, center=tuple(0.2 * shift))
    return W.taylor_green(x + math.pi * shift)


def _options(c):
    o = dict(volume_flux=32, riemann=1, parabolic=c["parabolic"], lifting=c["lifting"],
             precision=NT.FX_PREC_FP32_SPLIT if c["fp32"] else NT.FX_PREC_FP64)
    if c["parabolic"]:
        o.update(mu0=MU0, Pr=0.72)
    if c["flow"] == "sedov":
        o.update(nfvse=True, alpha_max=0.5, alpha_min=0.01, sweeps=1, prop_factor=0.5)
    return o


_MHD_RES = dict(mu=0.0, eta=1.0e-3, Pr=0.72)


def prepare(case, seed):
    c = dict(case)
    if c["kind"] == "serve":
        return _prepare_serve(c, seed)
    mesh = _mesh(c)
    U = _state(c, mesh, seed)
    if c["kind"] == "rhs":
        m, keep = NT.fx_mesh(), []
        for field, key in NT._MESH_KEYS:
            keep.append(torch.from_numpy(np.ascontiguousarray(mesh[key])).cuda())
            setattr(m, field, keep[-1].data_ptr())
        cfg = NT.make_config(c["N"], mesh["nElems"], mesh["nSides"], **_options(c))
        Ud = torch.from_numpy(U).cuda()
        return dict(kind="rhs", cfg=cfg, mesh=m, keep=keep, U=Ud, Ut=torch.empty_like(Ud))
    if c["flow"] == "ot":
        e = NT.MhdEngine(mesh, precision=_options(c)["precision"], resistive=_MHD_RES if c["parabolic"] else None)
    else:
        e = NT.Engine(mesh, **_options(c))
    return dict(kind=c["kind"], engine=e, U=U, steps=c["steps"], cfl=c["cfl"])


def _requests(c, seed):
    """The requests of a burst: degree, size and flow drawn as in the serving stream."""
    rng = random.Random(c["requests"] * 1000003 + c["Kmax"])
    reqs = []
    for s in range(c["requests"]):
        K = int(round(math.exp(rng.uniform(math.log(4.0), math.log(c["Kmax"])))))
        flow = "wave" if s % 2 == 0 else "tgv"
        r = _run("", flow, rng.randint(2, 5), K, c["steps"], False, parabolic=s % 4 == 3, cfl=0.5)
        mesh = _mesh(r)
        reqs.append((mesh, _state(r, mesh, seed * 1000 + s), r["parabolic"]))
    return reqs


def _prepare_serve(c, seed):
    # room for the requests of every pass
    srv = NT.Server(mu0=MU0, Pr=0.72, cfl=0.5, dfl=0.5, hbm_budget=32 << 30, max_requests=200000)
    return dict(kind="serve", server=srv, requests=_requests(c, seed), steps=c["steps"])


def run(state):
    kind = state["kind"]
    if kind == "rhs":
        rc = NT.lib().fx_rhs_noalloc(C.byref(state["cfg"]), C.byref(state["mesh"]), state["U"].data_ptr(),
                                     state["Ut"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        if rc:
            raise NT.FxError(NT.lib().fx_last_error().decode())
        return state["Ut"]
    if kind == "dropin":
        state["engine"].upload(state["U"])
        return state["engine"].rhs()
    if kind == "run":
        e = state["engine"]
        e.upload(state["U"])
        t, dt, err = e.run(state["steps"], state["cfl"], state["cfl"])
        return {"U": e.download(), "t": t, "dt": dt, "err": err}
    srv = state["server"]
    sub = [srv.submit(m, U, state["steps"], parabolic=p) for m, U, p in state["requests"]]
    srv.wait(timeout=300.0)
    for i, _ in sub:  # the results are this program's now
        srv._keep.pop(i)
    return [out for _, out in sub]


# flop per node and stage of the algorithm (profiles/flops.json, all variables)
_FLOPS = {"wave": 681.0, "sedov": 795.0, "tgv": 681.0, "tgv_ns": 1577.0, "ot": 4300.0, "ot_res": 5893.0}


def _stage_work(nodes, nvar, fp32, flops, stages):
    # U and Ut_tmp read and written, the metrics (nine, in single precision for FP32) and sJ read
    metric = 4 if fp32 else 8
    return nodes * stages * (8 * (4 * nvar + 1) + 9 * metric), nodes * stages * flops


def work(case):
    c = case
    if c["kind"] == "serve":
        b = f = 0.0
        rng = random.Random(c["requests"] * 1000003 + c["Kmax"])
        for s in range(c["requests"]):
            K = int(round(math.exp(rng.uniform(math.log(4.0), math.log(c["Kmax"])))))
            nodes = K ** 3 * (rng.randint(2, 5) + 1) ** 3
            fl = _FLOPS["tgv_ns"] if s % 4 == 3 else _FLOPS["wave"]
            wb, wf = _stage_work(nodes, 5, False, fl, 5 * c["steps"])
            b, f = b + wb, f + wf
        return {"bytes": b, "flops": f}
    nv = 9 if c["flow"] == "ot" else 5
    key = c["flow"] + ({"tgv": "_ns", "ot": "_res"}.get(c["flow"], "") if c["parabolic"] else "")
    nodes, fl = _nodes(c), _FLOPS[key]
    if c["kind"] in ("rhs", "dropin"):  # U, metrics, sJ in, Ut out
        return {"bytes": nodes * 8 * (2 * nv + 10), "flops": nodes * fl}
    b, f = _stage_work(nodes, nv, c["fp32"], fl, 5 * c["steps"])
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------------------
# The same numbers in plain torch, 64 bits: split-form DGSEM on the box mesh's metrics.  Arrays are
# (variable, k, j, i, element) with the elements of the box numbered x fastest.

_DEV = "cuda" if torch.cuda.is_available() else "cpu"
_AXIS = (2, 1, 0)  # node axis of xi, eta, zeta


def _lgl(N):
    P = np.polynomial.legendre.Legendre.basis(N)
    x = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
    for _ in range(3):  # Newton on P_N' at the inner nodes
        x[1:-1] -= P.deriv()(x[1:-1]) / P.deriv(2)(x[1:-1])
    w = 2.0 / (N * (N + 1) * P(x) ** 2)
    b = np.array([1.0 / np.prod([x[i] - x[j] for j in range(N + 1) if j != i]) for i in range(N + 1)])
    D = np.zeros((N + 1, N + 1))
    for i in range(N + 1):
        for j in range(N + 1):
            if i != j:
                D[i, j] = b[j] / b[i] / (x[i] - x[j])
        D[i, i] = -D[i].sum()
    return x, w, D


def _ln_mean(a, b):
    xi = b / a
    u = (xi * (xi - 2.0) + 1.0) / (xi * (xi + 2.0) + 1.0)
    series = (a + b) * 52.5 / (105.0 + u * (35.0 + u * (21.0 + u * 15.0)))
    return torch.where(u < 1e-4, series, (b - a) / torch.log(xi))


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


class _Solver:
    """Right-hand side, time step and LSERK loop of one case."""

    KAPPA = 1.4
    NV = 5

    def __init__(self, c, mesh):
        self.c, self.N, self.n = c, c["N"], c["N"] + 1
        self.K = (c["Kz"], c["Ky"], c["Kx"])
        E, n = mesh["nElems"], self.n
        x, self.w, self.D = _lgl(self.N)
        self.x = x
        self.L0 = 1.0 / self.w[0]
        self.M = [torch.from_numpy(mesh[k]).to(_DEV).permute(4, 1, 2, 3, 0).contiguous() for k in ("Mf", "Mg", "Mh")]
        self.sJ = torch.from_numpy(mesh["sJ"]).to(_DEV).permute(1, 2, 3, 0).contiguous()
        Dh = -(self.D.T * self.w[None, :]) / self.w[:, None]
        self.Dt = torch.tensor(self.D, device=_DEV)
        self.Dht = torch.tensor(Dh, device=_DEV)
        self.ch = 0.0
        assert self.sJ.shape == (n, n, n, E)

    def load(self, U):
        return torch.from_numpy(U).to(_DEV).permute(4, 1, 2, 3, 0).contiguous()

    def save(self, U):
        return U.permute(4, 1, 2, 3, 0).contiguous().cpu().numpy()

    def right(self, f, d):
        """Face values (..., element) of each element's neighbour in +d."""
        return f.reshape(f.shape[:-1] + self.K).roll(-1, dims=f.dim() + 1 - d).reshape(f.shape)

    def left(self, f, d):
        return f.reshape(f.shape[:-1] + self.K).roll(1, dims=f.dim() + 1 - d).reshape(f.shape)

    def deriv(self, op, f, d):
        """sum_l op(i, l) f(l) along direction d; f (v, k, j, i, E)."""
        y = torch.tensordot(op, f, dims=([1], [1 + _AXIS[d]]))
        return y.movedim(0, 1 + _AXIS[d])

    # -- physics of the Euler / Navier-Stokes equations
    def aux(self, U):
        r, km1 = U[0], self.KAPPA - 1.0
        v = [U[1] / r, U[2] / r, U[3] / r]
        return dict(r=r, v=v, p=km1 * (U[4] - 0.5 * r * _dot(v, v)))

    def pick(self, a, axis, i):
        return {k: ([q.select(axis, i) for q in x] if isinstance(x, list) else x.select(axis, i))
                for k, x in a.items()}

    def two_point(self, a, b, m):
        r = _ln_mean(a["r"], b["r"])
        vm = [0.5 * (x + y) for x, y in zip(a["v"], b["v"])]
        pa = 0.5 * (a["p"] + b["p"])
        qa, qb = _dot(a["v"], m), _dot(b["v"], m)
        f0 = r * 0.5 * (qa + qb)
        rp = _ln_mean(a["r"] / a["p"], b["r"] / b["p"])
        F = [f0] + [f0 * vm[i] + m[i] * pa for i in range(3)]
        F.append(f0 * (0.5 * _dot(a["v"], b["v"]) + 1.0 / (rp * (self.KAPPA - 1.0))) + 0.5 * (a["p"] * qb + b["p"] * qa))
        return F

    def volume(self, U):
        a = self.aux(U)
        out = torch.zeros_like(U)
        for d in range(3):
            ax = _AXIS[d]
            nodes = [self.pick(a, ax, i) for i in range(self.n)]
            met = [[self.M[d][c].select(ax, i) for c in range(3)] for i in range(self.n)]
            for i in range(self.n):
                for l in range(i + 1, self.n):
                    m = [0.5 * (met[i][c] + met[l][c]) for c in range(3)]
                    for v, f in enumerate(self.two_point(nodes[i], nodes[l], m)):
                        out[v].select(ax, i).add_(f, alpha=2.0 * self.D[i, l])
                        out[v].select(ax, l).add_(f, alpha=2.0 * self.D[l, i])
        return out

    def flux_n(self, U, a, nv):
        q = _dot(a["v"], nv)
        return [U[0] * q] + [U[1 + i] * q + a["p"] * nv[i] for i in range(3)] + [(U[4] + a["p"]) * q]

    def wave_speed(self, UL, UR, aL, aR, nv):
        c2 = torch.maximum(self.KAPPA * aL["p"] / aL["r"], self.KAPPA * aR["p"] / aR["r"])
        return torch.maximum(_dot(aL["v"], nv).abs(), _dot(aR["v"], nv).abs()) + torch.sqrt(c2)

    def riemann(self, UL, UR, nv):
        """Local Lax-Friedrichs flux in the direction of the unit normal nv."""
        aL, aR = self.aux(UL), self.aux(UR)
        lam = self.wave_speed(UL, UR, aL, aR, nv)
        fl, fr = self.flux_n(UL, aL, nv), self.flux_n(UR, aR, nv)
        return torch.stack([0.5 * (fl[v] + fr[v] - lam * (UR[v] - UL[v])) for v in range(self.NV)])

    def powell(self, UL, UR, nv):
        return None

    def entropy_vars(self, U):
        a, km1 = self.aux(U), self.KAPPA - 1.0
        rp = a["r"] / a["p"]
        s = torch.log(a["p"]) - self.KAPPA * torch.log(a["r"])
        return torch.stack([(self.KAPPA - s) / km1 - 0.5 * rp * _dot(a["v"], a["v"])] +
                           [rp * q for q in a["v"]] + [-rp])

    def grad_prim(self, U, g):
        a, skm1 = self.aux(U), 1.0 / (self.KAPPA - 1.0)
        t = a["p"] / a["r"]
        ek = 0.5 * a["r"] * _dot(a["v"], a["v"])
        gv = [t * (g[1 + i] + a["v"][i] * g[4]) for i in range(3)]
        g0 = a["r"] * g[0] - g[4] * (ek - a["p"] * skm1) + a["r"] / a["p"] * a["r"] * _dot(a["v"], gv)
        return [g0] + gv + [t * (g0 + a["p"] * g[4])]

    def diff_flux(self, U, g):
        """Viscous fluxes (three Cartesian directions) from primitive gradients g[d][v]."""
        a, mu, skm1 = self.aux(U), MU0, 1.0 / (self.KAPPA - 1.0)
        lam = mu * self.KAPPA / 0.72
        div = g[0][1] + g[1][2] + g[2][3]
        out = []
        for d in range(3):
            f = [torch.zeros_like(U[0])]
            f += [-mu * (g[d][1 + i] + g[i][1 + d] - ((2.0 / 3.0) * div if i == d else 0.0)) for i in range(3)]
            dT = skm1 / a["r"] * (g[d][4] - a["p"] / a["r"] * g[d][0])
            f.append(_dot(a["v"], f[1:4]) - lam * dT)
            out.append(torch.stack(f))
        return out

    # -- lifting: gradients in the volume and on the two faces of every direction
    def gradients(self, U):
        w = self.entropy_vars(U)
        g = [torch.zeros_like(w) for _ in range(3)]
        for d in range(3):
            dw = self.deriv(self.Dt, w, d)
            for c in range(3):
                g[c] += self.M[d][c] * dw
        g = [q * self.sJ for q in g]
        faces = []  # per direction: primitive gradients at the upper and at the lower face
        lift = []
        for d in range(3):
            ax = _AXIS[d]
            hi, lo = w.select(1 + ax, self.N), w.select(1 + ax, 0)
            jump = 0.5 * (self.right(lo, d) - hi) * self.L0  # slave minus master
            m = [self.M[d][c].select(ax, self.N) for c in range(3)]
            ml = [self.left(q, d) for q in m]
            jl = self.left(jump, d)
            up = [jump * m[c] * self.sJ.select(ax, self.N) for c in range(3)]
            dn = [jl * ml[c] * self.sJ.select(ax, 0) for c in range(3)]
            lift.append((up, dn))
        if self.c["lifting"] == 2:
            faces = [([g[c].select(1 + _AXIS[d], self.N) + 2.0 * lift[d][0][c] for c in range(3)],
                      [g[c].select(1 + _AXIS[d], 0) + 2.0 * lift[d][1][c] for c in range(3)]) for d in range(3)]
        for d in range(3):
            for c in range(3):
                g[c].select(1 + _AXIS[d], self.N).add_(lift[d][0][c])
                g[c].select(1 + _AXIS[d], 0).add_(lift[d][1][c])
        if self.c["lifting"] == 1:
            faces = [([g[c].select(1 + _AXIS[d], self.N) for c in range(3)],
                      [g[c].select(1 + _AXIS[d], 0) for c in range(3)]) for d in range(3)]
        return g, faces

    # -- sub-cell shock capturing
    def blending(self, U):
        a, n, N = self.aux(U), self.n, self.N
        V = np.stack([np.polynomial.legendre.Legendre.basis(j)(self.x) * math.sqrt(j + 0.5) for j in range(n)], 1)
        op = torch.tensor(np.linalg.inv(V), device=_DEV)
        m = (a["r"] * a["p"])[None]
        for d in range(3):
            m = self.deriv(op, m, d)
        m = m[0] ** 2
        s0, s1, s2 = (m[:k, :k, :k].sum(dim=(0, 1, 2)) for k in (n, n - 1, n - 2))
        eta = torch.clamp(torch.maximum((s0 - s1) / s0, (s1 - s2) / s1), min=float(np.finfo(float).eps))
        T = 0.5 * 10.0 ** (-1.8 * (N + 1.0) ** 0.25)
        al = 1.0 / (1.0 + torch.exp(-math.log((1.0 - 1e-4) / 1e-4) * (eta - T) / T))
        al = torch.where(al < 0.01, torch.zeros_like(al), torch.clamp(al, max=0.5))
        top = al
        for d in range(3):
            top = torch.maximum(top, torch.maximum(0.5 * self.right(al, d), 0.5 * self.left(al, d)))
        return top

    def subcell(self, U):
        """Volume part of the first-order finite-volume scheme on the sub-cells."""
        out = torch.zeros_like(U)
        for d in range(3):
            ax = _AXIS[d]
            line = [U.select(1 + ax, i) for i in range(self.n)]
            met = self.M[d].movedim(1 + ax, 0)  # (line, component, ...)
            nv = met[0].clone()
            for f in range(self.N):
                for q in range(self.n):
                    nv = nv + self.w[f] * self.D[f, q] * met[q]
                size = torch.sqrt(_dot(nv, nv))
                F = self.riemann(line[f], line[f + 1], nv / size) * size
                out.select(1 + ax, f).add_(F, alpha=1.0 / self.w[f])
                out.select(1 + ax, f + 1).add_(F, alpha=-1.0 / self.w[f + 1])
        return out

    # -- the operator
    def rhs(self, U):
        c = self.c
        out = self.volume(U)
        if c["flow"] == "sedov":
            al = self.blending(U)
            out = (1.0 - al) * out + al * self.subcell(U)
        faces = None
        if c["parabolic"]:
            g, faces = self.gradients(U)
            F = self.diff_flux(U, [self.grad_prim(U, q) for q in g])
            for d in range(3):
                t = sum(F[k] * self.M[d][k] for k in range(3))
                out += self.deriv(self.Dht, t, d)
        for d in range(3):
            ax = _AXIS[d]
            UL, UR = U.select(1 + ax, self.N), self.right(U.select(1 + ax, 0), d)
            m = torch.stack([self.M[d][k].select(ax, self.N) for k in range(3)])
            size = torch.sqrt(_dot(m, m))
            nv = m / size
            F = self.riemann(UL, UR, nv)
            if c["parabolic"]:
                hi, lo = faces[d][0], [self.right(q, d) for q in faces[d][1]]
                fh = self.diff_flux(UL, [self.grad_prim(UL, q) for q in hi])
                fl = self.diff_flux(UR, [self.grad_prim(UR, q) for q in lo])
                F = F + 0.5 * sum(nv[k] * (fh[k] + fl[k]) for k in range(3))
            Fm, Fs = F, F
            pw = self.powell(UL, UR, nv)
            if pw is not None:
                Fm, Fs = F + pw[0], F + pw[1]
            out.select(1 + ax, self.N).add_(Fm * size, alpha=self.L0)
            out.select(1 + ax, 0).sub_(self.left(Fs * size, d), alpha=self.L0)
        return -self.sJ * out

    def speeds(self, U):
        """Per direction the largest |contravariant velocity| + sound speed per node."""
        a = self.aux(U)
        cs = torch.sqrt(self.KAPPA * a["p"] / a["r"])
        return [self.sJ * (_dot(a["v"], m).abs() + cs * torch.sqrt(_dot(m, m))) for m in self.M]

    def diffusivity(self, U):
        mu = max(4.0 / 3.0, self.KAPPA / 0.72) * MU0
        return [mu / U[0] * _dot(m, m) * self.sJ ** 2 for m in self.M]

    def visc_limit(self, U):
        return sum(q.amax(dim=(0, 1, 2)) for q in self.diffusivity(U))

    def time_step(self, U, scale):
        N = self.N
        cfl = scale * {2: 3.4144, 3: 2.8451, 4: 2.4739, 5: 2.2027}[N] / (2.0 * N + 1.0)
        dfl = scale * 1.853 * {2: 1.95, 3: 1.18, 4: 0.79, 5: 0.56}[N] / (2.0 * N + 1.0) ** 2
        dt = float((2.0 * cfl / sum(q.amax(dim=(0, 1, 2)) for q in self.speeds(U))).min())
        if self.NV == 9:
            unit = [self.sJ * torch.sqrt(_dot(m, m)) for m in self.M]
            self.dtch1 = float((2.0 * cfl / sum(q.amax(dim=(0, 1, 2)) for q in unit)).min())
        if self.c["parabolic"]:
            dt = min(dt, float((4.0 * dfl / self.visc_limit(U)).min()))
        if self.NV == 9:
            self.ch = 0.5 * self.dtch1 / dt
        return dt

    RKA = (0.0, 567301805773.0 / 1357537059087.0, 2404267990393.0 / 2016746695238.0,
           3550918686646.0 / 2091501179385.0, 1275806237668.0 / 842570457699.0)
    RKB = (1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0,
           1720146321549.0 / 2090206949498.0, 3134564353537.0 / 4481467310338.0,
           2277821191437.0 / 14882151754819.0)

    def run(self, U, steps, scale):
        t = dt = 0.0
        for _ in range(steps):
            dt = self.time_step(U, scale)
            k = torch.zeros_like(U)
            for A, B in zip(self.RKA, self.RKB):
                k = self.rhs(U) - A * k
                U = U + (B * dt) * k
            t += dt
        return U, t, dt


class _MhdSolver(_Solver):
    """Resistive or ideal GLM-MHD (mu_0 = 1): Derigs flux, Powell terms, Rusanov."""

    KAPPA = 5.0 / 3.0
    NV = 9

    def aux(self, U):
        r, v, B = U[0], [U[1 + i] / U[0] for i in range(3)], [U[5], U[6], U[7]]
        b2, v2 = _dot(B, B), _dot(v, v)
        p = (self.KAPPA - 1.0) * (U[4] - 0.5 * r * v2 - 0.5 * b2 - 0.5 * U[8] ** 2)
        return dict(r=r, v=v, B=B, psi=U[8], p=p, beta=0.5 * r / p, v2=v2, b2=b2, vB=_dot(v, B))

    def two_point(self, a, b, m):
        ch, mean = self.ch, lambda k: 0.5 * (a[k] + b[k])
        v = [0.5 * (x + y) for x, y in zip(a["v"], b["v"])]
        B = [0.5 * (x + y) for x, y in zip(a["B"], b["B"])]
        pt = 0.5 * ((a["r"] + b["r"]) / (a["beta"] + b["beta"]) + mean("b2"))
        vm, Bm, psi = _dot(v, m), _dot(B, m), mean("psi")
        f0 = _ln_mean(a["r"], b["r"]) * vm
        fm = [f0 * v[i] - Bm * B[i] + pt * m[i] for i in range(3)]
        fB = [vm * B[i] - Bm * v[i] + ch * psi * m[i] for i in range(3)]
        f8 = ch * Bm
        fE = (f0 * 0.5 * (1.0 / ((self.KAPPA - 1.0) * _ln_mean(a["beta"], b["beta"])) - mean("v2")) + _dot(v, fm) +
              _dot(B, fB) - 0.25 * (a["b2"] * _dot(a["v"], m) + b["b2"] * _dot(b["v"], m)) + mean("vB") * Bm +
              f8 * psi - 0.5 * ch * (a["psi"] * _dot(a["B"], m) + b["psi"] * _dot(b["B"], m)))
        return [f0] + fm + [fE] + fB + [f8]

    def volume(self, U):
        out = super().volume(U)
        a = self.aux(U)
        phi = [0.5 * q for q in a["B"]] + [0.5 * a["vB"]] + [0.5 * q for q in a["v"]]
        for d in range(3):  # Powell terms: sum_l Ds(i, l) phi_i (m_i.B_i + {{m}}.B_l)
            ax = _AXIS[d]
            m = [[self.M[d][c].select(ax, i) for c in range(3)] for i in range(self.n)]
            B = [[q.select(ax, i) for q in a["B"]] for i in range(self.n)]
            for i in range(self.n):
                s = 0.0
                for l in range(self.n):
                    ds = 2.0 * self.D[i, l]
                    if i == l:  # the split form's diagonal: boundary terms cancel D(i, i)
                        ds += {0: 1.0 / self.w[0], self.N: -1.0 / self.w[0]}.get(i, 0.0)
                    s = s + ds * (_dot(m[i], B[i]) + 0.5 * (_dot(m[i], B[l]) + _dot(m[l], B[l])))
                for v, q in enumerate(phi):
                    out[1 + v].select(ax, i).add_(q.select(ax, i) * s)
        return out

    def flux_n(self, U, a, nv):
        q, bn, ch = _dot(a["v"], nv), _dot(a["B"], nv), self.ch
        pt = a["p"] + 0.5 * a["b2"]
        F = [U[0] * q] + [U[1 + i] * q + pt * nv[i] - bn * a["B"][i] for i in range(3)]
        F.append((U[4] - 0.5 * a["psi"] ** 2 + pt) * q - bn * a["vB"] + ch * bn * a["psi"])
        return F + [q * a["B"][i] - bn * a["v"][i] + ch * a["psi"] * nv[i] for i in range(3)] + [ch * bn]

    def fast_speed(self, a, nv):
        # the wave speed's pressure counts psi among the magnetic components, as does p here
        c2, va2 = self.KAPPA * a["p"] / a["r"], a["b2"] / a["r"]
        ca2 = _dot(a["B"], nv) ** 2 / a["r"]
        return torch.sqrt(0.5 * (c2 + va2 + torch.sqrt((c2 + va2) ** 2 - 4.0 * c2 * ca2)))

    def wave_speed(self, UL, UR, aL, aR, nv):
        return torch.maximum(_dot(aL["v"], nv).abs() + self.fast_speed(aL, nv),
                             _dot(aR["v"], nv).abs() + self.fast_speed(aR, nv))

    def powell(self, UL, UR, nv):
        bn = 0.5 * (_dot(UL[5:8], nv) + _dot(UR[5:8], nv))
        out = []
        for U in (UL, UR):
            a = self.aux(U)
            z = torch.zeros_like(bn)
            out.append(torch.stack([z] + [bn * q for q in a["B"]] + [bn * a["vB"]] + [bn * q for q in a["v"]] + [z]))
        return out

    def entropy_vars(self, U):
        a, km1 = self.aux(U), self.KAPPA - 1.0
        rp = a["r"] / a["p"]
        s = torch.log(a["p"]) - self.KAPPA * torch.log(a["r"])
        return torch.stack([(self.KAPPA - s) / km1 - 0.5 * rp * a["v2"]] + [rp * q for q in a["v"]] + [-rp] +
                           [rp * q for q in a["B"]] + [rp * a["psi"]])

    def grad_prim(self, U, g):
        t = self.aux(U)
        t = t["p"] / t["r"]
        return super().grad_prim(U, g) + [t * (g[i] + U[i] * g[4]) for i in range(5, 9)]

    def diff_flux(self, U, g):
        """Resistive fluxes, viscosity zero."""
        a, eta = self.aux(U), _MHD_RES["eta"]
        z = torch.zeros_like(U[0])
        out = []
        for d in range(3):
            fB = [-eta * (g[d][5 + i] - g[i][5 + d]) if i != d else z for i in range(3)]
            out.append(torch.stack([z, z, z, z, _dot(a["B"], fB)] + fB + [z]))
        return out

    def speeds(self, U):
        a = self.aux(U)
        cf = torch.sqrt((self.KAPPA * a["p"] + a["b2"]) / a["r"])
        return [self.sJ * (_dot(a["v"], m).abs() + cf * torch.sqrt(_dot(m, m))) for m in self.M]

    def visc_limit(self, U):
        s = sum(_dot(m, m) for m in self.M) * self.sJ ** 2
        return _MHD_RES["eta"] * s.amax(dim=(0, 1, 2))


def exact(case, seed):
    c = case
    if c["kind"] == "serve":  # many small solves one after the other: more than twenty seconds
        return None
    mesh = _mesh(c)
    s = (_MhdSolver if c["flow"] == "ot" else _Solver)(c, mesh)
    U = s.load(_state(c, mesh, seed))
    if c["kind"] in ("rhs", "dropin"):
        return s.save(s.rhs(U))
    U, t, dt = s.run(U, c["steps"], c["cfl"])
    return {"U": s.save(U), "t": t, "dt": dt, "err": 0}
