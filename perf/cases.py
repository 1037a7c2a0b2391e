"""The work whose speed is followed: what a user of this framework has it do, through its public entry
points, over the range of sizes, orders and options that the dynamical core is run with.

listed() names twelve cases, draw() gives further ones of the same kinds and ranges, prepare() makes what a
program holds before the call (mesh context, stepper, device fields), run() is one pass, work() the bytes and
operations a pass cannot do without, exact() the outputs in plain 64-bit torch where that is short.
"""
import ctypes as C
import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "fe-project_amd"))

import fedg  # noqa: E402
from fedg import cases as setups  # noqa: E402
from fedg.tracer import TracerAdvection  # noqa: E402

GRAV, RDRY, CPDRY, CVDRY, P00 = 9.80665, 287.04, 1004.64, 1004.64 - 287.04, 1.0e5
BVF, THETA0 = 0.01, 300.0
# three water species (vapour, liquid, ice): TRACER_MASS, _R, _CV, _CP and internal-energy offset
WATER = (np.array([1.0, 1.0, 1.0]), np.array([461.5, 0.0, 0.0]), np.array([1390.0, 4218.0, 2106.0]),
         np.array([1851.5, 4218.0, 2106.0]), np.array([2.5e6, 0.0, -3.3e5]))
DIAGNOSTICS = ("T", "PT", "U", "W", "QDRY", "ENGT")
MLP_DIMS = (641, 256, 256, 256, 320)  # the learned guess of a line of 8 elements at p = 7


def listed():
    return [
        # one step of the small warm bubble with the modal filter (the reference's test case): launches and latency
        dict(name="heve_p3_small", kind="heve", p=3, nx=8, ny=8, nz=4, terrain=False, bits=64, filter=True),
        # the flagship: one classic RK4 step of the 160 km box
        dict(name="heve_p7_large", kind="heve", p=7, nx=64, ny=64, nz=16, terrain=False, bits=64, filter=False),
        # the step with the tendency in the FP32 perturbation form
        dict(name="heve_p7_fp32", kind="heve", p=7, nx=32, ny=32, nz=16, terrain=False, bits=32, filter=False),
        # the step over a ridge: every metric array of the terrain-following coordinate is read
        dict(name="heve_p7_terrain", kind="heve", p=7, nx=27, ny=19, nz=11, terrain=True, bits=64, filter=False),
        # another polynomial order on a ragged box
        dict(name="heve_p5_ragged", kind="heve", p=5, nx=41, ny=37, nz=13, terrain=False, bits=64, filter=False),
        # a quarter of the inertia-gravity-wave channel: twenty HEVI steps, then the state to the host for output
        dict(name="hevi_p7_channel", kind="hevi", p=7, nx=60, ny=16, nz=8, steps=20, rtol=0.0),
        # a small HEVI run with Newton to a tolerance: many small launches and residual norms
        dict(name="hevi_p3_newton", kind="hevi", p=3, nx=12, ny=6, nz=6, steps=5, rtol=1e-10),
        # the implicit stage of a host that drives its own loop, on the whole channel
        dict(name="implicit_p7_channel", kind="implicit", p=7, nx=240, ny=16, nz=8),
        # such a host's right-hand side: halo exchange, pressure, boundary values, tendency (explicit HEVE)
        dict(name="tendency_p7", kind="tendency", p=7, nx=40, ny=32, nz=16),
        # one SSP RK3 step of a tracer with the limiter and the mass fixer
        dict(name="tracer_p7", kind="tracer", p=7, nx=48, ny=48, nz=16),
        # moist air after the tracer step: specific heats, negative fixer, pressure, history diagnostics
        dict(name="moist_p7", kind="moist", p=7, nx=32, ny=32, nz=16),
        # sixteen minibatches of the learned-guess network (backward and Adam), then its weights
        dict(name="guess_training", kind="mlp", batch=512, steps=16),
    ]


def draw(rng):
    kind = rng.choice(["heve", "heve", "heve", "hevi", "implicit", "tendency", "tracer", "moist", "mlp"])
    if kind == "mlp":
        return dict(kind=kind, batch=int(round(math.exp(rng.uniform(math.log(100), math.log(2048))))),
                    steps=rng.randint(4, 16))
    p = rng.choice([2, 3, 3, 4, 5, 6, 7, 7, 7, 7])
    lo, hi = {"heve": (2.0e4, 1.0e7), "hevi": (2.0e4, 3.0e6), "implicit": (1.0e5, 1.2e7)}.get(kind, (5.0e4, 1.0e7))
    ne = math.exp(rng.uniform(math.log(lo), math.log(hi))) / (p + 1) ** 3
    nz = rng.randint(3, 12 if kind in ("hevi", "implicit") else 16)
    side = math.sqrt(max(ne / nz, 9.0))
    nx = max(3, int(round(side * math.exp(rng.uniform(-0.5, 0.9)))))
    ny = max(2, int(round(side * side / nx)))
    c = dict(kind=kind, p=p, nx=nx, ny=ny, nz=nz)
    if kind == "heve":
        c["terrain"] = rng.random() < 0.3
        c["bits"] = 32 if not c["terrain"] and rng.random() < 0.25 else 64
        c["filter"] = p <= 4
    if kind == "hevi":
        c["steps"] = rng.randint(4, 16)
        c["rtol"] = rng.choice([0.0, 0.0, 1e-10])
    return c


# ---------------------------------------------------------------------------------------------------------
# Meshes, base states and smooth initial states


def _extent(c):
    """Element sizes (m) and the time step of a case (acoustic limit of the smallest node distance)."""
    if c["kind"] in ("hevi", "implicit"):
        return 1250.0, 1250.0, 1250.0, 0.05 * (7 / c["p"]) ** 2
    if c["kind"] == "heve" and c["filter"]:
        return 2500.0, 2500.0, 2500.0, 0.2 * (3 / c["p"]) ** 2
    return 2500.0, 2500.0, 625.0, 0.024 * (7 / c["p"]) ** 2


def _base_kind(c):
    return "constBVFreq" if c["kind"] in ("hevi", "implicit") or c.get("terrain") else "constT"


@functools.lru_cache(maxsize=2)
def _plan(kind, p, nx, ny, nz, terrain, filt):
    """What is set up once for a mesh, whatever the state: mesh, context, base state, node coordinates."""
    c = dict(kind=kind, p=p, nx=nx, ny=ny, nz=nz, terrain=terrain, filter=filt)
    dx, dy, dz, dt = _extent(c)
    mesh = fedg.BoxMesh(p, nx, ny, nz, (0.0, nx * dx), (0.0, ny * dy), (0.0, nz * dz), periodic=(True, True, False))
    if terrain:
        half = 0.5 * nx * dx
        mesh.set_topography(lambda x, y: 300.0 / (1.0 + ((x - half) / 8.0e3) ** 2), zTop=nz * dz)
    bs = setups.base_state(mesh, _base_kind(c))
    dm = fedg.DeviceMesh(mesh)
    if filt:
        f = fedg.modalfilter_matrix(p, *setups.RISING_BUBBLE_FILTER)
        dm.setup_modalfilter(f, f)
    grad = fedg.calc_phyd_hgrad(dm, bs.PRES_hyd, bs.PRES_hyd_ref)
    n = mesh.Np * mesh.Ne
    xyz = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (mesh.x, mesh.y, mesh.height)]
    hyd = [torch.from_numpy(a[:n]).cuda() for a in (bs.DENS_hyd, bs.PRES_hyd, bs.THERM_hyd)]
    return dict(mesh=mesh, bs=bs, dm=dm, grad=grad, n=n, nA=mesh.Np * mesh.NeA, xyz=xyz, hyd=hyd, dt=dt,
                size=(nx * dx, ny * dy, nz * dz))


def _plan_of(c):
    return _plan(c["kind"], c["p"], c["nx"], c["ny"], c["nz"], bool(c.get("terrain")), bool(c.get("filter")))


def _bell(xyz, size, rng):
    """A smooth bubble of unit height with seeded centre and width."""
    x, y, z = xyz
    xc, yc, zc = (rng.uniform(0.3, 0.7) * s for s in size)
    r = rng.uniform(0.15, 0.25)
    return torch.exp(-(((x - xc) / (r * size[0])) ** 2 + ((y - yc) / (r * size[1])) ** 2 +
                       ((z - zc) / (0.7 * r * size[2])) ** 2))


def _state(c, xyz, size, hyd, seed):
    """DDENS, DRHOT, MOMZ, MOMX, MOMY of warm bubbles in a wind (or of the wave in the channel's wind)."""
    rng = np.random.default_rng(seed)
    Dh, Ph, Th = hyd
    x, y, z = xyz
    theta = Th / Dh
    if c["kind"] in ("hevi", "implicit"):
        xc, a = rng.uniform(0.2, 0.8) * size[0], 5.0e3
        bump = rng.uniform(0.005, 0.05) * torch.sin(math.pi * z / size[2]) / (1.0 + ((x - xc) / a) ** 2)
        u, v, w = rng.uniform(10.0, 30.0), 0.0, torch.zeros_like(z)
        if c["kind"] == "implicit":
            w = rng.uniform(0.5, 1.5) * torch.sin(math.pi * z / size[2]) * _bell(xyz, size, rng)
    else:
        bump = sum(rng.uniform(0.5, 2.0) * _bell(xyz, size, rng) for _ in range(3))
        u, v = rng.uniform(0.0, 8.0), rng.uniform(-4.0, 4.0)
        if c.get("terrain"):
            u = v = 0.0
        w = torch.zeros_like(z)
        if c["kind"] in ("tendency", "moist"):
            w = torch.sin(math.pi * z / size[2]) * _bell(xyz, size, rng)
    dens = Th / (theta + bump)  # the hydrostatic pressure (rhotheta) kept
    return [dens - Dh, torch.zeros_like(z), dens * w, dens * u, dens * v]


def _full(pl, t):
    """A (Np, NeA) device field of a state's (Np, Ne) values."""
    f = torch.zeros(pl["nA"], dtype=torch.float64, device="cuda")
    f[: pl["n"]] = t
    return f


class _Mem:
    """n float64 values of device memory that a framework object owns, for torch.as_tensor: the tensor keeps this
    object, and with it the memory's owner, alive."""

    def __init__(self, ptr, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(ptr, False), version=2)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


# ---------------------------------------------------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        g = torch.Generator(device="cuda").manual_seed(seed)
        net = fedg.Mlp(MLP_DIMS[0], MLP_DIMS[1], 3, MLP_DIMS[-1], seed=1 + seed % 1000)
        rows = case["batch"] * case["steps"]
        X = torch.randn(rows, MLP_DIMS[0], generator=g, device="cuda")
        T = torch.tanh(X[:, : MLP_DIMS[-1]] + 0.5 * X[:, MLP_DIMS[-1]: 2 * MLP_DIMS[-1]])
        torch.cuda.synchronize()
        return dict(case=case, net=net, X=X, T=T)
    pl = _plan_of(case)
    dm, bs, (Dx, Dy), n = pl["dm"], pl["bs"], pl["grad"], pl["n"]
    q = _state(case, pl["xyz"], pl["size"], pl["hyd"], seed)
    s = dict(case=case, plan=pl)
    if kind == "heve":
        st = fedg.HeveStepper(dm, bs, Dx, Dy, pl["dt"])
        st.set_precision(case["bits"])
        st.set_state([a.cpu().numpy() for a in q])
        if case["filter"]:
            st.set_modalfilter(True)
        s["st"] = st
    elif kind == "hevi":
        s["st"] = fedg.HeviStepper(dm, bs, Dx, Dy, pl["dt"], max_it=8 if case["rtol"] else 1, rtol=case["rtol"])
        s["st"].set_state([a.cpu().numpy() for a in q])
    elif kind in ("implicit", "tendency"):
        s["q"] = [_full(pl, a) for a in q]
        s["out"] = [torch.zeros(pl["nA"], dtype=torch.float64, device="cuda") for _ in range(5)]
        for name in ("DENS_hyd", "PRES_hyd", "PRES_hyd_ref", "THERM_hyd", "CORIOLIS", "Rtot", "CVtot", "CPtot"):
            s[name] = torch.from_numpy(getattr(bs, name)).cuda()
        if kind == "implicit":  # the stage state is a stage's increment away from q^n
            s["q0"] = [a.clone() for a in s["q"]]
            rng = np.random.default_rng(seed + 7)
            for a, amp in zip(s["q"], (1.0e-4, 3.0e-2, 5.0e-2, 5.0e-2, 5.0e-2)):
                a[:n] += amp * _bell(pl["xyz"], pl["size"], rng)
        else:
            s["Dx"], s["Dy"] = torch.from_numpy(Dx).cuda(), torch.from_numpy(Dy).cuda()
            s["P"], s["DP"] = torch.zeros_like(s["out"][0]), torch.zeros_like(s["out"][0])
    elif kind == "tracer":
        s["dt"] = 0.5 * pl["dt"] * 10.0
        host = [_full(pl, a).cpu().numpy() for a in q]
        s["st"] = TracerAdvection(dm, host[3], host[4], host[2], host[0], bs.DENS_hyd, pl["mesh"].J, s["dt"])
        s["Q"] = _full(pl, _mixing_ratio(case, pl["xyz"], pl["size"], seed))
    else:  # moist
        s["q"] = q
        s["Q"] = _water(pl["xyz"], pl["size"], seed)
        for name in ("R", "CV", "CP", "P", "DP"):
            s[name] = torch.zeros_like(q[0])
        s["P"].copy_(pl["hyd"][1])
        s["J"] = torch.from_numpy(pl["mesh"].J).cuda()
        s["z"] = torch.from_numpy(np.ascontiguousarray(pl["mesh"].z)).cuda()
        s["out"] = [torch.zeros_like(q[0]) for _ in DIAGNOSTICS]
    torch.cuda.synchronize()
    return s


def _mixing_ratio(c, xyz, size, seed):
    """A tracer bubble on a background, with the sharp edge the limiter is for."""
    rng = np.random.default_rng(seed + 3)
    return 1.0e-3 * torch.clamp(3.0 * _bell(xyz, size, rng) - 1.0, min=0.0) + 1.0e-5


def _water(xyz, size, seed):
    """Vapour, liquid and ice with the small negative values that transport leaves at their edges."""
    rng = np.random.default_rng(seed + 5)
    vapour = 1.4e-2 * torch.exp(-xyz[2] / 2.5e3) * (1.0 + 0.2 * _bell(xyz, size, rng))
    return [vapour] + [a * (_bell(xyz, size, rng) - 0.02) for a in (1.0e-3, 4.0e-4)]


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "heve":
        st = state["st"]
        st.run(1)
        q = (C.c_void_p * 5)()
        fedg.check(fedg.LIB.fedg_heve_state_dev(st.handle, q), "fedg_heve_state_dev")
        return [torch.as_tensor(_Mem(q[v], state["plan"]["n"], st), device="cuda") for v in range(5)]
    if kind == "hevi":
        state["st"].run(c["steps"])
        return state["st"].get_state()
    if kind == "mlp":
        net, X, T, b = state["net"], state["X"], state["T"], c["batch"]
        losses = []
        for k in range(c["steps"]):
            px = C.c_void_p(X.data_ptr() + 4 * X.shape[1] * b * k)
            pt = C.c_void_p(T.data_ptr() + 4 * T.shape[1] * b * k)
            losses.append(net.loss_grad(px, pt, b))
            net.adam_step(1e-3)
        return dict(losses=np.array(losses, dtype=np.float32), params=net.params())
    pl = state["plan"]
    dm = pl["dm"]
    if kind == "tracer":
        state["st"].step(_ptr(state["Q"]), 1)
        return state["Q"][: pl["n"]]
    P = lambda k: _ptr(state[k])  # noqa: E731
    if kind == "implicit":
        q, q0 = [_ptr(a) for a in state["q"]], [_ptr(a) for a in state["q0"]]
        fedg.hevi_cal_vi(dm, [_ptr(a) for a in state["out"]], q[0], q[3], q[4], q[2], q[1], P("DENS_hyd"), P("PRES_hyd"),
                         q0[0], q0[3], q0[4], q0[2], q0[1], P("Rtot"), P("CVtot"), P("CPtot"), 0.4358665215 * pl["dt"],
                         pl["dt"])
        return [a[: pl["n"]] for a in state["out"]]
    if kind == "tendency":
        q = [_ptr(a) for a in state["q"]]
        fedg.halo_exchange(dm, q)
        fedg.calc_pressure(dm, P("P"), P("DP"), q[1], P("PRES_hyd"), P("THERM_hyd"), P("Rtot"), P("CVtot"), P("CPtot"))
        fedg.halo_exchange(dm, [P("DP")])
        fedg.apply_bc(dm, q[0], q[3], q[4], q[2], q[1], P("DENS_hyd"), P("PRES_hyd"))
        fedg.heve_cal_tend(dm, [_ptr(a) for a in state["out"]], q[0], q[3], q[4], q[2], q[1], P("DP"), P("DENS_hyd"),
                           P("PRES_hyd"), P("PRES_hyd_ref"), P("THERM_hyd"), P("CORIOLIS"), P("Rtot"), P("CVtot"),
                           P("CPtot"), P("Dx"), P("Dy"))
        return [a[: pl["n"]] for a in state["out"]]
    q, Q = [_ptr(a) for a in state["q"]], [_ptr(a) for a in state["Q"]]
    Dh, Ph, Th = (_ptr(a) for a in pl["hyd"])
    mass, _, cv, _, e0 = WATER
    fedg.tracer_specific_heat(dm, Q, WATER[:4], P("R"), P("CV"), P("CP"))
    fedg.trc_negative_fixer(dm, Q, q[0], P("P"), P("CV"), P("CP"), P("R"), Dh, Ph, P("J"), P("z"), WATER[:4], QLA=1,
                            QIA=1, DRHOT=q[1])
    fedg.calc_pressure(dm, P("P"), P("DP"), q[1], Ph, Th, P("R"), P("CV"), P("CP"))
    for name, o in zip(DIAGNOSTICS, state["out"]):
        fedg.atmos_calc_diagvar(dm, name, _ptr(o), q[0], q[3], q[4], q[2], P("P"), Dh, Ph, P("R"), P("CV"), P("CP"), Q=Q,
                                mass=mass, cv=cv, engi0=e0, zlev=P("z"), pos_z=P("z"))
    return dict(Q=state["Q"], DDENS=state["q"][0], DRHOT=state["q"][1], PRES=state["P"], DPRES=state["DP"],
                R=state["R"], CV=state["CV"], CP=state["CP"], diag=state["out"])


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        pairs = list(zip(MLP_DIMS[:-1], MLP_DIMS[1:]))
        weights = sum(a * b + b for a, b in pairs)
        gemm = 6 * sum(a * b for a, b in pairs) - 2 * pairs[0][0] * pairs[0][1]  # no gradient of the input
        return dict(bytes=float(case["steps"] * 4 * (6 * weights + case["batch"] * (MLP_DIMS[0] + MLP_DIMS[-1]))),
                    flops=float(case["steps"] * case["batch"] * gemm))
    n1 = case["p"] + 1
    nodes = float(case["nx"] * case["ny"] * case["nz"] * n1 ** 3)
    lines = float(case["nx"] * case["ny"] * n1 * n1)
    tend = 32 * n1 + 250  # 15 line contractions, the filter, fluxes, faces and the pressure's power
    n3 = 3 * n1
    # block LU of a line: elimination of every block, four right-hand sides, the residuals
    implicit = lines * case["nz"] * (2 * n3 ** 3 / 3 + 8 * n3 * n3 + 2 * n1 ** 3 / 3) + nodes * 300
    if kind == "heve":  # state in and out, three base fields and their gradient (metrics over terrain); four stages
        return dict(bytes=8 * nodes * (15 + (6 if case["terrain"] else 0)), flops=4 * nodes * tend)
    if kind == "hevi":  # per step; three implicit stages of four
        return dict(bytes=case["steps"] * 8 * nodes * 15 + 8 * nodes * 5, flops=case["steps"] * (3 * implicit + 4 * nodes * tend))
    if kind == "implicit":  # stage state, q^n, base state and heat capacities in, five tendencies out
        return dict(bytes=8 * nodes * 20, flops=implicit)
    if kind == "tendency":  # state, base state and heat capacities in; pressure and five tendencies out
        return dict(bytes=8 * nodes * (5 + 8 + 7), flops=nodes * tend)
    if kind == "tracer":  # tracer in and out, mass fluxes, density, source and J
        return dict(bytes=8 * nodes * 9, flops=3 * nodes * (6 * n1 + 60))
    return dict(bytes=8 * nodes * (3 + 5 + 5 + 3 + 3 + 8 + len(DIAGNOSTICS)), flops=nodes * 600)


# ---------------------------------------------------------------------------------------------------------
# The same outputs in plain 64-bit torch (flat box): fields are (nz, ny, nx, k, j, i)


def _legendre(p, x):
    L = [np.ones_like(x), x]
    for k in range(1, p):
        L.append(((2 * k + 1) * x * L[k] - k * L[k - 1]) / (k + 1))
    return L[: p + 1]


class _Element:
    """1-D LGL operators of order p: nodes, weights, derivative, inverse mass, order p - 1 projection."""

    def __init__(self, p):
        c = np.zeros(p + 1)
        c[p] = 1.0
        inner = np.polynomial.legendre.legroots(np.polynomial.legendre.legder(c)) if p > 1 else []
        x = np.concatenate([[-1.0], np.sort(np.real(inner)), [1.0]])
        for _ in range(3):  # Newton on (1 - x^2) L_p'
            L = _legendre(p, x)
            x[1:-1] -= ((x * L[p] - L[p - 1]) / ((p + 1) * L[p]))[1:-1]
        L = _legendre(p, x)
        self.x, self.w = x, 2.0 / (p * (p + 1) * L[p] ** 2)
        V = np.stack([L[m] * math.sqrt(m + 0.5) for m in range(p + 1)], axis=1)
        dV = np.stack([np.polynomial.legendre.legval(x, np.polynomial.legendre.legder(np.eye(p + 1)[m])) *
                       math.sqrt(m + 0.5) for m in range(p + 1)], axis=1)
        Vi = np.linalg.inv(V)
        keep = np.ones(p + 1)
        keep[p] = 0.0
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        self.D, self.invM, self.low = t(dV @ Vi), t(V @ V.T), t((V * keep) @ Vi)
        eta = np.arange(p + 1) / p
        etac, alpha, order = setups.RISING_BUBBLE_FILTER
        sig = np.where(eta > etac, np.exp(-alpha * ((eta - etac) / (1 - etac)) ** order), 1.0)
        self.filt = t((V * sig) @ Vi)


def _along(f, M, axis):
    """M applied along the node axis (0: x, 1: y, 2: z) of f."""
    return torch.movedim(torch.movedim(f, -1 - axis, -1) @ M.T, -1, -1 - axis)


class _Box:
    def __init__(self, c):
        self.p, self.shape = c["p"], (c["nz"], c["ny"], c["nx"])
        self.e = _Element(c["p"])
        h = _extent(c)
        self.h, self.dt = h[:3], h[3]
        n = c["p"] + 1
        self.size = tuple(m * d for m, d in zip((c["nx"], c["ny"], c["nz"]), self.h))
        ref = torch.from_numpy((self.e.x + 1.0) / 2.0).cuda()
        co = [((torch.arange(m, device="cuda")[:, None] + ref[None, :]) * d) for m, d in
              zip((c["nx"], c["ny"], c["nz"]), self.h)]
        full = self.shape + (n, n, n)
        self.xyz = [co[0][None, None, :, None, None, :].expand(full), co[1][None, :, None, None, :, None].expand(full),
                    co[2][:, None, None, :, None, None].expand(full)]
        z = self.xyz[2]
        if _base_kind(c) == "constT":
            H = RDRY * 300.0 / GRAV
            P = P00 * torch.exp(-z / H)
            D = P / (RDRY * 300.0)
        else:
            PT = THETA0 * torch.exp(BVF ** 2 / GRAV * z)
            ex = 1.0 + GRAV ** 2 / (CPDRY * BVF ** 2) * (1.0 / PT - 1.0 / THETA0)
            P = P00 * ex ** (CPDRY / RDRY)
            D = P / (RDRY * ex * PT)
        self.hyd = [D, P, P00 / RDRY * (P / P00) ** (CVDRY / CPDRY)]

    def sides(self, axis):
        """(face slot, outward sign, M and P selectors) of the two faces across an axis; closed in z."""
        dim = 2 - axis
        def pick(f, end):
            return f.select(3 + dim, -1 if end else 0)
        for end in (0, 1):
            def M(f, end=end):
                return pick(f, end)
            def P(f, end=end):
                g = torch.roll(pick(f, 1 - end), -1 if end else 1, dims=dim)
                if axis == 2:
                    g = g.clone()
                    g[-1 if end else 0] = pick(f, end)[-1 if end else 0]
                return g
            yield end, (1.0 if end else -1.0), M, P

    def lift(self, out, jump, axis, end):
        col = self.e.invM[:, -1 if end else 0] * (2.0 / self.h[axis])
        view = [1] * 6
        view[5 - axis] = len(col)
        return out + col.reshape(view) * jump.unsqueeze(5 - axis)


def _exact_tendency(b, q, DP):
    """The explicit tendency of DDENS, DRHOT, MOMZ, MOMX, MOMY."""
    Dh, Ph, Th = b.hyd
    mom = (q[3], q[4], q[2])
    gam = CPDRY / CVDRY
    dens, rhot = Dh + q[0], Th + q[1]
    carried = [dens, rhot, q[2], q[3], q[4]]
    pressed = {2: 2, 3: 0, 4: 1}  # variable -> the axis its pressure term acts along
    out = [torch.zeros_like(q[0]) for _ in range(5)]
    for axis in range(3):
        vel = mom[axis] / dens
        for v in range(5):
            f = carried[v] * vel if v else mom[axis]
            if pressed.get(v) == axis:
                f = f + DP
            out[v] = out[v] + _along(f, b.e.D, axis) * (2.0 / b.h[axis])
        for end, sgn, M, P in b.sides(axis):
            mM, mP = M(mom[axis]), P(mom[axis])
            own = {2: 2, 0: 3, 1: 4}[axis]
            if axis == 2:
                mP = mP.clone()
                mP[-1 if end else 0] *= -1.0
            dM, dP = M(dens), P(dens)
            uM, uP = sgn * mM / dM, sgn * mP / dP
            a = torch.maximum(torch.sqrt(gam * M(Ph + DP) / dM) + uM.abs(), torch.sqrt(gam * P(Ph + DP) / dP) + uP.abs())
            for v in range(5):
                gM, gP = M(q[v]), (mP if v == own else P(q[v]))
                cM, cP = M(carried[v]), (mP if v == own else P(carried[v]))
                j = cP * uP - cM * uM - a * (gP - gM)
                if pressed.get(v) == axis:
                    j = j + sgn * (P(DP) - M(DP))
                out[v] = b.lift(out[v], 0.5 * j, axis, end)
    out = [-f for f in out]
    out[2] = out[2] - GRAV * _along(q[0], b.e.low, 2)
    return out


def _pressure(b, drhot):
    return P00 * (RDRY / P00 * (b.hyd[2] + drhot)) ** (CPDRY / CVDRY) - b.hyd[1]


def _exact_heve(c, b, q):
    A = (0.5, 0.5, 1.0)
    B = (1 / 6, 1 / 3, 1 / 3, 1 / 6)
    stage, acc = q, [a.clone() for a in q]
    for s in range(4):
        k = _exact_tendency(b, stage, _pressure(b, stage[1]))
        acc = [a + b.dt * B[s] * t for a, t in zip(acc, k)]
        if s < 3:
            stage = [a + b.dt * A[s] * t for a, t in zip(q, k)]
    if c["filter"]:
        for axis in range(3):
            acc = [_along(f, b.e.filt, axis) for f in acc]
    return acc


def _exact_tracer(c, b, q, Q):
    mom, dens = (q[3], q[4], q[2]), b.hyd[0] + q[0]
    dt = 0.5 * b.dt * 10.0
    w = torch.from_numpy(b.e.w).cuda()
    W = w[:, None, None] * w[:, None] * w
    J = b.h[0] * b.h[1] * b.h[2] / 8.0
    W2 = w[:, None] * w
    faces = []
    for axis in range(3):
        for end, sgn, M, P in b.sides(axis):
            mM, mP = sgn * M(mom[axis]), sgn * P(mom[axis])
            al = torch.maximum((mM / M(dens)).abs(), (mP / P(dens)).abs())
            faces.append((axis, end, M, P, mM, mP, al * M(dens), al * P(dens)))

    def numflux(Q):
        return [0.5 * (P(Q) * mP + M(Q) * mM - aP * P(Q) + aM * M(Q)) for _, _, M, P, mM, mP, aM, aP in faces]

    def total(f):
        return (f * W).sum(dim=(3, 4, 5), keepdim=True) * J

    def net(f, axis):
        return (f * W2).sum(dim=(3, 4), keepdim=True) * J * 2.0 / b.h[axis]

    SSP = ((0.0, 1.0, 1.0, 1.0), (0.75, 0.25, 0.25, 0.25), (1 / 3, 2 / 3, 2 / 3, 1.0))  # var0, q, tendency, dt of FCT
    v0 = Q * dens
    for a0, a1, g, gdt in SSP:
        nf = numflux(Q)
        outs = [net(f, face[0]) for f, face in zip(nf, faces)]
        drain = sum(torch.clamp(o, min=0.0) for o in outs).unsqueeze(5)
        R = torch.clamp(total(dens * Q / (dt * gdt)) / (drain + 1e-10), 0.0, 1.0).expand_as(Q)
        T = torch.zeros_like(Q)
        for axis in range(3):
            T = T + _along(mom[axis] * Q, b.e.D, axis) * (2.0 / b.h[axis])
        for f, o, (axis, end, M, P, mM, mP, aM, aP) in zip(nf, outs, faces):
            up = torch.where(o >= 0, M(R), P(R))
            T = b.lift(T, f * up - M(Q) * mM, axis, end)
        Q = (a0 * v0 + a1 * Q * dens - g * dt * T) / dens
    cut = torch.clamp(Q, min=0.0)
    return total(dens * Q) / (total(dens * cut) + 1e-32) * cut


def _exact_moist(b, q, Q):
    w = torch.from_numpy(b.e.w).cuda()
    W = w[:, None, None] * w[:, None] * w
    Dh, Ph, Th = b.hyd
    mass, Rq, CVq, CPq, e0 = WATER

    def heats(Q):
        dry = 1.0 - sum(a * m for a, m in zip(Q, mass))
        return [sum(a * x for a, x in zip(Q, t)) + dry * d for t, d in ((Rq, RDRY), (CVq, CVDRY), (CPq, CPDRY))]

    def total(f):
        return (f * W).sum(dim=(3, 4, 5), keepdim=True)

    R, CV, CP = heats(Q)
    DD0 = q[0]
    dens = Dh + DD0
    IE0 = CV * Ph / R
    T = IE0 / (dens * CV)
    DD, IE, kept = DD0, IE0, []
    for a, cv in zip(Q, CVq):
        m0 = dens * a
        m1 = torch.clamp(m0, min=1e-128)
        m1 = torch.clamp(total(m0), min=0.0) / total(m1) * m1
        DD, IE = DD + (m1 - m0), IE + (m1 - m0) * cv * T
        kept.append(m1)
    dens = Dh + DD
    Q = [m / dens for m in kept]
    IE = total(IE0) / total(IE) * IE
    R, CV, CP = heats(Q)
    IE = IE - (DD - DD0) * GRAV * b.xyz[2]
    P = IE * R / CV
    DT = P00 / R * (P / P00) ** (CV / CP) - P00 / RDRY * (Ph / P00) ** (CVDRY / CPDRY)
    P = P00 * (R / P00 * (Th + DT)) ** (CP / CV)
    dry = 1.0 - sum(a * m for a, m in zip(Q, mass))
    engi = dry * P / R * CVDRY + sum(a * (P / R * cv + dens * e) for a, cv, e in zip(Q, CVq, e0))
    engk = 0.5 * (q[3] ** 2 + q[4] ** 2 + q[2] ** 2) / dens
    temp = P / (R * dens)
    diag = [temp, temp * (P00 / P) ** (R / CP), q[3] / dens, q[2] / dens, dry, engk + engi + dens * GRAV * b.xyz[2]]
    return dict(Q=Q, DDENS=DD, DRHOT=DT, PRES=P, DPRES=P - Ph, R=R, CV=CV, CP=CP, diag=diag)


def exact(case, seed):
    kind = case["kind"]
    # the implicit solves and the network's training have no short plain form (a block-tridiagonal Newton step of
    # every line; BF16 products under Adam); nor has the step over terrain (its metrics come from the mesh builder)
    if kind in ("hevi", "implicit", "mlp") or case.get("terrain"):
        return None
    b = _Box(case)
    q = _state(case, b.xyz, b.size, b.hyd, seed)
    flat = lambda v: (v.contiguous().reshape(-1) if isinstance(v, torch.Tensor) else  # noqa: E731
                      {k: flat(x) for k, x in v.items()} if isinstance(v, dict) else [flat(x) for x in v])
    if kind == "heve":
        return flat(_exact_heve(case, b, q))
    if kind == "tendency":
        t = _exact_tendency(b, q, _pressure(b, q[1]))
        return flat([t[0], t[3], t[4], t[2], t[1]])
    if kind == "tracer":
        return flat(_exact_tracer(case, b, q, _mixing_ratio(case, b.xyz, b.size, seed)))
    return flat(_exact_moist(b, q, _water(b.xyz, b.size, seed)))
