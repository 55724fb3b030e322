"""Performance cases of the fluid step: what programs that use this library
have it do, through its public entry points.

A pass is one unit of such a program's loop:
  monitor   one step, then the body wrench and per-vertex forces of that step
  frame     `steps` steps, then the flow field read back (a saved frame)
  action    a control action (new wave parameters), `steps` steps, then the
            per-step wrench and power of the interval and the body's shape
  coupled   the caller's own solid moves the boundary, one step, and the
            per-vertex forces go back to it
  batch     the action loop over many uneven domains stepped together
  served    one iteration of the rollout server over its active episodes
  dropin    `steps` calls of the fsi_simulator module's step(), then
            get_fluid_moments() (its configuration saves every 100th step)

exact() restates the step in 64 bits with plain torch.
"""
import numpy as np
import torch

import freeflow_amd
from freeflow_amd import capi, serve
from freeflow_amd import workloads as wl

DEV = "cuda" if torch.cuda.is_available() else "cpu"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # drag and lift watched every step of the small vortex street: launches and readback latency
        dict(name="monitor_street_400x200", kind="monitor", dim=2, nx=400, ny=200, nz=1, seg=128, fast=False,
             storage="f32"),
        # the same street, a frame every 100 steps
        dict(name="frame_street_400x200", kind="frame", dim=2, nx=400, ny=200, nz=1, scene="street", seg=128,
             fast=False, storage="f32", steps=100, tune=False),
        # one control action of the 2D swimmer in the reference's operation order
        dict(name="action_swimmer_1200x400", kind="action", dim=2, nx=1200, ny=400, nz=1, seg=600, fast=False,
             storage="f32", steps=10),
        # a swimmer moved by the caller's own solid solver: upload, one step, forces, at an odd size
        dict(name="coupled_swimmer_601x303", kind="coupled", dim=2, nx=601, ny=303, nz=1, seg=400, fast=False,
             storage="f32"),
        # large 2D decaying flow in the fast form, no body
        dict(name="frame_2d_2048x1536_fast", kind="frame", dim=2, nx=2048, ny=1536, nz=1, scene="box", seg=0,
             fast=True, storage="f32", steps=100, tune=True),
        # small odd 3D box: few blocks, latency of one launch per step
        dict(name="frame_3d_61x47x39_fast", kind="frame", dim=3, nx=61, ny=47, nz=39, scene="box", seg=0, fast=True,
             storage="f32", steps=100, tune=False),
        # the headline 3D flow (Taylor-Green + vortex ring), FP32, fast form, tuned as the benchmark does
        dict(name="frame_tg_256x128x128_fast", kind="frame", dim=3, nx=256, ny=128, nz=128, scene="box", seg=0,
             fast=True, storage="f32", steps=500, tune=True),
        # a larger 3D flow held in 16 bits
        dict(name="frame_tg_256x192x160_f16", kind="frame", dim=3, nx=256, ny=192, nz=160, scene="box", seg=0,
             fast=True, storage="f16", steps=500, tune=True),
        # the reference's module: 3D channel with inlet, outlet and walls, default options, a frame every 100 steps
        dict(name="dropin_channel_203x101x97", kind="dropin", dim=3, nx=203, ny=101, nz=97, seg=0, fast=False,
             storage="f32", steps=100),
        # one control action of an oscillating sphere in 3D
        dict(name="action_sphere_160x96x96", kind="action", dim=3, nx=160, ny=96, nz=96, seg=2, fast=True,
             storage="f32", steps=10),
        # 64 uneven swimmers stepped together, one action each
        dict(name="batch_64_swimmers_f16", kind="batch", dim=2, n=64, layout=1234, fast=True, storage="f16", steps=10),
        # the rollout server at work: 2D swimmers and 3D spheres of uneven sizes
        dict(name="served_24_episodes", kind="served", n=24, layout=1234, fast=True, storage="f16", steps=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["monitor", "frame2d", "frame3d", "frame3d", "action2d", "action3d", "coupled", "batch",
                       "served", "dropin"])
    fast = rng.random() < 0.5
    if kind == "monitor":
        return dict(kind="monitor", dim=2, nx=_log_int(rng, 200, 1600), ny=_log_int(rng, 96, 600), nz=1,
                    seg=_log_int(rng, 64, 400), fast=fast, storage="f32")
    if kind == "frame2d":
        scene = rng.choice(["street", "box"])
        return dict(kind="frame", dim=2, nx=_log_int(rng, 200, 2048), ny=_log_int(rng, 96, 1536), nz=1, scene=scene,
                    seg=_log_int(rng, 64, 400) if scene == "street" else 0, fast=fast,
                    storage=rng.choice(["f32", "f32", "f16", "f16u"]) if fast else "f32", steps=100,
                    tune=rng.random() < 0.5)
    if kind == "frame3d":
        fast = rng.random() < 0.75
        return dict(kind="frame", dim=3, nx=_log_int(rng, 32, 256), ny=_log_int(rng, 24, 160),
                    nz=_log_int(rng, 24, 160), scene="box", seg=0, fast=fast,
                    storage=rng.choice(["f32", "f32", "f16", "f16u"]) if fast else "f32",
                    steps=rng.choice([100, 300]), tune=rng.random() < 0.5)
    if kind == "action2d":
        return dict(kind="action", dim=2, nx=_log_int(rng, 256, 1200), ny=_log_int(rng, 128, 400), nz=1,
                    seg=_log_int(rng, 200, 800), fast=fast, storage="f32", steps=10)
    if kind == "action3d":
        return dict(kind="action", dim=3, nx=_log_int(rng, 96, 192), ny=_log_int(rng, 64, 112),
                    nz=_log_int(rng, 64, 112), seg=2, fast=fast, storage="f32", steps=10)
    if kind == "coupled":
        return dict(kind="coupled", dim=2, nx=_log_int(rng, 256, 1200), ny=_log_int(rng, 128, 400), nz=1,
                    seg=_log_int(rng, 200, 800), fast=fast, storage="f32")
    if kind == "batch":
        return dict(kind="batch", dim=2, n=_log_int(rng, 8, 64), layout=rng.randrange(1 << 20), fast=True,
                    storage=rng.choice(["f16", "f16u"]), steps=10)
    if kind == "served":
        return dict(kind="served", n=_log_int(rng, 6, 24), layout=rng.randrange(1 << 20), fast=True, storage="f16", steps=10)
    return dict(kind="dropin", dim=3, nx=_log_int(rng, 48, 208), ny=_log_int(rng, 32, 104), nz=_log_int(rng, 32, 104),
                seg=0, fast=False, storage="f32", steps=100)


# ------------------------------------------------------------------ inputs
U_IN = 0.05  # inlet velocity of the streets and channels


def _flow(case, seed):
    """Moments (n, NM) in FP32 of a Taylor-Green field of amplitude about 0.04
    with a random phase, plus a vortex ring in 3D; Pi of the equilibrium."""
    g = np.random.default_rng(seed)
    ph, amp = g.uniform(0, 2 * np.pi, 3), 0.04 * g.uniform(0.8, 1.0)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    ax = [torch.arange(n, dtype=torch.float64, device=DEV) for n in (nz, ny, nx)]
    z, y, x = torch.meshgrid(*ax, indexing="ij")
    X, Y, Z = 2 * np.pi * x / nx + ph[0], 2 * np.pi * y / ny + ph[1], 2 * np.pi * z / nz + ph[2]
    if case["dim"] == 2:
        u = [amp * torch.sin(X) * torch.cos(Y), -amp * torch.cos(X) * torch.sin(Y)]
    else:
        u = [amp * torch.sin(X) * torch.cos(Y) * torch.cos(Z), -amp * torch.cos(X) * torch.sin(Y) * torch.cos(Z),
             torch.zeros_like(X)]
        rr = torch.hypot(x - nx / 2, y - ny / 2)
        dr, dz = rr - min(20.0, 0.2 * min(nx, ny)), z - nz / 2
        core = torch.exp(-(dr ** 2 + dz ** 2) / 18.0) * (amp / (3.0 * np.exp(-0.5)))
        r1 = torch.clamp(rr, min=1e-9)
        u = [u[0] - dz * core * (x - nx / 2) / r1, u[1] - dz * core * (y - ny / 2) / r1, dr * core]
    pairs = [(0, 0), (1, 1), (0, 1)] if case["dim"] == 2 else [(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]
    m = [torch.ones_like(X)] + u + [u[a] * u[b] for a, b in pairs]
    return torch.stack([q.reshape(-1) for q in m], 1).float().cpu().numpy()


def _street(case, seed):
    """Flags, noisy start and cylinder (vertices, elements) of a vortex street."""
    nx, ny = case["nx"], case["ny"]
    flags = wl.vortex_street_flags(nx, ny)
    u = np.random.default_rng(seed).uniform(-1e-3, 1e-3, (nx * ny, 2))
    u[:, 0] += U_IN  # the whole channel already flows past the cylinder
    m = wl.equilibrium_moments(u).astype(np.float32)
    v, e = wl.cylinder(case["seg"], 0.25 * nx, 0.5 * ny - 0.5, 0.1 * ny)
    return flags, m, v.astype(np.float32), e


def _channel_flags(case):
    """Walls on the y and z faces, the inlet at x = 0, the outlet at the other end."""
    f = np.full((case["nz"], case["ny"], case["nx"]), wl.FLUID, np.uint8)
    f[:, :, 0], f[:, :, -1] = wl.INLET_LEFT, wl.OUTLET_RIGHT
    f[:, 0], f[:, -1], f[0], f[-1] = wl.WALL, wl.WALL, wl.WALL, wl.WALL
    return f


def _inlet_of(seed):
    return float(np.float32(U_IN * np.random.default_rng(seed).uniform(0.8, 1.2)))


def _scene(case, seed):
    """Scene of an action case: a 2D swimmer or a 3D oscillating sphere."""
    rng = np.random.default_rng(seed)
    if case["dim"] == 2:
        return wl.SwimmerScene2D(case["nx"], case["ny"], case["seg"], rng)
    return serve.Scene3D(case["nx"], case["ny"], case["nz"], rng)


def _params_of(scene):
    return (scene.swimmer.params if hasattr(scene, "swimmer") else scene.params).copy()


def _action(params, a, phi):
    p = params.copy()
    p[0], p[2] = p[0] * a, phi
    return p


def _actions(seed, n=16):
    g = np.random.default_rng(seed + 77)
    return np.stack([g.uniform(0.5, 1.0, n), g.uniform(0, 2 * np.pi, n)], 1)


def _members(case, seed):
    """Uneven swimmers: the sizes of the benchmark's batch (by `layout`), the waves by the seed."""
    rng = np.random.default_rng(seed)
    return [wl.SwimmerScene2D(sc.nx, sc.ny, len(sc.swimmer.elems), rng)
            for sc in wl.batched_scenes(case["n"], case["layout"])]


def _episodes(case, seed):
    """Episodes that outlast any run: sizes of the server's default mix (by `layout`), swimmers and actions by the seed."""
    rng = np.random.default_rng(seed)
    eps = serve.make_episodes(1000.0, 1.0, case["layout"], steps=500)[:case["n"]]
    for ep in eps:
        ep.steps, ep.seed = 1 << 30, int(rng.integers(1 << 30))
        ep.actions = np.stack([rng.uniform(0.5, 1.0, 16), rng.uniform(0, 2 * np.pi, 16)], 1)
    return eps


def _domain(case, **kw):
    args = dict(storage=case["storage"], fast_math=case["fast"])
    args.update(kw)
    return capi.Domain(**args)


# ------------------------------------------------------------------ a pass
def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, k=0)
    if kind in ("monitor", "frame"):
        grid = dict(dim=case["dim"], nx=case["nx"], ny=case["ny"], nz=case["nz"])
        if kind == "monitor" or case["scene"] == "street":
            flags, m, v, e = _street(case, seed)
            d = _domain(case, **grid, viscosity=0.005)
            d.set_flags(flags)
            d.set_moments(m)
            d.set_boundary(v, np.zeros_like(v), e)
        else:
            d = _domain(case, **grid, viscosity=0.01, periodic=True)
            d.set_moments(_flow(case, seed))
        if case.get("tune"):
            d.autotune()
        s["dom"] = d
    elif kind == "action":
        sc = _scene(case, seed)
        d = _domain(case, **sc.domain_args())
        sc.setup(d, history=case["steps"])
        s.update(dom=d, params=_params_of(sc), actions=_actions(seed))
    elif kind == "coupled":
        sc = _scene(case, seed)
        d = _domain(case, **sc.domain_args())
        sc.setup(d)
        path = [tuple(a.astype(np.float32) for a in sc.swimmer.state(k * sc.dt)) for k in range(64)]
        s.update(dom=d, path=path)
    elif kind == "batch":
        b = capi.Batch(case["dim"], case["storage"], fast_math=case["fast"])
        doms, params = [], []
        for sc in _members(case, seed):
            d = _domain(case, **sc.domain_args())
            sc.setup(d, history=case["steps"])
            b.add(d)
            doms.append(d)
            params.append(_params_of(sc))
        s.update(batch=b, doms=doms, params=params, actions=_actions(seed))
    elif kind == "served":
        srv = serve.Server(storage=case["storage"], fast_math=case["fast"])
        eps = _episodes(case, seed)
        for ep in eps:
            ep.footprint = srv.footprint(ep)
            srv.admit(ep, 0.0)
        s.update(srv=srv, eps=eps)
    else:
        s["sim"], s["params"] = _simulator(case, seed)
    return s


def _simulator(case, seed):
    fs = freeflow_amd.enable_dropin()
    p = fs.SimulationParameters3D()
    p.fluid_nx, p.fluid_ny, p.fluid_nz = case["nx"], case["ny"], case["nz"]
    p.fluid_dx, p.dt, p.fluid_viscosity, p.fluid_density = 1.0, 1.0, 0.01, 1.0
    p.output_path = ""
    p.boundary_velocities = [_inlet_of(seed), 0.0, 0.0, 0.0, 0.0, 0.0]
    flags = _channel_flags(case)
    bcs = []
    for z, y, x in np.argwhere(flags != wl.FLUID).tolist():
        b = fs.BoundaryCondition()
        b.position, b.flag = [x, y, z], int(flags[z, y, x])
        bcs.append(b)
    p.boundaries = bcs
    sim = fs.Simulator3D(p)
    sim.initialize()
    return sim, p


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    k, s["k"] = s["k"], s["k"] + 1
    if kind == "monitor":
        s["dom"].step(1)
        return dict(wrench=s["dom"].body_wrench(), forces=s["dom"].step_vertex_forces())
    if kind == "frame":
        s["dom"].step(case["steps"])
        return dict(moments=s["dom"].moments())
    if kind == "action":
        d, a = s["dom"], s["actions"][k % len(s["actions"])]
        d.set_wave_params(_action(s["params"], *a)[None, :])
        d.step(case["steps"])
        v, u = d.boundary()
        return dict(wrench=d.wrench_history(case["steps"]), power=d.power_history(case["steps"]), verts=v, vels=u)
    if kind == "coupled":
        s["dom"].update_boundary(*s["path"][k % len(s["path"])])
        s["dom"].step(1)
        return dict(forces=s["dom"].step_vertex_forces())
    if kind == "batch":
        a = s["actions"][k % len(s["actions"])]
        for d, p in zip(s["doms"], s["params"]):
            d.set_wave_params(_action(p, *a)[None, :])
        s["batch"].step(case["steps"])
        s["batch"].sync()
        # the controller's readings, and the flow of the member being watched
        return dict(wrench=np.concatenate([d.wrench_history(case["steps"]) for d in s["doms"]]),
                    power=np.concatenate([d.power_history(case["steps"]) for d in s["doms"]]),
                    moments=s["doms"][0].moments())
    if kind == "served":
        s["srv"].step_all()
        out = dict(w2=np.concatenate([ep.wrench[-1] for ep in s["eps"] if ep.kind == 2]))
        if any(ep.kind == 3 for ep in s["eps"]):
            out["w3"] = np.concatenate([ep.wrench[-1] for ep in s["eps"] if ep.kind == 3])
        for ep in s["eps"]:
            del ep.wrench[:]
        s["srv"].lat.clear()
        return out
    for _ in range(case["steps"]):
        s["sim"].step()
    return dict(moments=s["sim"].get_fluid_moments())


# ------------------------------------------------------------------ what a pass cannot do without
def _cells(case):
    if case["kind"] == "batch":
        return [(2, sc.nx * sc.ny) for sc in wl.batched_scenes(case["n"], case["layout"])]
    if case["kind"] == "served":
        return [(ep.kind, ep.cells) for ep in _episodes(case, 1)]
    return [(case["dim"], case["nx"] * case["ny"] * case["nz"])]


def work(case):
    """Every stored moment read and written and the flag read once per cell and
    step (the bodies add far less), and the field that a frame returns; the
    operations are those of rebuilding, summing and relaxing the populations."""
    size = {"f32": 4, "f16": 2, "bf16": 2, "f16u": 2}[case["storage"]]
    bytes_, flops = 0.0, 0.0
    for dim, n in _cells(case):
        planes = (6 if dim == 2 else 10) + (dim if case["storage"] == "f16u" else 0)
        steps = case.get("steps", 1)
        bytes_ += steps * n * (2 * planes * size + 1)
        flops += steps * n * (150 if dim == 2 else 420)
        if case["kind"] in ("frame", "dropin"):
            bytes_ += n * (6 if dim == 2 else 10) * 4
    return dict(bytes=bytes_, flops=flops)


# ------------------------------------------------------------------ the step in 64 bits
_C2 = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)]
_C3 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, -1, 0),
       (1, 0, 1), (-1, 0, -1), (0, 1, 1), (0, -1, -1), (1, -1, 0), (-1, 1, 0), (1, 0, -1), (-1, 0, 1), (0, 1, -1),
       (0, -1, 1), (1, 1, 1), (-1, -1, -1), (1, 1, -1), (-1, -1, 1), (1, -1, 1), (-1, 1, -1), (-1, 1, 1), (1, -1, -1)]
_PAIRS = {2: [(0, 0), (1, 1), (0, 1)], 3: [(0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2)]}
# outlet flag -> (axis of its velocity, step to the neighbour, outward sign)
_OUTLETS = {2: {21: (1, -1, 1), 22: (1, 1, -1), 19: (0, 1, -1), 20: (0, -1, 1)},
            3: {21: (2, -1, 1), 22: (2, 1, -1), 19: (0, 1, -1), 20: (0, -1, 1), 23: (1, 1, -1), 24: (1, -1, 1)}}


def _t(a, dtype=torch.float64):
    return torch.as_tensor(np.asarray(a), device=DEV).to(dtype)


class _Exact:
    """Stream-collide with walls, outlets and one moving body, in FP64."""

    def __init__(self, dim, nx, ny, nz, viscosity, dx=1.0, dt=1.0, rho=1.0, flags=None, periodic=False):
        self.dim, self.n = dim, (nx, ny, nz)[:dim]
        self.shape = tuple(reversed(self.n))
        self.c = _C2 if dim == 2 else _C3
        w1 = {0: 2 / 3, 1: 1 / 6, -1: 1 / 6}
        D, mix = dim, [(a, b) for a in range(dim) for b in range(dim) if a != b]
        rows = []  # weights of the populations over the Hermite coefficients of coefs()
        for c in self.c:
            h2 = [c[a] * c[a] - 1 / 3 for a in range(D)]
            r = [1.0] + [3.0 * c[a] for a in range(D)]
            r += [4.5 * h2[a] if a == b else 9.0 * c[a] * c[b] for a, b in _PAIRS[D]]
            r += [13.5 * h2[a] * c[b] for a, b in mix] + ([27.0 * c[0] * c[1] * c[2]] if D == 3 else [])
            rows.append(np.array(r) * np.prod([w1[a] for a in c]))
        self.mix, self.W = mix, _t(np.array(rows))
        self.S = _t(np.array([[1.0] * len(self.c)] + [[c[a] for c in self.c] for a in range(D)]
                             + [[c[a] * c[b] for c in self.c] for a, b in _PAIRS[D]]))
        self.inv = [self.c.index(tuple(-a for a in c)) for c in self.c]
        self.omega = float(np.float32(1.0 / (float(np.float32(viscosity)) * 3.0 + 0.5)))
        self.dx, self.dt, self.periodic = dx, dt, periodic
        cells = int(np.prod(self.shape))
        f = np.full(cells, wl.FLUID, np.uint8) if flags is None else np.asarray(flags).reshape(-1)
        self.flags = _t(f, torch.int64).reshape(self.shape)
        self.upd = (self.flags == 1) | (self.flags == 4)
        self.wall = (self.flags == 3) | ((self.flags >= 5) & (self.flags <= 11))
        self.walls = bool(self.wall.any())
        self.cf = capi.cf_of(dim, rho, dx, dt)
        self.body = None

    def set(self, m):
        m = _t(m).reshape(self.shape + (-1,))
        self.m = [m[..., q].contiguous() for q in range(m.shape[-1])]
        self.old = list(self.m)
        self.outlets = self._outlet_cells()

    def rest(self, inlet=0.0):
        u = [torch.where(self.flags == 13, inlet, 0.0).double()] + [torch.zeros(self.shape, device=DEV).double()] * (
            self.dim - 1)
        self.set(torch.stack([torch.ones_like(u[0])] + u + [u[a] * u[b] for a, b in _PAIRS[self.dim]], -1).cpu())

    def set_body(self, verts, elems):
        self.v = _t(np.asarray(verts, np.float32))
        self.e = _t(np.asarray(elems).astype(np.int64), torch.int64)
        self.ref = self.v.mean(0)
        self.body = True

    def coefs(self, m):
        """Hermite coefficients (rows) of moments m; 2D leaves rho out of the third order's first two terms."""
        D, rho, u = self.dim, m[0], m[1:1 + self.dim]
        pi = {}
        for (a, b), p in zip(_PAIRS[D], m[1 + D:]):
            pi[(a, b)] = pi[(b, a)] = p
        r = rho if D == 3 else 1.0
        out = [rho] + [rho * x for x in u] + [rho * p for p in m[1 + D:]]
        out += [r * (pi[(a, a)] * u[b] + 2 * pi[(a, b)] * u[a]) - 2 * rho * u[a] * u[a] * u[b] for a, b in self.mix]
        if D == 3:
            out.append(rho * (pi[(0, 1)] * u[2] + pi[(1, 2)] * u[0] + pi[(0, 2)] * u[1] - 2 * u[0] * u[1] * u[2]))
        return torch.stack(out).reshape(len(out), -1)

    def shift(self, a, c, wrap):
        if wrap:
            return torch.roll(a, tuple(reversed(c)), tuple(range(self.dim)))
        for k, s in enumerate(c):
            if s:
                n, ax = self.n[k], self.dim - 1 - k
                a = a.index_select(ax, (torch.arange(n, device=DEV) - s).clamp(0, n - 1))
        return a

    def _outlet_cells(self):
        out = []
        for f, (axis, step, sign) in _OUTLETS[self.dim].items():
            at, ax = torch.nonzero(self.flags == f), self.dim - 1 - axis
            nb = at.clone()
            nb[:, ax] += step
            ok = (nb[:, ax] >= 0) & (nb[:, ax] < self.n[axis])
            at, nb = at[ok], nb[ok]
            ok = self.flags[tuple(nb.T)] == 1
            if ok.any():
                out.append((1 + axis, 1 + self.dim + axis, sign, tuple(at[ok].T), tuple(nb[ok].T)))
        return out

    def step(self, verts=None, vels=None):
        """One step with the body at `verts`; returns (wrench, power, vertex forces)."""
        D, Q, om, res = self.dim, len(self.c), self.omega, None
        f = (self.W @ self.coefs(self.m)).reshape((Q,) + self.shape)
        p = torch.empty_like(f)
        for i in range(Q):
            p[i] = self.shift(f[i], self.c[i], self.periodic)
            if D == 3 and self.walls:
                p[i] = torch.where(self.shift(self.wall, self.c[i], True), f[self.inv[i]], p[i])
        p.clamp_(min=0.0)
        if self.body:
            res = self._links(f, p, verts, vels)
        m = (self.S @ p.reshape(Q, -1)).reshape((-1,) + self.shape)
        rho, u, pi = m[0], m[1:1 + D] / m[0], m[1 + D:] / m[0]
        tr, uu = sum(pi[:D]) / D, (u * u).sum(0) / D
        new = [rho] + list(u)
        for j, (a, b) in enumerate(_PAIRS[D]):
            if a == b:
                new.append(uu + (1 - om) * (pi[j] - tr) + om * (u[a] * u[a] - uu))
            else:
                new.append((1 - om) * pi[j] + om * u[a] * u[b])
        new = [torch.where(self.upd, x, o) for x, o in zip(new, self.old)]
        for comp, pcomp, sign, at, nb in self.outlets:
            up = new[comp][nb]
            new[comp][at] = torch.where(sign * up > 0, up, new[comp][at])
            new[pcomp][at] = up * up
        self.old, self.m = self.m, new
        return res

    def _hit(self, x1, x2, tri):
        """Links x1 -> x2 against elements tri (..., D, D): hit, depth, barycentrics, point."""
        if self.dim == 2:
            (ax, ay), (bx, by) = (tri[..., 0, 0], tri[..., 0, 1]), (tri[..., 1, 0], tri[..., 1, 1])
            a1 = (x1[..., 0] - x2[..., 0]) * (ay - by) - (x1[..., 1] - x2[..., 1]) * (ax - bx)
            t = ((bx - x2[..., 0]) * (ay - by) - (by - x2[..., 1]) * (ax - bx)) / a1
            pt = t[..., None] * x1 + (1 - t)[..., None] * x2
            hit = (a1 != 0) & (t > 0) & (t < 1) & ((ax - pt[..., 0]) * (bx - pt[..., 0]) < 0)
            b0 = (tri[..., 1, :] - pt).norm(dim=-1) / (tri[..., 1, :] - tri[..., 0, :]).norm(dim=-1)
            return hit, 1 - t, torch.stack([b0, 1 - b0], -1), pt
        v0 = tri[..., 0, :]
        e1, e2, dd = tri[..., 1, :] - v0, tri[..., 2, :] - v0, x2 - x1
        n = torch.linalg.cross(e1, e2)
        n = n / n.norm(dim=-1, keepdim=True)
        den = (n * dd).sum(-1)
        t = (n * (v0 - x1)).sum(-1) / den
        pt = x1 + t[..., None] * dd
        w = pt - v0
        d00, d01, d11 = (e1 * e1).sum(-1), (e1 * e2).sum(-1), (e2 * e2).sum(-1)
        d20, d21 = (w * e1).sum(-1), (w * e2).sum(-1)
        q = d00 * d11 - d01 * d01
        b1, b2 = (d11 * d20 - d01 * d21) / q, (d00 * d21 - d01 * d20) / q
        hit = (t >= 0) & (t <= 1) & ((den / dd.norm(dim=-1)).abs() > 1e-6)
        hit = hit & (b1 >= -1e-6) & (b2 >= -1e-6) & (b1 + b2 <= 1 + 1e-6)
        return hit, t, torch.stack([1 - b1 - b2, b1, b2], -1), pt

    def _links(self, f, p, verts, vels):
        D, K, dx = self.dim, len(self.c) - 1, self.dx
        tri = verts[self.e]  # (E, D vertices, D)
        size = _t(self.n, torch.int64)
        lo = ((tri.amin(1) / dx).trunc().long() - 1).clamp(min=0)
        hi = torch.minimum((tri.amax(1) / dx).trunc().long() + 1, size - 1)
        span = (hi - lo + 1).clamp(min=0)
        grid = torch.meshgrid(*[torch.arange(int(s), device=DEV) for s in span.amax(0)], indexing="ij")
        off = torch.stack([g.reshape(-1) for g in grid], -1)
        ok = (off[None] < span[:, None]).all(-1)
        el, k = torch.nonzero(ok, as_tuple=True)
        cell = lo[el] + off[k]
        ok = self.upd[tuple(cell.flip(-1).T)]
        el, cell = el[ok], cell[ok]
        c = _t(self.c[1:], torch.int64)
        hit = self._hit((cell * dx).double()[:, None], ((cell[:, None] - c) * dx).double(), tri[el][:, None])
        at, l = torch.nonzero(hit[0], as_tuple=True)
        el, cell = el[at], cell[at]
        depth = hit[1][at, l]
        flat = cell[:, 0] + self.n[0] * cell[:, 1] + (self.n[0] * self.n[1] * cell[:, 2] if D == 3 else 0)
        link, back = torch.unique(flat * K + l, return_inverse=True)
        key = (depth * 32768).long() * 65536 + el  # nearest element of a link
        best = torch.full_like(link, 1 << 60).scatter_reduce(0, back, key, "amin")
        won = torch.nonzero(best[back] == key)[:, 0]
        el, cell, l, at = el[won], cell[won], l[won], at[won]
        src = cell - c[l]
        ok = ((src >= 0) & (src < size)).all(-1)
        ok &= ~self.wall[tuple((src % size).flip(-1).T)]
        el, cell, l, at, src = el[ok], cell[ok], l[ok], at[ok], src[ok]
        bary, pt = hit[2][at, l], hit[3][at, l]
        idx = tuple(cell.flip(-1).T)
        uv = vels[self.e[el]]
        uw = (uv * bary[..., None]).sum(1) * (self.dt / dx)
        mc = [q[idx] for q in self.m]
        ms = [mc[0]] + [uw[:, a] for a in range(D)]
        ms += [mc[1 + D + j] + uw[:, a] * uw[:, b] - mc[1 + a] * mc[1 + b] for j, (a, b) in enumerate(_PAIRS[D])]
        l1 = l + 1  # direction of the link
        fin = f[(_t(self.inv, torch.int64)[l1],) + idx].clamp(min=0.0)
        fout = (self.coefs(ms) * self.W[l1].T).sum(0)
        p[(l1,) + idx] = fout
        cc = c[l].double()
        F = (fin[:, None] * (-cc - uw) - fout[:, None] * (cc - uw)) * self.cf
        share = F[:, None, :] * bary[..., None]  # (links, D vertices, D)
        vf = torch.zeros_like(verts).index_add(0, self.e[el].reshape(-1), share.reshape(-1, D))
        r = pt - self.ref
        if D == 2:
            tq = (r[:, 0] * F[:, 1] - r[:, 1] * F[:, 0]).sum()[None]
        else:
            tq = torch.linalg.cross(r, F).sum(0)
        return torch.cat([F.sum(0), tq]), -(vf * vels).sum(), vf

    def moments(self):
        return torch.stack(self.m, -1).reshape(-1, len(self.m))


def _exact_scene(sc, dim):
    a = sc.domain_args()
    x = _Exact(dim, a["nx"], a["ny"], a.get("nz", 1), a["viscosity"], a.get("dx", 1.0), a.get("dt", 1.0),
               a.get("fluid_density", 1.0), getattr(sc, "flags", None))
    x.rest()
    if dim == 2:
        x.set_body(sc.swimmer.state(0.0)[0], sc.swimmer.elems)
        x.at_rest, x.s = _t(sc.swimmer.rest.astype(np.float32)), _t(sc.swimmer.s.astype(np.float32))
    else:
        x.set_body(sc.v, sc.f)
        x.at_rest, x.s = _t(sc.v.astype(np.float32)), _t(sc.s)
    return x


def _wave(x, p, t):
    th = 2 * np.pi * (x.s * p[3] - p[1] * t) + p[2]
    v, u = x.at_rest.clone(), torch.zeros_like(x.at_rest)
    v[:, 1] += p[0] * x.s * torch.sin(th)
    u[:, 1] = -2 * np.pi * p[1] * p[0] * x.s * torch.cos(th)
    return v, u


def _exact_action(sc, dim, p, steps):
    """An action's interval from the start: wrenches, powers, last shape, moments."""
    x = _exact_scene(sc, dim)
    w, pw = [], []
    for k in range(steps):
        v, u = _wave(x, p, k * x.dt)
        a, b, _ = x.step(v, u)
        w.append(a)
        pw.append(b)
    return torch.stack(w)[:, None], torch.stack(pw)[:, None], v, u, x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("monitor", "frame"):
        street = kind == "monitor" or case["scene"] == "street"
        flags, m, v, e = _street(case, seed) if street else (None, _flow(case, seed), None, None)
        x = _Exact(case["dim"], case["nx"], case["ny"], case["nz"], 0.005 if street else 0.01, flags=flags,
                   periodic=not street)
        x.set(m)
        if street:
            x.set_body(v, e)
        for _ in range(case.get("steps", 1)):
            r = x.step(_t(v), torch.zeros_like(_t(v))) if street else x.step()
        return dict(wrench=r[0][None], forces=r[2]) if kind == "monitor" else dict(moments=x.moments())
    if kind == "action":
        sc = _scene(case, seed)
        w, pw, v, u, _ = _exact_action(sc, case["dim"], _action(_params_of(sc), *_actions(seed)[0]), case["steps"])
        return dict(wrench=w, power=pw, verts=v, vels=u)
    if kind == "coupled":
        sc = _scene(case, seed)
        x = _exact_scene(sc, 2)
        return dict(forces=x.step(*(_t(a.astype(np.float32)) for a in sc.swimmer.state(0.0)))[2])
    if kind == "batch":
        a, got = _actions(seed)[0], []
        for sc in _members(case, seed):
            got.append(_exact_action(sc, 2, _action(_params_of(sc), *a), case["steps"]))
            if len(got) > 1:
                got[-1] = got[-1][:2]
        return dict(wrench=torch.cat([g[0] for g in got]), power=torch.cat([g[1] for g in got]),
                    moments=got[0][4].moments())
    if kind == "served":
        w = {2: [], 3: []}
        for ep in _episodes(case, seed):
            rng = np.random.default_rng(ep.seed)
            sc = (wl.SwimmerScene2D(ep.nx, ep.ny, int(rng.integers(200, 801)), rng) if ep.kind == 2
                  else serve.Scene3D(ep.nx, ep.ny, ep.nz, rng))
            w[ep.kind].append(_exact_action(sc, ep.kind, _action(_params_of(sc), *ep.actions[0]), case["steps"])[0])
        return {"w%d" % d: torch.cat(v) for d, v in w.items() if v}
    x = _Exact(3, case["nx"], case["ny"], case["nz"], 0.01, flags=_channel_flags(case))
    x.rest(_inlet_of(seed))
    for _ in range(case["steps"]):
        x.step()
    return dict(moments=x.moments().reshape(case["nz"], case["ny"], case["nx"], 10))
