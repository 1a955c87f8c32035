"""The work whose time is kept: what users of the engine have it do.

A *flow* case is one call of the time loop (``Solver.step``) on a lattice whose
solver the program already holds, followed by reading the fields back
(``Solver.macro``) and the residual or force rows of those steps; a *sweep*
case is the same for a packed lattice of many cavities; a *net* case is one
prediction or one gradient of the warm-start network on host arrays.  The
state is the solver or network itself, so a second pass continues the run.

``exact`` evolves the same lattice in float64 with plain torch operations, and
evaluates the same network in float64.
"""
import math

import numpy as np
import torch

import parallellbmcranfield_amd as lbm

CX = (0, 1, 0, -1, 0, 1, -1, -1, 1)
CY = (0, 0, 1, 0, -1, 1, 1, -1, -1)
OPP = (0, 3, 4, 1, 2, 7, 8, 5, 6)
WEIGHT = (4 / 9,) + (1 / 9,) * 4 + (1 / 36,) * 4
MODEL = {"bgk": lbm.BGKW, "trt": lbm.TRT, "mrt": lbm.MRT}
STORE = {"f64": lbm.PREC_F64, "f32": lbm.PREC_F32, "f16": lbm.PREC_F16, "f16sr": lbm.PREC_F16_SR}
WORD = {"f64": 8, "f32": 4, "f16": 2, "f16sr": 2}
RESID = {"reference": lbm.RESID_REFERENCE, "full": lbm.RESID_FULL, "velocity": lbm.RESID_VELOCITY,
         "none": lbm.RESID_NONE}
LID = 0.1
# Flops of one node update: streaming has none; moments, equilibrium, relaxation.
FLOPS = {"bgk": 120, "trt": 150, "mrt": 150}


# ------------------------------------------------------------------ the cases
def cavity(nx, ny, model, store, steps, re, resid="none", every=100, rects=0, start="field"):
    return dict(kind="cavity", nx=nx, ny=ny, model=model, store=store, steps=steps, re=re,
                resid=resid, every=every, rects=rects, start=start)


def channel(nx, ny, d, model, store, steps, every=10, re=100.0):
    return dict(kind="channel", nx=nx, ny=ny, d=d, model=model, store=store, steps=steps, re=re,
                resid="none", every=every)


def sweep(count, lo, hi, store, steps):
    return dict(kind="sweep", count=count, lo=lo, hi=hi, store=store, steps=steps, model="mrt",
                every=100)


def net(task, grid, batch, samples, channels=8, dilation=4):
    return dict(kind="net", task=task, grid=grid, batch=batch, samples=samples, channels=channels,
                dilation=dilation)


def listed():
    return [
        # a monitored run: one step of a small lattice at a time, fields read after it
        dict(cavity(33, 33, "bgk", "f64", 1, 50.0, "reference", start="reference"),
             name="monitor_33_f64"),
        # the reference program on its coarse mesh between two autosaves: its own
        # start, its own residual after every step
        dict(cavity(125, 125, "trt", "f64", 200, 1000.0, "reference", start="reference"),
             name="coarse_125_trt_f64"),
        # the small validation cavity (Re 100), change of the velocity every 100 steps
        dict(cavity(129, 129, "bgk", "f64", 1000, 100.0, "velocity"), name="cavity_129_bgk_f64"),
        # one cavity of a sweep run alone (uneven sides, an obstacle)
        dict(cavity(257, 181, "mrt", "f32", 1000, 400.0, "velocity", rects=1),
             name="cavity_257x181_mrt_f32"),
        # a mid-size production cavity
        dict(cavity(1025, 1025, "mrt", "f32", 2000, 1000.0), name="cavity_1025_mrt_f32"),
        # half-precision storage, ragged sides
        dict(cavity(1501, 1403, "bgk", "f16", 2000, 1000.0), name="cavity_1501x1403_bgk_f16"),
        # the reference's precision on a large lattice
        dict(cavity(2049, 2049, "bgk", "f64", 1500, 1000.0), name="cavity_2049_bgk_f64"),
        # the headline lattice
        dict(cavity(4097, 4097, "mrt", "f32", 4000, 1000.0), name="cavity_4097_mrt_f32"),
        # cylinder wake: curved walls, parabolic inlet, pressure outlet, force series
        dict(channel(2049, 513, 64, "mrt", "f32", 2000), name="cylinder_2049x513_mrt_f32"),
        # many cavities in one lattice, each watched for its own convergence
        dict(sweep(48, 65, 257, "f32", 1000), name="sweep_48_f32"),
        # warm starts for a batch of new cavities
        dict(net("predict", 257, 16, 32), name="net_predict_257"),
        # one training gradient of the same network
        dict(net("gradients", 257, 16, 16), name="net_gradients_257"),
    ]


def log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cavity"] * 6 + ["channel"] * 2 + ["sweep"] * 2 + ["net"] * 2)
    if kind == "net":
        task = rng.choice(["predict", "gradients"])
        grid = log_size(rng, 48, 257)
        batch = rng.choice([4, 8, 16])
        samples = rng.randint(1, 2 * batch) if task == "predict" else rng.randint(1, batch)
        return net(task, grid, batch, samples, rng.choice([3, 8]), rng.choice([1, 2, 4]))
    model = rng.choice(["bgk", "trt", "mrt"])
    store = rng.choice(["f64", "f64", "f32", "f32", "f32", "f16", "f16sr"])
    if kind == "sweep":
        count = log_size(rng, 4, 96)
        lo = rng.randint(24, 96)
        return sweep(count, lo, rng.randint(lo + 16, 280), rng.choice(["f32", "f32", "f16"]),
                     100 * rng.randint(1, 8))
    if kind == "channel":
        ny = log_size(rng, 40, 520)
        nx = int(ny * rng.uniform(2.0, 5.0))
        steps = max(10, min(1000, int(1e9 / (nx * ny))))
        return channel(nx, ny, max(6, ny // rng.randint(5, 9)), model,
                       "f64" if store == "f64" else "f32", steps, rng.choice([5, 10, 50]))
    nx = log_size(rng, 24, 4000)
    ny = min(4000, max(24, int(nx * rng.uniform(0.5, 1.5))))
    steps = max(1, min(rng.choice([10, 100, 1000]), int(8e9 / (nx * ny))))
    resid, every = rng.choice([("none", 1), ("velocity", 100), ("full", 50), ("velocity", 10)])
    start = "field"
    if store == "f64" and nx <= 600 and rng.random() < 0.5:
        resid, every, start = "reference", 1, "reference"
    return cavity(nx, ny, model, store, steps, rng.uniform(50.0, 1000.0), resid, every,
                  rng.randint(0, 2) if min(nx, ny) >= 64 else 0, start)


# ------------------------------------------------- inputs, made from the seed
def obstacles(rng, nx, ny, count):
    out = []
    for _ in range(count):
        w, h = (max(2, int(rng.uniform(0.05, 0.25) * s)) for s in (nx, ny))
        i0, j0 = int(rng.integers(4, nx - w - 3)), int(rng.integers(4, ny - h - 3))
        out.append((i0, j0, i0 + w - 1, j0 + h - 1))
    return out


def swirl(rng, n, m):
    """A smooth start: rho, u, v on n x m cells, a few divergence-free modes."""
    x = (np.arange(n) + 0.5) / n * math.pi
    y = (np.arange(m) + 0.5) / m * math.pi
    u, v = np.zeros((m, n)), np.zeros((m, n))
    for k, l in ((1, 1), (2, 1), (1, 2), (3, 2)):
        a = rng.uniform(-0.02, 0.02)
        u += np.outer(a * l * np.cos(l * y), np.sin(k * x))
        v -= np.outer(a * k * np.sin(l * y), np.cos(k * x))
    rho = 1.0 + 0.5 * (u * u).mean() * np.outer(np.cos(y), np.cos(x))
    return rho.ravel(), u.ravel(), v.ravel()


def rates(nu):
    om = 1.0 / (3.0 * float(np.float32(nu)) + 0.5)
    return (0.0, 1.4, 1.4, 0.0, 1.2, 0.0, 1.2, om, om)


def flow_inputs(case, seed):
    """Numbers and arrays of a cavity or channel case: what both sides start from."""
    rng = np.random.default_rng([seed, 17])
    nx, ny = case["nx"], case["ny"]
    f = dict(rects=[], field=None, crit=-1.0)
    vary = rng.uniform(0.9, 1.1)
    if case["kind"] == "channel":
        f.update(uavg=vary * 0.05 / 1.5, rho=1.0, inlet=1, curved=1, outlet=lbm.OUTLET_PRESSURE)
        f["nu"] = f["uavg"] * case["d"] / case["re"]
        f["centre"] = (0.25 * nx + rng.uniform(-1, 1), 0.5 * ny + rng.uniform(-1, 1))
        return f
    f.update(inlet=2, curved=2, outlet=2)
    if case["start"] == "reference":  # the shipped cases' parameters
        f.update(uavg=vary * 0.08, rho=5.0)
    else:
        f.update(uavg=vary * LID, rho=1.0, field=swirl(rng, nx + 2, ny + 3), crit=1e-30)
    f["nu"] = f["uavg"] * nx / case["re"]
    f["rects"] = obstacles(rng, nx, ny, case["rects"])
    return f


def sweep_inputs(case, seed):
    # the sides belong to the case, so that every seed is the same amount of work
    shape = np.random.default_rng([case["count"], case["lo"], case["hi"]])
    rng = np.random.default_rng([seed, 23])
    specs = []
    for _ in range(case["count"]):
        nx, ny = (int(shape.integers(case["lo"], case["hi"] + 1)) for _ in range(2))
        re = math.exp(rng.uniform(math.log(100.0), math.log(1000.0)))
        lid = rng.uniform(0.08, 0.1)
        specs.append(dict(nx=nx, ny=ny, nu=lid * nx / re, lid=lid,
                          rects=obstacles(rng, nx, ny, int(rng.integers(0, 4)))))
    return specs


def net_shapes(base=32, levels=4):
    c = [base << l for l in range(levels)]
    convs = []
    for l in range(levels):
        convs += [(32 if l == 0 else c[l - 1], 0, c[l]), (c[l], 0, c[l])]
    for l in range(levels - 2, -1, -1):
        convs += [(c[l], c[l + 1], c[l]), (c[l], 0, c[l])]
    return convs


def net_inputs(case, seed):
    rng = np.random.default_rng([seed, 31])
    g, nb, ch = case["grid"], case["samples"], case["channels"]
    parts = []
    for i, (c0, c1, co) in enumerate(net_shapes()):
        ci = c0 + c1
        real = ch if i == 0 else ci
        w = rng.normal(0, math.sqrt(2.0 / (9 * real)), (co, 9, ci)).astype(np.float32)
        w[:, :, real:] = 0
        parts += [w.ravel(), rng.normal(0, 0.05, co).astype(np.float32)]
    parts += [rng.normal(0, 0.02, 3 * 32).astype(np.float32), np.zeros(3, np.float32)]
    x = np.zeros((nb, g, g, ch), np.float32)
    t = np.zeros((nb, g, g, 3), np.float32)
    s = np.arange(g, dtype=np.float32) / (g - 1)
    for b in range(nb):
        w, h = g, int(rng.uniform(0.5, 1.0) * g)
        mask = np.zeros((g, g), np.float32)
        mask[:h, :w] = 1
        i0, j0, q = int(rng.integers(3, w // 2)), int(rng.integers(3, h // 2)), g // 8
        mask[j0:j0 + q, i0:i0 + q] = 0
        x[b, ..., 0] = mask
        x[b, ..., 1], x[b, ..., 2] = rng.uniform(0, 1, 2)
        if ch == 8:
            x[b, ..., 3], x[b, ..., 4] = s, 1 - s
            x[b, ..., 5], x[b, ..., 6] = s[:, None], np.float32(h / g) - s[:, None]
            x[b, ..., 7] = np.minimum(s, 1 - s) * 0.5
            x[b, ..., 3:] *= mask[..., None]
        a = rng.uniform(-1, 1, 3).astype(np.float32)
        sx, sy = np.sin(math.pi * s), np.sin(2 * math.pi * s)
        t[b, ..., 0] = a[0] * np.outer(sy, sx) * mask
        t[b, ..., 1] = -a[1] * np.outer(sx, sy) * mask
        t[b, ..., 2] = a[2] * np.outer(np.cos(math.pi * s), sx) * mask
    return np.concatenate(parts), x, t


# ---------------------------------------------------------- the calls measured
def options(case, f):
    kw = dict(collision=MODEL[case["model"]], uavg=f["uavg"], rho_ini=f["rho"], viscosity=f["nu"],
              inlet_profile=f["inlet"], curved=f["curved"], outlet_profile=f["outlet"],
              precision=STORE[case["store"]], resid_kind=RESID[case["resid"]])
    if case["kind"] == "channel" or case["start"] != "reference":
        kw.update(init=lbm.INIT_REST, resid_every=case["every"], use_stop_rule=0)
        if case["model"] == "mrt":
            kw.update(mrt_textbook_meq=1, mrt_rates=rates(f["nu"]))
        if case["model"] == "trt":
            kw.update(trt_lambda=0.25, trt_fp64_parts=1)
    if case["kind"] == "channel":
        kw.update(force_id=5, force_every=case["every"], outlet_rho=1.0)
    elif case["resid"] == "velocity" and f["crit"] > 0:  # watched for convergence
        kw.update(use_stop_rule=1, crit_v=f["crit"], crit_rho=-1.0, max_iterations=2**31 - 1)
    return lbm.make_options(**kw)


def prepare(case, seed):
    if case["kind"] == "net":
        params, x, t = net_inputs(case, seed)
        n = lbm.Net(case["grid"], case["grid"], batch=case["batch"],
                    in_channels=case["channels"], dilation=case["dilation"])
        n.set_params(params)
        return dict(case=case, net=n, x=x, t=t)
    if case["kind"] == "sweep":
        specs = sweep_inputs(case, seed)
        packed = lbm.Case.pack([lbm.Case.cavity_ex(s["nx"], s["ny"], s["rects"]) for s in specs])
        o = lbm.make_options(collision=lbm.MRT, uavg=LID, rho_ini=1.0, viscosity=0.01,
                             precision=STORE[case["store"]], init=lbm.INIT_REST,
                             resid_kind=lbm.RESID_VELOCITY, resid_every=case["every"],
                             crit_v=1e-30, use_stop_rule=1, max_iterations=2**31 - 1,
                             mrt_textbook_meq=1, mrt_rates=rates(0.01))
        return dict(case=case, solver=lbm.Solver(packed, o,
                                                 instances=[(s["nu"], s["lid"]) for s in specs]))
    f = flow_inputs(case, seed)
    if case["kind"] == "channel":
        mesh = lbm.Case.channel(case["nx"], case["ny"], *f["centre"], case["d"] / 2)
    elif f["rects"] or case["nx"] != case["ny"]:
        mesh = lbm.Case.cavity_ex(case["nx"], case["ny"], f["rects"])
    else:
        mesh = lbm.Case.cavity(case["nx"])
    return dict(case=case, solver=lbm.Solver(mesh, options(case, f), field=f["field"]))


def run(state):
    case = state["case"]
    if case["kind"] == "net":
        if case["task"] == "predict":
            return state["net"].predict(state["x"])
        return state["net"].gradients(state["x"], state["t"])
    s = state["solver"]
    s.step(case["steps"])
    out = dict(zip(("rho", "u", "v"), s.macro()))
    if case["kind"] == "channel":
        out["force_at"], out["force"] = s.force_history()
    elif case["kind"] == "sweep":
        out["converged_at"], _, out["resid"] = s.batch_status()
    elif case["resid"] != "none":
        out["resid_at"], out["resid"] = s.residual_history()
    return out


def work(case):
    if case["kind"] == "net":
        # each conv: 2 * 9 * Cin * Cout per pixel of its level; a gradient has
        # the weight and data gradients beside it (none of the first conv's data)
        g, nb = case["grid"], case["samples"]
        px = [nb * (-(-g // 2**l))**2 for l in range(4)]
        level = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0]
        per = [2 * 9 * (c0 + c1) * co * px[l] for (c0, c1, co), l in zip(net_shapes(), level)]
        params = sum(9 * (c0 + c1) * co + co for c0, c1, co in net_shapes()) + 99
        io = 4 * px[0] * case["channels"] + 4 * params
        if case["task"] == "predict":
            return dict(bytes=io + 12 * px[0], flops=sum(per))
        return dict(bytes=io + 12 * px[0] + 4 * params, flops=3 * sum(per) - per[0])
    if case["kind"] == "sweep":
        nodes = sum(s["nx"] * s["ny"] for s in sweep_inputs(case, 0))
    else:
        nodes = case["nx"] * case["ny"]
    # the state read and written once, the fields written once
    return dict(bytes=nodes * (18 * WORD[case["store"]] + 24),
                flops=nodes * case["steps"] * FLOPS[case["model"]])


# ------------------------------------------------------------- in 64 bits
def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def links(kind, nx, ny, n, m, rects=(), centre=None, d=0):
    """Fluid flags [m, n], link types [9, m, n], cut distances, boundary ids."""
    jj, ii = np.mgrid[0:m, 0:n]
    inside = (ii >= 1) & (ii <= nx) & (jj >= 1) & (jj <= ny)
    fluid = inside.copy()
    for i0, j0, i1, j1 in rects:
        fluid[j0:j1 + 1, i0:i1 + 1] = False
    delta = 1.0 / (ny if kind == "channel" else max(nx, ny))
    x, y = ((np.arange(k) - 0.5) * delta for k in (n, m))
    if centre is not None:
        fluid &= ~((ii - centre[0])**2 + (jj - centre[1])**2 <= 0.25 * d * d)
    bc = np.zeros((9, m, n), np.int8)
    q = np.full((9, m, n), 0.5)
    body = np.zeros((m, n), bool)
    step = float(np.float32(x[1])) - float(np.float32(x[0]))  # spacing as the mesh file holds it
    for k in range(1, 9):
        ti, tj = ii + CX[k], jj + CY[k]
        out = fluid & ~np.roll(fluid, (-CY[k], -CX[k]), (0, 1))
        if kind == "channel":
            t = np.where((tj == 0) | (tj == ny + 1), 1, np.where(ti == 0, 2, 3))
        else:
            t = np.where((tj == ny + 1) & (ti != nx + 1), 2, 1)
        obstacle = out & (ti >= 1) & (ti <= nx) & (tj >= 1) & (tj <= ny)
        t = np.where(obstacle, 1, t)
        bc[k] = np.where(out, t, 0)
        body |= obstacle
        j, i = np.nonzero(out)
        cut = np.full(i.shape, 0.5)
        if centre is not None:
            dx, dy = i - centre[0], j - centre[1]
            a, b = CX[k]**2 + CY[k]**2, 2 * (dx * CX[k] + dy * CY[k])
            root = np.sqrt(np.maximum(b * b - 4 * a * (dx * dx + dy * dy - 0.25 * d * d), 0))
            cut = np.where(obstacle[j, i], np.clip((-b - root) / (2 * a), 1e-3, 1.0), 0.5)
        # through the mesh's single-precision coordinates
        ex = np.float32(x[i] + cut * CX[k] * delta).astype(float) - np.float32(x[i]).astype(float)
        ey = np.float32(y[j] + cut * CY[k] * delta).astype(float) - np.float32(y[j]).astype(float)
        q[k][j, i] = np.hypot(ex, ey) / (step * math.hypot(CX[k], CY[k]))
    some = bc.max(0)
    low = np.where(bc > 0, bc, 99).min(0)
    corner = (some > 0) & (low != some)  # links of different types
    boundary = np.where(corner, 1, some)
    for k, a, b in ((5, 1, 2), (8, 1, 4), (6, 2, 3), (7, 3, 4)):
        bc[k] = np.where(corner & (bc[a] != 0) & (bc[b] != 0), 1, bc[k])
    return fluid, bc, q, boundary, corner, body, np.float32(y).astype(float), step


class Lattice:
    """The same lattice in float64: collide, stream, boundary rules, moments."""

    def __init__(self, fluid, bc, q, boundary, corner, body, uo, om, model, textbook, rho0, dev,
                 curved=False, lam=0.0, s=None, channel=False):
        self.dev, self.model, self.curved = dev, model, curved
        self.m, self.n = fluid.shape
        put = lambda a: torch.as_tensor(a, device=dev)  # noqa: E731
        self.fluid = put(fluid)
        self.at = {}  # flat cells of a rule
        flat = lambda mask: put(np.flatnonzero(mask & fluid))  # noqa: E731
        self.stay = [flat(bc[OPP[k]] != 0) for k in range(9)]
        self.wall = [flat(bc[k] == 1) for k in range(9)]
        self.wall_q = [put(q[k][(bc[k] == 1) & fluid]) for k in range(9)]
        self.lid = flat((boundary == 2) & (bc[2] == 2) & ~corner)
        self.west = flat((boundary == 2) & (bc[3] == 2) & ~corner)
        self.east = flat(bc[1] == 3) if channel else None
        self.body = [flat((bc[k] == 1) & body) for k in range(9)]
        self.uo, self.om = put(uo).double(), put(om).double()
        self.rho0, self.textbook = rho0, textbook
        om_a = 8 * (2 - self.om) / (8 - self.om)
        self.om_a = 1 / (lam / (1 / self.om - 0.5) + 0.5) if lam else om_a
        c = np.array([CX, CY], float)
        e = (c * c).sum(0)
        self.M = put(np.stack([np.ones(9), -4 + 3 * e, 4 - 10.5 * e + 4.5 * e * e, c[0],
                               (-5 + 3 * e) * c[0], c[1], (-5 + 3 * e) * c[1],
                               c[0]**2 - c[1]**2, c[0] * c[1]]))
        self.Minv = torch.linalg.inv(self.M)
        self.s = s

    def equilibrium(self, rho, u, v):
        usq = 1.5 * (u * u + v * v)
        cu = torch.stack([CX[k] * u + CY[k] * v for k in range(9)])
        w = torch.tensor(WEIGHT, dtype=torch.float64, device=self.dev)[:, None]
        return w * rho * (1 + 3 * cu + 4.5 * cu * cu - usq)

    def collide(self, F, rho, u, v):
        if self.model == "bgk":
            M = F + self.om * (self.equilibrium(rho, u, v) - F)
        elif self.model == "trt":
            d = F - self.equilibrium(rho, u, v)
            o = d[list(OPP)]
            M = F - 0.5 * self.om * (d + o) - 0.5 * self.om_a * (d - o)
        else:
            usq = 3 * (u * u + v * v) * (1 if self.textbook else rho)
            eq = torch.stack([rho, rho * (usq - 2), rho * (1 - usq), rho * u, -rho * u, rho * v,
                              -rho * v, rho * (u * u - v * v), rho * u * v])
            d = self.M @ F - eq
            for l, r in enumerate(self.s):
                d[l] *= self.om if r is None else r
            M = F - self.Minv @ d
        return M * self.fluid.reshape(-1)

    def start(self, F, rho, u, v):
        self.M_now = self.collide(F, rho, u, v)
        self.rho, self.u, self.v = rho, u, v

    def step(self):
        M, m, n = self.M_now, self.m, self.n
        F = torch.empty_like(M)
        for k in range(9):
            F[k] = torch.roll(M[k].view(m, n), (CY[k], CX[k]), (0, 1)).reshape(-1)
            F[k, self.stay[k]] = M[k, self.stay[k]]
        uo = self.uo
        if len(self.lid):
            a = self.lid
            r = F[0, a] + F[1, a] + F[3, a] + 2 * (F[2, a] + F[6, a] + F[5, a])
            F[4, a] = F[2, a]
            F[8, a] = F[6, a] + r * uo[a] / 6
            F[7, a] = F[5, a] - r * uo[a] / 6
        if len(self.west):
            a = self.west
            r = (F[0, a] + F[2, a] + F[4, a] + 2 * (F[3, a] + F[6, a] + F[7, a])) / (1 - uo[a])
            F[1, a] = F[3, a] + 2 * r * uo[a] / 3
            F[5, a] = F[7, a] + r * uo[a] / 6
            F[8, a] = F[6, a] + r * uo[a] / 6
        for k in range(1, 9):
            a, o = self.wall[k], OPP[k]
            if not len(a):
                continue
            if self.curved:
                q, mk = self.wall_q[k], M[k, a]
                back = M[k, a - CX[k] - CY[k] * n]
                F[o, a] = torch.where(q < 0.5, 2 * q * mk + (1 - 2 * q) * back,
                                      mk / 2 / q + (2 * q - 1) / (2 * q) * M[o, a])
            else:
                F[o, a] = F[k, a]
        if self.east is not None:
            a = self.east
            ux = F[0, a] + F[2, a] + F[4, a] + 2 * (F[1, a] + F[5, a] + F[8, a]) - 1
            h = 0.5 * (F[2, a] - F[4, a])
            F[3, a] = F[1, a] - 2 * ux / 3
            F[7, a] = F[5, a] + h - ux / 6
            F[6, a] = F[8, a] - h - ux / 6
        live = self.fluid.reshape(-1)
        rho = torch.where(live, F.sum(0), self.rho)
        u = torch.where(live, (F[1] - F[3] + F[5] - F[6] - F[7] + F[8]) / rho, self.u)
        v = torch.where(live, (F[2] - F[4] + F[5] + F[6] - F[7] - F[8]) / rho, self.v)
        if self.east is not None:
            v[self.east] = 0
        self.M_before, self.F = M, F
        self.rho, self.u, self.v = rho, u, v
        self.M_now = self.collide(F, rho, u, v)

    def force(self):
        f = torch.zeros(2, dtype=torch.float64, device=self.dev)
        for k in range(1, 9):
            a = self.body[k]
            if len(a):
                t = (self.M_before[k, a] + self.F[OPP[k], a]).sum()
                f += torch.tensor([CX[k], CY[k]], device=self.dev) * t
        return f


def run_exact(lat, case, rows=()):
    """Steps of the lattice; the residual or force rows of the steps."""
    live = lat.fluid.reshape(-1)
    old = (lat.rho, lat.u, lat.v)
    got = []
    for t in range(1, case["steps"] + 1):
        before = lat.M_now
        lat.step()
        if t % case["every"]:
            continue
        if rows == "force":
            got.append(lat.force().tolist())
        elif rows == "velocity":
            new = (lat.rho, lat.u, lat.v)
            dr, du, dv = ((a - b)[live] for a, b in zip(new, old))
            r, u, v = (a[live] for a in new)
            k = case["every"]
            got.append([float(((du * du + dv * dv).sum() / (u * u + v * v).sum()).sqrt() / k),
                        float(((dr * dr).sum() / (r * r).sum()).sqrt() / k), 0.0, 0.0])
            old = new
        elif rows == "full":
            d = float(((lat.F - before) ** 2)[:, live].sum())
            got.append([math.sqrt(d), math.sqrt(d / live.numel()), 0.0, 0.0])
    return np.array(got, float).reshape(-1, 2 if rows == "force" else 4)


def fields(lat):
    return dict(rho=lat.rho.cpu().numpy(), u=lat.u.cpu().numpy(), v=lat.v.cpu().numpy())


def exact_flow(case, seed):
    f = flow_inputs(case, seed)
    nx, ny = case["nx"], case["ny"]
    is_channel = case["kind"] == "channel"
    n, m = nx + 2, ny + (2 if is_channel else 3)
    if n * m * case["steps"] > 1e10:
        return None
    g = links(case["kind"], nx, ny, n, m, f["rects"], f.get("centre"), case.get("d", 0))
    fluid, bc, y, step = g[0], g[1], g[6], g[7]
    uavg, nu, rho0 = (float(np.float32(f[k])) for k in ("uavg", "nu", "rho"))
    uo = np.full((m, n), uavg)
    if f["inlet"] == 1:
        j = np.nonzero((bc[1:5] == 2).any(0))[0]
        lo, hi = y[j].min() - step / 2, y[j].max() + step / 2
        uo = np.repeat((6 * uavg * (y - lo) * (hi - y) / (hi - lo)**2)[:, None], n, 1)
    om = 1.0 / (3.0 * nu + 0.5)
    plain = not is_channel and case["start"] == "reference"
    dev = device()
    lat = Lattice(*g[:6], uo.ravel(), om, case["model"], not plain, rho0, dev, bool(is_channel),
                  0.0 if plain else 0.25, [1, 1.4, 1.4, 1, 1.2, 1, 1.2, None, None] if plain else
                  [0, 1.4, 1.4, 0, 1.2, 0, 1.2, None, None], is_channel)
    put = lambda a: torch.as_tensor(a, device=dev).double().reshape(-1)  # noqa: E731
    live = put(fluid.astype(float))
    rho, u, v = put(np.full(n * m, rho0)), put(uo), put(np.zeros(n * m))
    if f["field"] is not None:
        rho, u, v = (torch.where(live > 0, put(a), b) for a, b in zip(f["field"], (rho, u, v)))
    elif not plain:
        u = u * (1 - live)
    F = torch.zeros(9, n * m, dtype=torch.float64, device=dev) if plain else \
        lat.equilibrium(rho, u, v)
    lat.start(F * live, rho, u, v)
    kind = "force" if is_channel else case["resid"]
    rows = run_exact(lat, case, kind)
    out = fields(lat)
    if is_channel:
        out["force_at"], out["force"] = None, rows
    elif kind != "none":
        out["resid_at"], out["resid"] = None, None if kind == "reference" else rows
    return out


def exact_sweep(case, seed):
    specs = sweep_inputs(case, seed)
    sizes = [(s["nx"] + 2, s["ny"] + 3) for s in specs]
    # shelves, tallest first
    width = max(max(a for a, _ in sizes), math.ceil(math.sqrt(sum(a * b for a, b in sizes) * 1.15)))
    x = y = shelf = 0
    place = {}
    for k in sorted(range(len(specs)), key=lambda k: -sizes[k][1]):
        if x + sizes[k][0] > width:
            x, y, shelf = 0, y + shelf, 0
        place[k] = (x, y)
        x, shelf = x + sizes[k][0], max(shelf, sizes[k][1])
    n, m = width, y + shelf
    if n * m * case["steps"] > 1e10:
        return None
    whole = [np.zeros((m, n), bool), np.zeros((9, m, n), np.int8), np.full((9, m, n), 0.5),
             np.zeros((m, n), np.int8), np.zeros((m, n), bool), np.zeros((m, n), bool)]
    uo, om = np.full((m, n), float(np.float32(LID))), np.ones((m, n))
    for k, s in enumerate(specs):
        (a, b), (w, h) = place[k], sizes[k]
        one = links("cavity", s["nx"], s["ny"], w, h, s["rects"])
        for to, part in zip(whole, one):
            to[..., b:b + h, a:a + w] = part
        uo[b:b + h, a:a + w] = float(np.float32(s["lid"]))
        om[b:b + h, a:a + w] = 1.0 / (3.0 * float(np.float32(s["nu"])) + 0.5)
    dev = device()
    lat = Lattice(*whole, uo.ravel(), om.ravel(), "mrt", True, 1.0, dev,
                  s=[0, 1.4, 1.4, 0, 1.2, 0, 1.2, None, None])
    live = lat.fluid.reshape(-1).double()
    rho, v = torch.ones_like(live), torch.zeros_like(live)
    u = lat.uo * (1 - live)
    lat.start(lat.equilibrium(rho, u, v) * live, rho, u, v)
    run_exact(lat, case)
    return dict(fields(lat), converged_at=None, resid=None)


def exact_net(case, seed):
    p, x, t = net_inputs(case, seed)
    dev = device()
    p = torch.as_tensor(p, device=dev).double()
    grad = case["task"] == "gradients"
    p.requires_grad_(grad)
    x, t = torch.as_tensor(x, device=dev).double(), torch.as_tensor(t, device=dev).double()
    at = 0

    def conv(v, cout, dil=1):
        nonlocal at
        b, h, w, cin = v.shape
        k = p[at:at + cout * 9 * cin].view(cout, 9, cin)
        at += cout * 9 * cin
        out = p[at:at + cout]
        at += cout
        pad = torch.nn.functional.pad(v, (0, 0, dil, dil, dil, dil))
        for tap in range(9):
            dy, dx = tap // 3 * dil, tap % 3 * dil
            out = out + pad[:, dy:dy + h, dx:dx + w] @ k[:, tap].t()
        return torch.relu(out)

    def halve(v):
        b, h, w, c = v.shape
        v = torch.nn.functional.pad(v, (0, 0, 0, w % 2, 0, h % 2))
        one = torch.nn.functional.pad(torch.ones(h, w, dtype=torch.float64, device=dev),
                                      (0, w % 2, 0, h % 2))
        count = one.view(one.shape[0] // 2, 2, -1, 2).sum((1, 3))
        return v.view(b, one.shape[0] // 2, 2, -1, 2, c).sum((2, 4)) / count[..., None]

    def double(v, h, w):
        return v.repeat_interleave(2, 1).repeat_interleave(2, 2)[:, :h, :w]

    v = torch.nn.functional.pad(x, (0, 32 - x.shape[-1]))
    skip = []
    for l in range(4):
        d = (case["dilation"], 2 * case["dilation"]) if l == 3 else (1, 1)
        v = conv(conv(v, 32 << l, d[0]), 32 << l, d[1])
        skip.append(v)
        if l < 3:
            v = halve(v)
    for l in (2, 1, 0):
        s = skip[l]
        v = torch.cat([s, double(v, *s.shape[1:3])], -1)
        v = conv(conv(v, 32 << l), 32 << l)
    y = v @ p[at:at + 96].view(3, 32).t() + p[at + 96:at + 99]
    if not grad:
        return y.detach().cpu().numpy()
    mask = x[..., :1]
    loss = (mask * (y - t) ** 2).sum() / (3 * mask.sum())
    loss.backward()
    return float(loss), p.grad.cpu().numpy()


def exact(case, seed):
    if case["kind"] == "net":
        return exact_net(case, seed)
    return exact_sweep(case, seed) if case["kind"] == "sweep" else exact_flow(case, seed)
