"""The workloads this framework's speed is measured on.

Three ways in, as programs use them:

* ``solver``: ``pysweep_amd.Solver`` called on a host array, the reference's
  own way: kernels chosen by the solver, state uploaded, solved, and the
  result brought back to the host.
* ``resident``: a run object of ``pysweep_amd.device`` (``BandRun``,
  ``SweptRun``, ``StandardRun``) whose initial condition and result are GPU
  tensors, for programs that keep their fields on the GPU between solves.
* ``engine``: ``pysweep_amd.batch.Engine`` given a list of problems, for
  batches and served streams.

``listed`` covers the sizes from a single small grid to 8192^2 cells, both
equations, both schemes of the heat plugin, swept and standard
decomposition, FP64 and FP32 state, and the per-cell ``step`` contract that
plugins without an update of their own run on; ``draw`` gives others of the
same ranges.
"""
import math

import numpy
import torch

from pysweep_amd import Solver, batch, device, hip, plugins, schedule
from pysweep_amd.equations import path as eq_path

HEAT, EULER = "heat", "euler"
GAMMA = 1.4
#: floating-point operations of one cell and stage: heat, two second
#: differences with 2*u shared, scaled, summed and added; Euler, the
#: reference device plugin's count (pysweep/equations/euler.cu:22-244)
STAGE_FLOPS = {HEAT: 9, EULER: 626}
NV = {HEAT: 1, EULER: 4}


def listed():
    return [
        # the reference's CPU-runnable heat case: b=8, 100 steps (99 stages after its quantization)
        dict(name="solver_heat_384", via="solver", eq=HEAT, nx=384, ny=384, b=8, its=1, steps=100, swept=True),
        # a small Euler grid through the solver: launches and latency count
        dict(name="solver_euler_128", via="solver", eq=EULER, nx=128, ny=128, b=16, its=2, steps=60, swept=True),
        # an ordinary, non-square Euler grid of the batch's range through the solver
        dict(name="solver_euler_480x352", via="solver", eq=EULER, nx=480, ny=352, b=16, its=2, steps=100, swept=True),
        # a user's plugin with nothing but the per-cell step: the five phase kernels
        dict(name="step_heat_1024", via="resident", run="phases", eq=HEAT, nx=1024, ny=1024, b=32, its=1, steps=300,
             real="double"),
        # midpoint RK2 heat on the study's grid sides (1424 and 1128, no powers of two)
        dict(name="heat_rk2_1424x1128", via="resident", run="band", eq=HEAT, nx=1424, ny=1128, its=2, steps=200,
             real="double"),
        # the headline: Euler vortex 1024^2, swept
        dict(name="euler_1024", via="resident", run="band", eq=EULER, nx=1024, ny=1024, its=2, steps=200,
             real="double"),
        # standard decomposition, a ragged grid
        dict(name="euler_standard_1000x1500", via="resident", run="standard", eq=EULER, nx=1000, ny=1500, its=2,
             steps=100, real="double"),
        # the precision study: Euler 2048^2 with FP32 state, heat 8192^2 with both
        dict(name="euler_2048_fp32", via="resident", run="band", eq=EULER, nx=2048, ny=2048, its=2, steps=100,
             real="float"),
        dict(name="heat_8192", via="resident", run="band", eq=HEAT, nx=8192, ny=8192, its=1, steps=480,
             real="double"),
        dict(name="heat_8192_fp32", via="resident", run="band", eq=HEAT, nx=8192, ny=8192, its=1, steps=240,
             real="float"),
        # batched: mixed heat and Euler problems, sides 64..1024, 200 steps each
        dict(name="engine_mix", via="engine", n=48, lo=64, hi=1024, steps=200, heat=0.5, fp32=0.0, pick=0),
        # a served stream at saturation: Euler, sides 128..1024, uneven step counts, 30 % with FP32 state
        dict(name="engine_stream", via="engine", n=16, lo=128, hi=1024, steps=500, heat=0.0, fp32=0.3, pick=1),
    ]


#: work (flops) no drawn case exceeds
MOST_FLOPS = 4.5e11


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["solver", "solver", "band", "band", "band", "band", "standard", "phases", "engine"])
    if kind == "engine":
        return dict(via="engine", n=rng.randint(4, 24), lo=64, hi=rng.choice([256, 512, 768, 1024]),
                    steps=rng.randint(40, 200), heat=rng.choice([0.0, 0.3, 0.5, 1.0]),
                    fp32=rng.choice([0.0, 0.0, 0.3]), pick=rng.randrange(1 << 20))
    eq = rng.choice([HEAT, EULER])
    its = 2 if eq == EULER else rng.choice([1, 1, 2])
    if kind == "solver":
        b = rng.choice([8, 16, 32]) if eq == HEAT else rng.choice([8, 16, 24])
        top = 1024 if eq == HEAT else 768
        side = lambda: max(2, round(_log(rng, 64, top) / b)) * b  # noqa: E731
        return dict(via="solver", eq=eq, nx=side(), ny=side(), b=b, its=its, steps=rng.randint(30, 150),
                    swept=rng.random() < 0.8)
    top = 8192 if eq == HEAT and kind == "band" else 4096 if eq == HEAT else 2048
    if kind == "phases":
        b = rng.choice([16, 32]) if eq == HEAT else 16
        nx, ny = (max(2, round(_log(rng, 64, 1536) / b)) * b for _ in range(2))
    else:
        b = 0
        nx, ny = (int(_log(rng, 64, top)) for _ in range(2))
    real = "float" if kind != "phases" and its == (2 if eq == EULER else 1) and rng.random() < 0.35 else "double"
    most = MOST_FLOPS / (STAGE_FLOPS[eq] * nx * ny * its)
    case = dict(via="resident", run=kind, eq=eq, nx=nx, ny=ny, its=its,
                steps=max(1, min(int(most), rng.randint(40, 300))), real=real)
    if b:
        case["b"] = b
    return case


# ------------------------------------------------------------------ inputs
def _vortex(nx, ny, eps, xc, yc, dev, L=5.0):
    """Isentropic vortex on [-L, L)^2 (conserved variables), advected with
    (1, 1)."""
    x = torch.arange(nx, dtype=torch.float64, device=dev) * (2 * L / nx) - L - xc
    y = torch.arange(ny, dtype=torch.float64, device=dev) * (2 * L / ny) - L - yc
    x, y = x[:, None], y[None, :]
    minf = math.sqrt(2 / GAMMA)
    om = minf * eps * math.sqrt(2) / 4 / math.pi * math.exp(0.5) * torch.exp(-0.5 * (x * x + y * y))
    dT = -(GAMMA - 1) * om * om / 2
    rho = (1 + dT) ** (1 / (GAMMA - 1))
    u, v = 1.0 - y * om, 1.0 + x * om
    p = (1 + dT) ** (GAMMA / (GAMMA - 1)) / GAMMA
    return torch.stack([rho, rho * u, rho * v, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)])


def _heat_field(nx, ny, kx, ky, amp, noise, seed, dev):
    """amp sin(2 pi kx x) sin(2 pi ky y) plus uniform noise."""
    x = torch.sin(2 * math.pi * kx / nx * torch.arange(nx, dtype=torch.float64, device=dev))
    y = torch.sin(2 * math.pi * ky / ny * torch.arange(ny, dtype=torch.float64, device=dev))
    u = amp * x[:, None] * y[None, :]
    if noise:
        gen = torch.Generator(device=dev).manual_seed(seed)
        u += noise * torch.rand((nx, ny), generator=gen, dtype=torch.float64, device=dev)
    return u[None]


def _field(eq, nx, ny, seed, dev):
    r = numpy.random.default_rng([seed, nx, ny])
    if eq == EULER:
        return _vortex(nx, ny, float(r.uniform(1, 5)), float(r.uniform(-5, 5)), float(r.uniform(-5, 5)), dev)
    return _heat_field(nx, ny, int(r.integers(1, 5)), int(r.integers(1, 5)), float(r.uniform(0.5, 2)), 1e-3, seed, dev)


def _globals(eq, nx, ny, its, steps):
    """[t0, tf, dt, dx, dy, equation args]; tf lies half a step past the last."""
    if eq == EULER:
        dx, dy = 10.0 / nx, 10.0 / ny
        dt = 0.1 * min(dx, dy)
        return [0.0, (steps + 0.5) * dt, dt, dx, dy, GAMMA]
    dx, dy = 1.0 / nx, 1.0 / ny
    dt = 0.1 * dx * dx
    return [0.0, (steps + 0.5) * dt, dt, dx, dy, 1.0, its == 1]


def _stages(case):
    """Stages of a pass: the solver quantizes a swept solve to whole
    pyramids, P = b/(2k) - 1 stages (the reference's createTimeStepData)."""
    n = case["its"] * case["steps"]
    if case["via"] == "solver" and case["swept"]:
        P = case["b"] // (2 if case["eq"] == HEAT else 4) - 1
        return P * (int(n / P - 1) + 1)
    return n


def _requests(case, seed):
    """The problems of an engine case: sizes, precisions and step counts from
    the case, fields from the seed."""
    r = numpy.random.default_rng(case["pick"])
    f = numpy.random.default_rng([seed, 7])
    out = []
    for i in range(case["n"]):
        eq = HEAT if (i + 1) * case["heat"] // 1 > i * case["heat"] // 1 else EULER
        if case["heat"]:  # the batch: sides uniform over the multiples of 32, the same step count
            side = [32 * int(r.integers(case["lo"] // 32, case["hi"] // 32 + 1)) for _ in range(2)]
            steps = case["steps"]
        else:  # the stream: sides log-uniform, step counts uniform
            side = [32 * max(case["lo"] // 32, round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]))) / 32))
                    for _ in range(2)]
            steps = int(r.integers(max(1, case["steps"] // 5), case["steps"] + 1))
        fp32 = bool(r.uniform() < case["fp32"])
        out.append(dict(eq=eq, nx=side[0], ny=side[1], steps=steps, its=2 if eq == EULER else 1, fp32=fp32,
                        eps=float(f.uniform(1, 5)), xc=float(f.uniform(-5, 5)), yc=float(f.uniform(-5, 5)),
                        kx=int(f.integers(1, 5)), ky=int(f.integers(1, 5)), amp=float(f.uniform(0.5, 2))))
    return out


def _request_field(q, dev):
    if q["eq"] == EULER:
        return _vortex(q["nx"], q["ny"], q["eps"], q["xc"], q["yc"], dev)
    return _heat_field(q["nx"], q["ny"], q["kx"], q["ky"], q["amp"], 0.0, 0, dev)


# ------------------------------------------------------------ prepare, run
def prepare(case, seed):
    hip.ensure_init(0)
    if case["via"] == "engine":
        probs = []
        for q in _requests(case, seed):
            probs.append(batch.Problem(q["eq"], _request_field(q, "cuda").cpu().numpy(),
                                       _globals(q["eq"], q["nx"], q["ny"], q["its"], q["steps"]), q["its"],
                                       precision="fp32" if q["fp32"] else "fp64", method="auto"))
        return {"case": case, "problems": probs}
    eq, nx, ny, its = case["eq"], case["nx"], case["ny"], case["its"]
    g = _globals(eq, nx, ny, its, case["steps"])
    field = _field(eq, nx, ny, seed, "cuda")
    if case["via"] == "solver":
        return {"case": case, "globals": g, "ic": field.cpu().numpy()}
    real = case["real"]
    cu = eq_path(eq + (".cu" if real == "double" else "_fp32.cu"))
    nv, ops = NV[eq], 1 if eq == HEAT else 2
    if case["run"] == "band":
        run = device.BandRun(cu, nv, ops, its, nx, ny, real=real)
    elif case["run"] == "standard":
        run = device.StandardRun(cu, nv, ops, its, nx, ny, real=real)
    else:
        run = device.SweptRun(cu, nv, ops, its, nx, ny, case["b"], real=real, generic=True)
    run.set_globals(plugins.load_cpu_module(eq_path(eq + ".py")), g)
    ic = field.to(torch.float64 if real == "double" else torch.float32).contiguous()
    state = {"case": case, "run": run, "ic": ic, "out": torch.empty_like(ic)}
    if case["run"] == "band":
        state["times"] = schedule.standard_times(case["steps"], 16, ops, its)
    elif case["run"] == "phases":
        state["times"] = schedule.swept_times(case["steps"], case["b"], ops, its, exact=True)
    torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    if case["via"] == "engine":
        engine = batch.Engine()
        tickets = [engine.submit(p, arrival=0.0) for p in state["problems"]]
        engine.run()
        return [t.result for t in tickets]
    if case["via"] == "solver":
        solver = Solver(state["ic"], sendWarning=False)
        solver.simulation = case["swept"]
        solver.operating, solver.intermediate = 1 if case["eq"] == HEAT else 2, case["its"]
        solver.blocksize = (case["b"], case["b"], 1)
        solver.globals = list(state["globals"])
        solver.setCPU(eq_path(case["eq"] + ".py"))
        solver.setGPU(eq_path(case["eq"] + ".cu"))
        solver()
        return solver.result
    r, ic, out = state["run"], state["ic"], state["out"]
    for A in range(r.its):  # levels 0 .. s-1 hold the initial condition
        hip.dtod_async(r.ring.ptr + (A % r.T) * r.level_bytes, ic.data_ptr(), r.level_bytes)
    if case["run"] == "standard":
        stages = case["its"] * case["steps"]
        r.run(1, stages + 1)
        last = r.its - 1 + stages
    else:
        last = r.run(state["times"])
    hip.dtod_async(out.data_ptr(), r.ring.ptr + (last % r.T) * r.level_bytes, r.level_bytes)
    return out


# -------------------------------------------------------------------- work
def _work(eq, cells, stages, value_bytes):
    return {"bytes": 2.0 * NV[eq] * cells * value_bytes, "flops": float(STAGE_FLOPS[eq]) * cells * stages}


def work(case):
    if case["via"] == "engine":
        total = {"bytes": 0.0, "flops": 0.0}
        for q in _requests(case, 0):
            w = _work(q["eq"], q["nx"] * q["ny"], q["its"] * q["steps"], 8)  # host arrays are FP64
            total = {k: total[k] + w[k] for k in total}
        return total
    return _work(case["eq"], case["nx"] * case["ny"], _stages(case), 4 if case.get("real") == "float" else 8)


# ------------------------------------------------------------------- exact
def _heat_exact(u, its, g, stages):
    c = g[5] * g[2] / g[3] / g[3]
    q = base = u[0]
    for s in range(1, stages + 1):
        lx = c * (torch.roll(q, -1, 0) - 2 * q + torch.roll(q, 1, 0))
        ly = c * (torch.roll(q, -1, 1) - 2 * q + torch.roll(q, 1, 1))
        d = lx + ly
        if its == 1:
            q = d + q
        else:
            q, base = (d + base if s % 2 == 0 else 0.5 * d + q), q
    return q[None]


def _pressure(q, gm1):
    return gm1 * (q[3] - (q[1] * q[1] + q[2] * q[2]) / (2 * q[0]))


def _limited(q1, q2, num, den):
    pr = num / den
    pr = torch.where(torch.isfinite(pr) & (pr <= 1e6) & (pr >= 0), pr, torch.zeros_like(pr))
    return q1 + torch.clamp(pr, max=1.0) / 2 * (q2 - q1)


def _face(q, p, axis):
    """Flux and dissipation of the face between each cell and its upper
    neighbour along ``axis`` (1 or 2)."""
    gm1 = GAMMA - 1
    up = torch.roll(q, -1, axis)
    pu = torch.roll(p, -1, axis - 1)
    dp = pu - p
    L = _limited(q, up, dp, torch.roll(dp, 1, axis - 1))
    R = _limited(up, q, dp, torch.roll(dp, -1, axis - 1))
    pl, pr = _pressure(L, gm1), _pressure(R, gm1)
    a, o = axis, 3 - axis
    f = [None] * 4
    f[0] = L[a] + R[a]
    f[a] = L[a] * L[a] / L[0] + pl + R[a] * R[a] / R[0] + pr
    f[o] = L[1] * L[2] / L[0] + R[1] * R[2] / R[0]
    f[3] = (L[3] + pl) * L[a] / L[0] + (R[3] + pr) * R[a] / R[0]
    sl, sr = torch.sqrt(L[0]), torch.sqrt(R[0])
    den = 1 / (sl + sr)
    a0 = sl * sr
    m = (sl * (L[1:] / L[0]) + sr * (R[1:] / R[0])) * den
    roe = torch.cat([a0[None], a0 * m])
    rad = torch.sqrt(GAMMA * _pressure(roe, gm1) / a0) + torch.abs(m[a - 1])
    return torch.stack(f), torch.nan_to_num(rad, nan=0.0) * (L - R)


def _divergence(q, p, axis):
    f, d = _face(q, p, axis)
    return ((torch.roll(f, 1, axis) + torch.roll(d, 1, axis)) - f - d) * 0.5


def _euler_exact(q, g, stages):
    k = g[2] / g[3]
    base = q
    for s in range(1, stages + 1):
        p = _pressure(q, GAMMA - 1)
        d = _divergence(q, p, 1) * k + _divergence(q, p, 2) * k
        q, base = (base + d if s % 2 == 0 else q + 0.5 * d), q
    return q


def _solve(eq, field, its, g, stages):
    return _euler_exact(field, g, stages) if eq == EULER else _heat_exact(field, its, g, stages)


def _seconds(eq, cells, stages):
    """About how long ``_solve`` takes on the GPU (measured: launches, then
    memory traffic of about 190 and 12 small operations a stage)."""
    return stages * (4.0e-3 + cells * 2.0e-8 if eq == EULER else 2.5e-4 + cells * 1.0e-10)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["via"] == "engine":
        out, left = [], 12.0
        for q in _requests(case, seed):
            stages = q["its"] * q["steps"]
            left -= _seconds(q["eq"], q["nx"] * q["ny"], stages)
            if left < 0 or q["fp32"]:
                out.append(None)
                continue
            field = _request_field(q, dev)
            out.append(_solve(q["eq"], field, q["its"], _globals(q["eq"], q["nx"], q["ny"], q["its"], q["steps"]),
                              stages).cpu().numpy())
        return out
    eq, nx, ny, its = case["eq"], case["nx"], case["ny"], case["its"]
    stages = _stages(case)
    stages -= stages % its  # the result is the last full step
    if _seconds(eq, nx * ny, stages) > 18:
        return None
    field = _field(eq, nx, ny, seed, dev)
    if case.get("real") == "float":
        field = field.to(torch.float32).to(torch.float64)
    out = _solve(eq, field, its, _globals(eq, nx, ny, its, case["steps"]), stages)
    return out.cpu().numpy() if case["via"] == "solver" else out
