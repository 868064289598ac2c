"""What this solver is timed on, and the float64 restatement its results are
held against.

A case is one thing a program does with the library, from arrays in host
memory to arrays in host memory, through the public entry points:

* ``run``: start a simulation from a state, step it, read its fields (the
  headless program, a parameter study, one request of a service);
* ``frame``: one frame of a viewer: step with the pointer's source, then the
  pixels and the path lines it draws;
* ``project``: the projection alone, with the divergence it leaves;
* ``batch``: several simulations of different sizes stepped together.

Sizes are those of the repository's workloads (64x36 to 3840x2160), and
generic ones.  States are a developed flow: smooth swirls of up to about a
cell per step, with noise on top, and smoke that has spread.  Nothing here
reuses a result: every pass of a ``run``, ``project`` or ``batch`` case
uploads its state again; a ``frame`` case goes on from the last frame, as a
viewer does.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from opensayal_amd import Batch, Fluid, Source, default_config

# ---------------------------------------------------------------------------
# cases


def _run(name=None, **kw):
    case = dict(kind="run", width=256, height=144, n=50, steps=1, storage="f32", pressure=False,
                viscosity=0.0, cell_size=1, drain=True, stripes=1, drag=0.0, decay=False,
                tuned=False)
    case.update(kw)
    return dict(case, name=name) if name else case


def _batch(name=None, **kw):
    # 21 members: three fields of each come back
    case = dict(kind="batch", sims=21, least=128, most=1024, multiple=64, f16=False, steps=20,
                spec=2024)
    case.update(kw)
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest grid of the mixes, one synchronous update: an
        # interactive or coupled program that looks at every step; latency
        # and launches are everything
        _run("tiny_update", width=64, height=36, n=20),
        # the plain small wind tunnel, a short run at the default launch shape
        _run("small_run", steps=20),
        # every option a configuration file turns on, on a ragged grid: cell
        # size 2, a closed box, stripes, drag, decay, the pressure field and
        # an odd number of sweeps
        _run("ragged_options", width=397, height=223, n=37, steps=10, pressure=True, cell_size=2,
             drain=False, stripes=3, drag=0.01, decay=True),
        # the projection as an entry point of its own, 16-bit storage, an odd
        # width, with the residual a convergence study reads
        dict(kind="project", name="project_f16", width=1001, height=563, n=100, storage="f16",
             tuned=False),
        # the benchmark's grid: a long run after the autotuner
        _run("full_run", width=1920, height=1080, steps=100, tuned=True),
        # the same grid as the headless program runs it when the file leaves
        # fluid.viscosity out (0.001: the diffusion pass), nothing tuned
        _run("full_viscous", width=1920, height=1080, steps=20, viscosity=0.001),
        # a viewer at the default grid with the pressure shown: pointer held
        # down, one step, pixels and path lines
        dict(kind="frame", name="viewer_frame", width=1920, height=1080, n=50, pressure=True,
             viscosity=0.0, distance=20, length=20),
        # the precision configuration, in 32 and in 16 bits (the largest)
        _run("large_f32", width=3840, height=2160, n=100, steps=10, pressure=True, tuned=True),
        _run("large_bf16", width=3840, height=2160, n=100, steps=10, pressure=True,
             storage="bf16", tuned=True),
        # uneven grids in one batch, as the batched workload draws them
        _batch("batch_mixed"),
        _batch("batch_small", least=64, most=384, multiple=32, steps=50, spec=99),
        # what a service has resident: any width, 32- and 16-bit requests,
        # one chunk of steps
        _batch("batch_serving", sims=12, least=64, most=2048, multiple=1, f16=True, steps=16,
               spec=7),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("run", "run", "run", "frame", "project", "batch"))
    if kind == "batch":
        small = rng.random() < 0.5
        return _batch(sims=rng.randint(4, 21), least=64, most=384 if small else 1024,
                      multiple=rng.choice((1, 32)), f16=rng.random() < 0.5,
                      steps=rng.randint(5, 30), spec=rng.randrange(1 << 20))
    width = _log(rng, 64, 2560)
    height = max(24, min(1440, int(width * rng.uniform(0.4, 1.1))))
    n = rng.choice((20, 37, 50, 75, 100))
    if kind == "project":
        return dict(kind="project", width=width, height=height, n=n,
                    storage=rng.choice(("f32", "f32", "f16", "bf16")), tuned=rng.random() < 0.4)
    if kind == "frame":
        return dict(kind="frame", width=width, height=height, n=n, pressure=rng.random() < 0.5,
                    viscosity=rng.choice((0.0, 0.001)), distance=rng.choice((15, 20)),
                    length=rng.choice((20, 30)))
    return _run(width=width, height=height, n=n, steps=rng.randint(1, 20),
                storage=rng.choice(("f32", "f32", "f16", "bf16")), pressure=rng.random() < 0.4,
                viscosity=rng.choice((0.0, 0.0, 0.001)), cell_size=rng.choice((1, 1, 1, 2)),
                drain=rng.random() < 0.7, stripes=rng.choice((1, 1, 3)),
                drag=rng.choice((0.0, 0.0, 0.01)), decay=rng.random() < 0.3,
                tuned=rng.random() < 0.4)


# ---------------------------------------------------------------------------
# configurations and states


def _options(case):
    """Configuration fields of a single-grid case, over the defaults."""
    W, H = case["width"], case["height"]
    stripes = case.get("stripes", 1)
    pipe = max(H // 4, 8)
    return dict(pipe_height=pipe, obstacle_center_x=W // 2, obstacle_center_y=H // 2,
                obstacle_radius=float(max(3, min(W, H) // 30)), wind_speed=2.0,
                projection_n=case["n"], projection_o=1.9, g=-5.0, d_t=0.05,
                enable_pressure=int(case.get("pressure", False)),
                enable_drain=int(case.get("drain", True)), enable_smoke=1, wind_smoke=1.0,
                smoke_length=1, smoke_count=stripes,
                smoke_height=pipe if stripes == 1 else pipe // (2 * stripes),
                enable_decay=int(case.get("decay", False)), decay_rate=0.05,
                drag_coeff=case.get("drag", 0.0), viscosity=case.get("viscosity", 0.0),
                density=1.0, cell_size=float(case.get("cell_size", 1)),
                storage=case.get("storage", "f32"))


def _members(case):
    """(width, height, options) of a batch case's simulations: widths drawn
    as the batched and serving workloads do, 16:9, obstacle, inflow and sweep
    count uneven."""
    rng = np.random.default_rng(case["spec"])
    out = []
    for k in range(case["sims"]):
        lo, hi = case["least"], case["most"]
        if case["f16"]:
            W = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        else:
            W = int(rng.integers(lo, hi + 1))
        W = max(lo, W // case["multiple"] * case["multiple"])
        H = max(int(round(W * 9 / 16)), 9)
        out.append((W, H, dict(
            pipe_height=max(H // 4, 1), obstacle_center_x=int(rng.uniform(0.2, 0.8) * W),
            obstacle_center_y=int(rng.uniform(0.2, 0.8) * H),
            obstacle_radius=float(np.float32(rng.uniform(0.02, 0.06) * W)),
            wind_speed=float(np.float32(rng.uniform(0.5, 3.0))),
            projection_n=int(rng.choice((20, 50, 100))), projection_o=1.9, g=-5.0, d_t=0.05,
            enable_pressure=0, enable_drain=1, enable_smoke=1, wind_smoke=1.0, smoke_length=1,
            smoke_count=1, smoke_height=H // 4, enable_decay=0, decay_rate=0.05, drag_coeff=0.0,
            viscosity=0.0, density=1.0, cell_size=1.0,
            storage="f16" if case["f16"] and rng.random() < 0.5 else "f32")))
    return out


def _state(W, H, seed):
    """u, v, smoke of a developed flow, (H, W) float32."""
    rng = np.random.default_rng(seed)
    x = np.arange(W, dtype=np.float32)[None, :] * np.float32(2 * math.pi / W)
    y = np.arange(H, dtype=np.float32)[:, None] * np.float32(2 * math.pi / H)
    a, b, c, d = rng.uniform(0.0, 2 * math.pi, 4).astype(np.float32)
    kx, ky = (int(k) for k in rng.integers(1, 5, 2))
    u = np.float32(2.0) + np.float32(9.0) * np.sin(kx * x + a) * np.cos(ky * y + b)
    v = np.float32(9.0) * np.cos(kx * x + c) * np.sin(ky * y + d) - np.float32(4.0)
    u += rng.random((H, W), dtype=np.float32) - np.float32(0.5)
    v += rng.random((H, W), dtype=np.float32) - np.float32(0.5)
    s = np.clip(np.sin(x + b) * np.cos(2 * y + c), 0, None)
    s *= rng.random((H, W), dtype=np.float32)
    return u, v, s.astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "batch":
        batch, members = Batch(), []
        for k, (W, H, opt) in enumerate(_members(case)):
            fl = Fluid(default_config(W, H, **opt))
            batch.add(fl)
            members.append((fl, _state(W, H, (seed, k))))
        return dict(case=case, batch=batch, members=members)
    W, H = case["width"], case["height"]
    fl = Fluid(default_config(W, H, **_options(case)))
    if case.get("tuned") and not fl.autotune_cached():
        fl.autotune()
    u, v, s = _state(W, H, seed)
    state = dict(case=case, fluid=fl, u=u, v=v, smoke=s)
    if case["kind"] == "frame":
        _upload(fl, u, v, s)
        src = Source()
        src.active, src.smoke, src.velocity = 1, 1.0, 0.25
        src.position_x, src.position_y = W // 4, H // 2
        state["source"] = src
    return state


# ---------------------------------------------------------------------------
# one pass


def _upload(fl, u, v, s):
    fl.set_field("vel_x", u)
    fl.set_field("vel_y", v)
    fl.set_field("smoke", s)


def _fields(fl):
    return {name: fl.get_field(name) for name in ("vel_x", "vel_y", "smoke")}


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        for fl, (u, v, s) in state["members"]:
            _upload(fl, u, v, s)
        state["batch"].step(case["steps"])
        return [_fields(fl) for fl, _ in state["members"]]
    fl = state["fluid"]
    if case["kind"] == "frame":
        fl.update(state["source"])
        tx, ty = fl.traces(case["distance"], case["length"])
        return dict(pixels=fl.render_rgba(), traces_x=tx, traces_y=ty)
    if case["kind"] == "project":
        fl.set_field("vel_x", state["u"])
        fl.set_field("vel_y", state["v"])
        fl.project(case["n"])
        l2, most = fl.divergence_norm()
        return dict(vel_x=fl.get_field("vel_x"), vel_y=fl.get_field("vel_y"), l2=l2, most=most)
    _upload(fl, state["u"], state["v"], state["smoke"])
    if case["steps"] == 1:
        fl.update()
    else:
        fl.step(case["steps"])
    out = _fields(fl)
    if case["pressure"]:
        out["pressure"] = fl.get_field("pressure")
        out["least"], out["most"] = fl.pressure_range
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _flops(cells, n, steps, pressure, viscous):
    """Operations of the update rule: a sweep's divergence, quotient and four
    faces (9 per cell, 4 more for the pressure sum), a diffusion round (7),
    the two advections (about 60 and 90)."""
    return cells * steps * (n * (9 + 4 * pressure + 7 * viscous) + 150)


def work(case):
    if case["kind"] == "batch":
        members = _members(case)
        return dict(bytes=sum(24 * W * H for W, H, _ in members),
                    flops=sum(_flops(W * H, opt["projection_n"], case["steps"], 0, 0)
                              for W, H, opt in members))
    cells = case["width"] * case["height"]
    if case["kind"] == "project":
        return dict(bytes=16 * cells, flops=9 * cells * case["n"])
    viscous = int(case["viscosity"] != 0)
    pressure = int(case["pressure"])
    if case["kind"] == "frame":  # the state once in and once out, the pixels
        seeds = (case["width"] // case["distance"]) * (case["height"] // case["distance"])
        elem = 24 + 4 * pressure + 4
        return dict(bytes=elem * cells + 8 * seeds * case["length"],
                    flops=_flops(cells, case["n"], 1, pressure, viscous)
                    + 30 * seeds * case["length"])
    return dict(bytes=(24 + 4 * pressure) * cells,
                flops=_flops(cells, case["n"], case["steps"], pressure, viscous))


# ---------------------------------------------------------------------------
# the update rule in float64 (plain torch): arrays are (H, W) with row j the
# cells (0..W-1, j), j = 0 the bottom


class _Exact:
    def __init__(self, W, H, opt, device):
        self.W, self.H, self.o, self.dev = W, H, opt, device
        self.cs = int(opt["cell_size"])
        f = lambda name: float(np.float32(opt[name]))  # noqa: E731  (a float32 field)
        self.dt, self.over, self.density = f("d_t"), f("projection_o"), f("density")
        self.speed, self.gdt = f("wind_speed"), f("g") * f("d_t")
        self.i = torch.arange(W, device=device)[None, :].expand(H, W)
        self.j = torch.arange(H, device=device)[:, None].expand(H, W)
        i, j = self.i, self.j
        r = f("obstacle_radius")
        dx, dy = i - opt["obstacle_center_x"], j - opt["obstacle_center_y"]
        solid = (i == 0) | (j == 0) | (j == H - 1) | ((dx * dx + dy * dy).double() < r * r)
        if not opt["enable_drain"]:
            solid = solid | (i == W - 1)
        self.fluid = ~solid
        fl = self.fluid.double()
        left, below = torch.zeros_like(fl), torch.zeros_like(fl)
        left[:, 1:] = fl[:, :-1]
        below[1:] = fl[:-1]
        right, above = torch.zeros_like(fl), torch.zeros_like(fl)
        right[:, :-1] = fl[:, 1:]
        above[:-1] = fl[1:]
        self.fu, self.fv = fl * left, fl * below  # faces that move
        count = left + right + below + above
        inner = self.fluid & (i >= 1) & (i <= W - 2) & (j >= 1) & (j <= H - 2)
        share = torch.where(inner & (count > 0), self.over / count.clamp(min=1), 0.0)
        self.share = [torch.where((i + j) % 2 == c, share, 0.0) for c in (0, 1)]

    def project(self, u, v, p=None):
        n, scale = self.o["projection_n"], self.density * self.cs / self.dt
        up = torch.zeros(self.H, self.W + 1, dtype=torch.float64, device=self.dev)
        vp = torch.zeros(self.H + 1, self.W, dtype=torch.float64, device=self.dev)
        up[:, :-1], vp[:-1] = u, v
        fu, fv = torch.zeros_like(up), torch.zeros_like(vp)
        fu[:, :-1], fv[:-1] = self.fu, self.fv
        for _ in range(n):
            for c in (0, 1):
                d = (up[:, 1:] - up[:, :-1]).add_(vp[1:]).sub_(vp[:-1]).mul_(self.share[c])
                if p is not None:
                    p.add_(d, alpha=scale)
                up[:, :-1].addcmul_(fu[:, :-1], d)
                up[:, 1:].addcmul_(fu[:, 1:], d, value=-1)
                vp[:-1].addcmul_(fv[:-1], d)
                vp[1:].addcmul_(fv[1:], d, value=-1)
        return up[:, :-1].contiguous(), vp[:-1].contiguous()

    def inside(self, i, j):
        return (i >= 0) & (i < self.W) & (j >= 0) & (j < self.H)

    def cell(self, x):
        return (x / self.cs).clamp(-(1 << 24), 1 << 24).nan_to_num(nan=-(1 << 24)).trunc().long()

    def read(self, a, i, j):
        """a at (i, j) where that is a fluid cell of the grid, else 0, and
        whether it is."""
        k = j.clamp(0, self.H - 1) * self.W + i.clamp(0, self.W - 1)
        ok = self.inside(i, j) & self.fluid.reshape(-1)[k]
        return torch.where(ok, a.reshape(-1)[k], 0.0), ok

    def sample_u(self, u, x, y):
        cs, i, j = self.cs, self.cell(x), self.cell(y)
        in_x, in_y = x - i * cs, y - j * cs
        low = in_y <= cs / 2
        wx = 1 - in_x / cs
        wy = 1 - torch.where(low, cs / 2 - in_y, in_y - cs / 2) / cs
        jo = torch.where(low, j - 1, j + 1)
        own, ok = self.read(u, i, j)
        acc = wy * wx * own + wy * (1 - wx) * self.read(u, i + 1, j)[0]
        acc += (1 - wy) * wx * self.read(u, i, jo)[0]
        acc += (1 - wy) * (1 - wx) * self.read(u, i + 1, jo)[0]
        return torch.where(ok, acc, 0.0)

    def sample_v(self, v, x, y):
        cs, i, j = self.cs, self.cell(x), self.cell(y)
        in_x, in_y = x - i * cs, y - j * cs
        left = in_x < cs / 2
        wx = 1 - torch.where(left, cs / 2 - in_x, in_x - cs / 2) / cs
        wy = 1 - in_y / cs
        io = torch.where(left, i - 1, i + 1)
        own, ok = self.read(v, i, j)
        acc = wy * wx * own + wy * (1 - wx) * self.read(v, io, j)[0]
        acc += (1 - wy) * (1 - wx) * self.read(v, io, j + 1)[0]
        acc += (1 - wy) * wx * self.read(v, i, j + 1)[0]
        return torch.where(ok, acc, 0.0)

    def sample_smoke(self, s, x, y):
        cs, i, j = self.cs, self.cell(x), self.cell(y)
        i2 = torch.where(x - i * cs < cs / 2, i - 1, i + 1)
        j2 = torch.where(y - j * cs < cs / 2, j - 1, j + 1)
        acc, total = 0.0, 0.0
        for a, b in ((i, j), (i2, j), (i, j2), (i2, j2)):
            w = 1 / (torch.hypot(x - (a + 0.5) * cs, y - (b + 0.5) * cs) + 1e-6)
            total = total + w
            acc = acc + w * self.read(s, a, b)[0]
        return acc / total

    def mean(self, a, others):
        """The mean of a and its neighbours at `others` that are fluid."""
        total, count = a.clone(), torch.ones_like(a)
        for di, dj in others:
            x, ok = self.read(a, self.i + di, self.j + dj)
            total += x
            count += ok
        return total / count

    def step(self, u, v, s):
        """One Fluid::update with an inactive source."""
        o, W, H, cs, dt = self.o, self.W, self.H, self.cs, self.dt
        i, j, pipe = self.i, self.j, o["pipe_height"]
        band = (i <= o["smoke_length"]) & (i != 0) & (j >= H // 2 - pipe // 2) & \
            (j <= H // 2 + pipe // 2)
        u = torch.where(band, self.speed, u)
        tall, many = o["smoke_height"], o["smoke_count"]
        if many == 1:
            inflow = band & (j >= H // 2 - tall // 2) & (j <= H // 2 + tall // 2)
        else:
            gap = int((pipe - many * tall) / (many - 1))
            inflow = band & ((H // 2 + pipe // 2 - j) % (gap + tall) < tall)
        s = torch.where(inflow, float(np.float32(o["wind_smoke"])), s)
        if o["drag_coeff"]:
            damp = math.exp(-float(np.float32(o["drag_coeff"])) * dt)
            u, v = u * damp, v * damp
        v = v + self.gdt
        if o["viscosity"]:
            a = float(np.float32(o["viscosity"])) * dt / (cs * cs)
            for _ in range(o["projection_n"]):
                near = u[1:-1, :-2] + u[1:-1, 2:] + u[:-2, 1:-1] + u[2:, 1:-1]
                nxt = u.clone()
                nxt[1:-1, 1:-1] = (u[1:-1, 1:-1] + a * near) / (1 + 4 * a)
                u = nxt
        p = torch.zeros_like(u) if o["enable_pressure"] else None
        u, v = self.project(u, v, p)
        # the edges
        u[0], u[H - 1] = u[1].clone(), u[H - 2].clone()
        v[1] = 0
        v[:, 0], v[:, W - 1] = v[:, 1].clone(), v[:, W - 2].clone()
        u[:, 1] = 0
        x, y = (i * cs).double(), (j * cs).double()
        cx, cy = (i + 0.5) * cs, (j + 0.5) * cs
        nu = self.sample_u(u, x - u * dt, cy - self.mean(v, ((-1, 1), (0, 1), (-1, 0))) * dt)
        nv = self.sample_v(v, cx - self.mean(u, ((1, 0), (0, -1), (1, -1))) * dt, y - v * dt)
        ns = self.sample_smoke(s, cx - self.sample_u(nu, cx, cy) * dt,
                               cy - self.sample_v(nv, cx, cy) * dt)
        if o["enable_decay"]:
            ns = (ns - float(np.float32(o["decay_rate"])) * dt).clamp(min=0)
        return nu, nv, ns, p


def _seconds(cells, n, steps, viscous):
    """About how long the restatement takes on the GPU."""
    return steps * (2 * n + 2 * n * viscous + 40) * max(9e-5, cells * 1.2e-10)


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def up(a):
        return torch.from_numpy(a).to(dev).double().flip(0)

    def down(a):
        return a.flip(0).cpu().numpy()

    if case["kind"] == "frame":  # pixels and integer path lines
        return None
    if case["kind"] == "batch":
        members = _members(case)
        if sum(_seconds(W * H, opt["projection_n"], case["steps"], 0)
               for W, H, opt in members) > 15:
            return None
        out = []
        for k, (W, H, opt) in enumerate(members):
            e = _Exact(W, H, opt, dev)
            u, v, s = (up(a) for a in _state(W, H, (seed, k)))
            for _ in range(case["steps"]):
                u, v, s, _p = e.step(u, v, s)
            out.append(dict(vel_x=down(u), vel_y=down(v), smoke=down(s)))
        return out
    W, H = case["width"], case["height"]
    if _seconds(W * H, case["n"], case.get("steps", 1), bool(case.get("viscosity"))) > 15:
        return None
    e = _Exact(W, H, _options(case), dev)
    u, v, s = (up(a) for a in _state(W, H, seed))
    if case["kind"] == "project":
        u, v = e.project(u, v)
        div = (u[1:-1, 2:] - u[1:-1, 1:-1] + v[2:, 1:-1] - v[1:-1, 1:-1])
        div = torch.where(e.fluid[1:-1, 1:-1], div, 0.0)
        return dict(vel_x=down(u), vel_y=down(v), l2=float(div.square().sum().sqrt()),
                    most=float(div.abs().max()))
    for _ in range(case["steps"]):
        u, v, s, p = e.step(u, v, s)
    out = dict(vel_x=down(u), vel_y=down(v), smoke=down(s))
    if case["pressure"]:
        out.update(pressure=down(p), least=float(p.min()), most=float(p.max()))
    return out
