"""Performance cases: what programs have this framework do, one pass each.

A case names a kind of work and its sizes.  ``prepare`` builds what a program
holds before the call (lattices with a flow in them, networks, input tensors),
``run`` makes one pass through the public entry points and returns the state
and results it leaves, ``work`` gives the bytes and operations such a pass
cannot do without, and ``exact`` the same results in 64-bit torch, written
from the scheme alone.

Kinds:

* ``lattice``: ``Lattice.step``, the FP64/FP32 cavity and periodic solver.
* ``steady``: one block of the steady-state loop, ``CavityStepper.advance`` (a
  replayed graph) and its velocity residual.
* ``deviation``: ``DeviationLattice.step``, FP32/BF16/FP16 storage.
* ``batch``: ``BatchedLattices.run``, the parameter sweep with its amplitude
  samples.
* ``pylb``: the drop-in calls of a driver loop on device tensors.
* ``ghost``: ``GhostLattice.step``, the ghost-layer flows.
* ``unet_forward``, ``unet_train``: the warm start's network.
"""

import math
import random

import numpy as np
import torch

DEVICE = "cuda"
DTYPES = {"f64": torch.float64, "f32": torch.float32}
CX = (0, 1, 0, -1, 0, 1, -1, -1, 1)
CY = (0, 0, 1, 0, -1, 1, 1, -1, -1)
W = (4 / 9,) + (1 / 9,) * 4 + (1 / 36,) * 4
U0 = 0.1  # lid velocity of the cavities
RHO_IN, RHO_OUT = 1.01, 0.99  # inlet and outlet of the canal
# floating-point operations of one BGK lattice update: moments with two
# divisions, nine equilibria, nine relaxations
FLOPS_PER_UPDATE = 120
SIDES = (64, 128, 256, 512, 1024)  # sides of the sweep's instances
WIDTHS, MID, OUT_CH = (32, 64, 128), 128, 3  # the network as it is trained


def listed():
    return [
        # the smallest grid anyone steps: two launches, all latency
        dict(name="cavity_f64_64", kind="lattice", nx=64, ny=64, dtype="f64", bc="cavity", steps=8),
        # time to steady state: blocks of 1000 graph-replayed steps and a
        # residual, at the size of the warm start's held-out cavities
        dict(name="steady_f64_256", kind="steady", n=256, steps=1000),
        # the benchmark's cavity
        dict(name="cavity_f64_2048", kind="lattice", nx=2048, ny=2048, dtype="f64", bc="cavity",
             steps=200),
        # the largest grid in use, far past the last-level cache
        dict(name="cavity_f64_8192", kind="lattice", nx=8192, ny=8192, dtype="f64", bc="cavity",
             steps=20),
        # single precision on a grid whose sides divide by nothing
        dict(name="periodic_f32_1537x1001", kind="lattice", nx=1537, ny=1001, dtype="f32",
             bc="periodic", steps=42),
        # reduced-precision storage in its default 16-bit form
        dict(name="cavity_f16_8192", kind="deviation", nx=8192, ny=8192, fmt="f16", store_every=0,
             bc="cavity", compute="f32", rounding="stochastic", steps=40),
        # the parameter sweep: 512 shear waves of 25 sizes, sampled amplitudes
        dict(name="sweep_512", kind="batch", count=512, steps=100, every=50),
        # a driver script that keeps its array on the GPU: walls, then collide
        dict(name="pylb_f64_2048", kind="pylb", nx=2048, ny=2048, dtype="f64", bc="cavity", steps=10),
        # the sliding-lid script at a size that fills the GPU
        dict(name="lid_f64_4098", kind="ghost", flow="lid", nx=4098, ny=4098, dtype="f64", steps=20),
        # the obstacle-canal script at its own size: launches count
        dict(name="canal_f64_102x52", kind="ghost", flow="canal", nx=102, ny=52, dtype="f64",
             steps=200),
        # one prediction of the warm start
        dict(name="unet_forward_1", kind="unet_forward", batch=1, side=128, in_ch=18),
        # one training step at the batch size it is trained with
        dict(name="unet_train_16", kind="unet_train", batch=16, side=128, in_ch=18),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _steps(rng, nodes, most, budget):
    """Steps of a drawn case: up to ``most``, within ``budget`` lattice updates."""
    return max(1, min(_log_int(rng, max(1, most // 8), most), int(budget // nodes)))


def draw(rng):
    kind = rng.choice(("lattice", "lattice", "lattice", "steady", "deviation", "deviation", "batch",
                       "pylb", "ghost", "ghost", "unet_forward", "unet_train"))
    if kind in ("lattice", "deviation", "pylb", "ghost"):
        nx, ny = _log_int(rng, 64, 6000), _log_int(rng, 64, 6000)
        c = dict(kind=kind, nx=nx, ny=ny)
        if kind == "lattice":
            c.update(dtype=rng.choice(("f64", "f64", "f32")), bc=rng.choice(("cavity", "periodic")),
                     steps=_steps(rng, nx * ny, 200, 8e8))
        elif kind == "deviation":
            c.update(fmt=rng.choice(("f16", "f16", "bf16", "f32")), store_every=rng.choice((0, 0, 1)),
                     bc=rng.choice(("cavity", "periodic")), compute=rng.choice(("f32", "f32", "f64")),
                     rounding="stochastic", steps=_steps(rng, nx * ny, 200, 8e8))
        elif kind == "pylb":
            c.update(dtype=rng.choice(("f64", "f64", "f32")), bc=rng.choice(("cavity", "periodic")),
                     steps=_steps(rng, nx * ny, 20, 2e8))
        else:
            flow = rng.choice(("lid", "canal"))
            c.update(flow=flow, dtype=rng.choice(("f64", "f64", "f32")),
                     steps=_steps(rng, nx * ny, 200, 3e8))
        return c
    if kind == "steady":
        n = _log_int(rng, 64, 1024)
        return dict(kind=kind, n=n, steps=2 * _steps(rng, n * n, 500, 3e8))
    if kind == "batch":
        return dict(kind=kind, count=_log_int(rng, 8, 400), steps=100, every=rng.choice((20, 50, 100)))
    return dict(kind=kind, batch=_log_int(rng, 1, 16), side=8 * rng.randint(8, 16),
                in_ch=6 + 4 * rng.randint(0, 3))


# ---- inputs --------------------------------------------------------------------

def _flow_fields(nx, ny, seed):
    """A smooth FP64 flow: density within 1 % of 1, velocity within 0.06, four modes each."""
    r = random.Random(seed)
    x = torch.arange(nx, dtype=torch.float64, device=DEVICE)[:, None] * (2 * math.pi / nx)
    y = torch.arange(ny, dtype=torch.float64, device=DEVICE)[None, :] * (2 * math.pi / ny)

    def field(amplitude):
        s = torch.zeros((nx, ny), dtype=torch.float64, device=DEVICE)
        for _ in range(4):
            kx, ky, phase = r.randint(1, 6), r.randint(1, 6), r.uniform(0, 2 * math.pi)
            s += amplitude / 4 * r.uniform(0.5, 1) * torch.sin(kx * x + phase) * torch.cos(ky * y + phase)
        return s

    return 1 + field(0.01), field(0.06), field(0.06)


def _omega(seed):
    return random.Random(seed + 77).uniform(0.6, 1.6)


def _instances(count, seed):
    """Shear waves: sides from SIDES (the same for every seed), omega in [0.3, 1.9],
    amplitude in [0.01, 0.1], either direction."""
    sides = _sides(count)
    r = np.random.default_rng(seed)
    return [dict(nx=nx, ny=ny, omega=float(r.uniform(0.3, 1.9)),
                 amplitude=float(r.uniform(0.01, 0.1)), direction="x" if r.random() < 0.5 else "y",
                 bc="periodic") for nx, ny in sides]


def _sides(count):
    r = np.random.default_rng(count)
    return [(int(r.choice(SIDES)), int(r.choice(SIDES))) for _ in range(count)]


def _cavity(n, seed):
    """(Re, U) of a held-out cavity."""
    r = random.Random(seed + 5)
    return 100.0 * 10 ** r.uniform(0, 1), r.uniform(0.05, 0.1)


def _obstacle(nx, ny):
    """A small rectangle in the middle of the canal: (sx, sy, ex, ey)."""
    return nx // 2, ny // 2 - 2, nx // 2 + 3, ny // 2 + 1


def _unet_layers(in_ch):
    """[(name, cin, cout, relu)] of the network."""
    out, c = [], in_ch
    for i, w in enumerate(WIDTHS):
        out += [("enc%da" % i, c, w, True), ("enc%db" % i, w, w, True)]
        c = w
    out += [("mida", c, MID, True), ("midb", MID, MID, True)]
    c = MID
    for i in reversed(range(len(WIDTHS))):
        out += [("dec%da" % i, c + WIDTHS[i], WIDTHS[i], True), ("dec%db" % i, WIDTHS[i], WIDTHS[i], True)]
        c = WIDTHS[i]
    return out + [("head", c, OUT_CH, False)]


def _unet_params(in_ch, seed):
    """Flat FP32 parameters as after some training: He-normal weights, small biases."""
    r = np.random.default_rng(seed)
    parts = []
    for _, cin, cout, _ in _unet_layers(in_ch):
        parts += [r.normal(0, math.sqrt(2 / (9 * cin)), 9 * cin * cout), r.normal(0, 0.05, cout)]
    return np.concatenate(parts).astype(np.float32)


def _unet_data(case, seed):
    """Smooth inputs and targets (as the cells of a flow have), FP32 NHWC."""
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def smooth(channels):
        s = case["side"] // 8
        a = torch.randn(case["batch"], channels, s, s, device=DEVICE, generator=g)
        a = torch.nn.functional.interpolate(a, scale_factor=8, mode="bilinear")
        return a.permute(0, 2, 3, 1).contiguous()

    return smooth(case["in_ch"]), smooth(OUT_CH)


# ---- prepare and run -------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "lattice":
        from latticeboltzmann_amd.lattice import Lattice
        lat = Lattice(case["nx"], case["ny"], _omega(seed), case["bc"], U0, DTYPES[case["dtype"]])
        lat.init_equilibrium(*_flow_fields(case["nx"], case["ny"], seed))
        return dict(case=case, lat=lat)
    if kind == "steady":
        from latticeboltzmann_amd.warmstart.solve import CavityStepper
        re, u = _cavity(case["n"], seed)
        stepper = CavityStepper(case["n"], re, u, every=case["steps"]).__enter__()
        stepper.lat.init_equilibrium(*_flow_fields(case["n"], case["n"], seed))
        stepper.residual()
        return dict(case=case, stepper=stepper)
    if kind == "deviation":
        from latticeboltzmann_amd.precision import DeviationLattice
        lat = DeviationLattice(case["nx"], case["ny"], _omega(seed), case["bc"], U0, fmt=case["fmt"],
                               rounding=case["rounding"], seed=seed, compute=case["compute"],
                               store_every=case["store_every"] or None)
        lat.init_equilibrium(*_flow_fields(case["nx"], case["ny"], seed))
        return dict(case=case, lat=lat)
    if kind == "batch":
        from latticeboltzmann_amd.batch import BatchedLattices
        return dict(case=case, bat=BatchedLattices(_instances(case["count"], seed), fmt="f32", seed=seed))
    if kind == "pylb":
        from latticeboltzmann_amd import PyLB
        dt = DTYPES[case["dtype"]]
        fields = [a.to(dt).reshape(-1).contiguous() for a in _flow_fields(case["nx"], case["ny"], seed)]
        f = torch.empty((9, case["nx"], case["ny"]), dtype=dt, device=DEVICE)
        PyLB.equilibrium(*fields, f.view(9, -1))
        return dict(case=case, f=f, omega=_omega(seed), pylb=PyLB)
    if kind == "ghost":
        from latticeboltzmann_amd import ghost
        nx, ny = case["nx"], case["ny"]
        if case["flow"] == "lid":
            rules, pbc = ghost.cavity_walls(nx, ny, U0), None
        else:
            rules = ghost.side_walls(nx, ny) + ghost.obstacle_faces(*_obstacle(nx, ny))
            pbc = ("after", RHO_IN, RHO_OUT)
        lat = ghost.GhostLattice(nx, ny, _omega(seed), rules, pbc, dtype=DTYPES[case["dtype"]])
        lat.init_equilibrium(*_flow_fields(nx, ny, seed))
        return dict(case=case, lat=lat, moments=lat.moment_buffers())
    from latticeboltzmann_amd.warmstart.network import Surrogate
    net = Surrogate(in_ch=case["in_ch"], widths=WIDTHS, mid=MID, out_ch=OUT_CH)
    net.load_flat(_unet_params(case["in_ch"], seed))
    x, target = _unet_data(case, seed)
    return dict(case=case, net=net, x=x, target=target)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "lattice":
        return state["lat"].step(case["steps"]).f
    if kind == "steady":
        s = state["stepper"]
        s.advance(case["steps"])
        return [s.residual(), s.lat.f]
    if kind == "deviation":
        d = state["lat"].step(case["steps"]).d
        return d.view({"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[case["fmt"]])
    if kind == "batch":
        _, amplitudes = state["bat"].run(case["steps"], sample_every=case["every"])
        return [amplitudes, state["bat"].a]
    if kind == "pylb":
        f, pylb = state["f"], state["pylb"]
        flat = f.view(9, -1)
        for _ in range(case["steps"]):
            if case["bc"] == "cavity":
                pylb.stream_and_bounce_back(f, U0)
            else:
                pylb.stream(f)
            pylb.collide(flat, state["omega"])
        return f
    if kind == "ghost":
        state["lat"].step(case["steps"], moments=state["moments"])
        return [state["lat"].f, list(state["moments"])]
    if kind == "unet_forward":
        return state["net"].forward(state["x"])
    net = state["net"]
    loss = net.train_step(state["x"], state["target"], 1e-4)
    return [loss, net.g, net.p]


def work(case):
    """Bytes of the state read once and written once, operations of every step."""
    kind = case["kind"]
    size = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}
    if kind == "steady":
        n = case["n"] ** 2
        return dict(bytes=n * (2 * 72 + 2 * 16), flops=FLOPS_PER_UPDATE * n * case["steps"])
    if kind == "batch":
        n = sum(nx * ny for nx, ny in _sides(case["count"]))
        return dict(bytes=2 * 36 * n, flops=FLOPS_PER_UPDATE * n * case["steps"])
    if kind.startswith("unet"):
        flops, px, params = 0, case["batch"] * case["side"] ** 2, 0
        for name, cin, cout, _ in _unet_layers(case["in_ch"]):
            level = 0 if name == "head" else int(name[3]) if name[3].isdigit() else len(WIDTHS)
            flops += 2 * 9 * cin * cout * px / 4 ** level
            params += 9 * cin * cout + cout
        io = 4 * px * (case["in_ch"] + OUT_CH)
        if kind == "unet_forward":
            return dict(bytes=io + 2 * params, flops=flops)
        # gradients with respect to weights and activations double the work
        # twice over; Adam reads and writes p, m, v
        return dict(bytes=io + 4 * 7 * params, flops=3 * flops)
    n = case["nx"] * case["ny"]
    if kind == "pylb":
        # each call by itself reads and writes the array
        return dict(bytes=4 * 9 * size[case["dtype"]] * n * case["steps"],
                    flops=FLOPS_PER_UPDATE * n * case["steps"])
    b = 2 * 9 * size[case.get("dtype") or case["fmt"]] * n
    return dict(bytes=b, flops=FLOPS_PER_UPDATE * n * case["steps"])


# ---- the same in 64 bits ---------------------------------------------------------

def _eq(rho, ux, uy):
    uu = 1.5 * (ux * ux + uy * uy)
    out = []
    for i in range(9):
        cu = 3 * (CX[i] * ux + CY[i] * uy)
        out.append(W[i] * rho * (1 + cu + 0.5 * cu * cu - uu))
    return torch.stack(out)


def _moments(f):
    rho = f.sum(0)
    ux = (f[1] - f[3] + f[5] - f[6] - f[7] + f[8]) / rho
    uy = (f[2] - f[4] + f[5] + f[6] - f[7] - f[8]) / rho
    return rho, ux, uy


def _pull(f):
    return torch.stack([torch.roll(f[i], (CX[i], CY[i]), (-2, -1)) for i in range(9)])


def _cavity_stream(f, u0):
    """Streaming with half-way walls at l = 0, k = 0, k = nx-1 and the lid at l = ny-1."""
    g = _pull(f)
    for to, of in ((2, 4), (5, 7), (6, 8)):
        g[to, :, 0] = f[of, :, 0]
    lid = f[6, :, -1] + f[2, :, -1] + f[5, :, -1] + g[6, :, -1] + g[2, :, -1] + g[5, :, -1] \
        + g[3, :, -1] + g[0, :, -1] + g[1, :, -1]
    t = lid * u0 / 6
    g[4, :, -1] = f[2, :, -1]
    g[8, :, -1] = f[6, :, -1] + t
    g[7, :, -1] = f[5, :, -1] - t
    for to, of in ((1, 3), (5, 7), (8, 6)):
        g[to, 0] = f[of, 0]
    for to, of in ((3, 1), (6, 8), (7, 5)):
        g[to, -1] = f[of, -1]
    return g


def _collide(g, omega):
    return g + omega * (_eq(*_moments(g)) - g)


def _evolve(f, omega, bc, u0, steps):
    for _ in range(steps):
        f = _collide(_cavity_stream(f, u0) if bc == "cavity" else _pull(f), omega)
    return f


def _lid_stream(f):
    """The sliding-lid script's streaming: walls one node inside the ghost layers."""
    p = _pull(f)
    g = p.clone()
    for to, of in ((1, 3), (5, 7), (8, 6)):
        g[to, 1, 1:-1] = p[of, 0, 1:-1]
    for to, of in ((3, 1), (6, 8), (7, 5)):
        g[to, -2, 1:-1] = p[of, -1, 1:-1]
    for to, of in ((2, 4), (5, 7), (6, 8)):
        g[to, 1:-1, 1] = p[of, 1:-1, 0]
    top = p[:, 1:-1, -1]
    wall = U0 / 6 * (2 * (top[2] + top[5] + top[6]) + top[0] + top[1] + top[3])
    g[4, 1:-1, -2] = top[2]
    g[7, 1:-1, -2] = top[5] - wall
    g[8, 1:-1, -2] = top[6] + wall
    return g


def _canal_stream(f, obstacle):
    """The obstacle-canal script's streaming: inlet and outlet columns from the
    streamed neighbours, resting walls, a rectangle that bounces back."""
    p = _pull(f)
    inlet = p[:, -2] - _eq(*_moments(p[:, -2]))
    outlet = p[:, 1] - _eq(*_moments(p[:, 1]))
    for col, rho, rest, of in ((0, RHO_IN, inlet, -2), (-1, RHO_OUT, outlet, 1)):
        r, ux, uy = _moments(p[:, of])
        rest = rest + _eq(torch.full_like(r, rho), ux, uy)
        if col == 0:
            first = rest
        else:
            last = rest
    p[:, 0], p[:, -1] = first, last
    g = p.clone()
    sx, sy, ex, ey = obstacle
    for to, of in ((2, 4), (5, 7), (6, 8)):
        g[to, :, 1] = p[of, :, 0]
    for to, of in ((4, 2), (7, 5), (8, 6)):
        g[to, :, -2] = p[of, :, -1]
    for to, of in ((3, 1), (7, 5), (6, 8)):
        g[to, sx - 1, sy:ey] = p[of, sx, sy:ey]
    for to, of in ((1, 3), (5, 7), (6, 8)):
        g[to, ex + 1, sy:ey] = p[of, ex, sy:ey]
    for to, of in ((2, 4), (5, 7), (6, 8)):
        g[to, sx:ex, ey + 1] = p[of, sx:ex, ey]
    for to, of in ((4, 2), (7, 5), (8, 6)):
        g[to, sx:ex, sy - 1] = p[of, sx:ex, sy]
    return g


def _unet(params, in_ch, x):
    """The network in FP64 from flat FP64 parameters; x (B, H, W, in_ch)."""
    pos, spec = 0, {}
    for name, cin, cout, relu in _unet_layers(in_ch):
        n = 9 * cin * cout
        spec[name] = (params[pos:pos + n].view(cout, 9 * cin), params[pos + n:pos + n + cout], relu)
        pos += n + cout

    def conv(name, h):
        wgt, bias, relu = spec[name]
        H, Wd = h.shape[1:3]
        pad = torch.nn.functional.pad(h, (0, 0, 1, 1, 1, 1))
        cols = torch.cat([pad[:, dy:dy + H, dx:dx + Wd] for dy in range(3) for dx in range(3)], dim=-1)
        y = cols.reshape(-1, wgt.shape[1]) @ wgt.t() + bias
        y = y.view(*h.shape[:3], -1)
        return torch.relu(y) if relu else y

    h, skips = x, []
    for i in range(len(WIDTHS)):
        h = conv("enc%db" % i, conv("enc%da" % i, h))
        skips.append(h)
        B, H, Wd, C = h.shape
        h = h.view(B, H // 2, 2, Wd // 2, 2, C).mean(dim=(2, 4))
    h = conv("midb", conv("mida", h))
    for i in reversed(range(len(WIDTHS))):
        h = h.repeat_interleave(2, 1).repeat_interleave(2, 2)
        h = conv("dec%db" % i, conv("dec%da" % i, torch.cat([h, skips[i]], dim=-1)))
    return conv("head", h)


def exact(case, seed):
    kind = case["kind"]
    w = torch.tensor(W, dtype=torch.float64, device=DEVICE)[:, None, None]
    if kind in ("lattice", "pylb", "deviation"):
        dt = DTYPES.get(case.get("dtype"), torch.float64)
        fields = [a.to(dt).double() for a in _flow_fields(case["nx"], case["ny"], seed)]
        f = _evolve(_eq(*fields), _omega(seed), case["bc"], U0, case["steps"])
        if kind == "pylb":
            return f
        if kind == "deviation":
            f = (f - w) * (1024.0 if case["fmt"] == "f16" else 1.0)
        return f.transpose(0, 1).contiguous()
    if kind == "steady":
        re, u = _cavity(case["n"], seed)
        omega = 1 / (3 * u * case["n"] / re + 0.5)
        f0 = _eq(*_flow_fields(case["n"], case["n"], seed))
        f = _evolve(f0, omega, "cavity", u, case["steps"])
        (_, ax, ay), (_, bx, by) = _moments(f0), _moments(f)
        res = float(torch.sqrt((bx - ax) ** 2 + (by - ay) ** 2).max()) / u
        return [res, f.transpose(0, 1).contiguous()]
    if kind == "batch":
        inst = _instances(case["count"], seed)
        amp = np.empty((case["steps"] // case["every"] + 1, len(inst)))
        pool = [None] * len(inst)
        groups = {}
        for i, p in enumerate(inst):
            groups.setdefault((p["nx"], p["ny"]), []).append(i)
        for (nx, ny), ids in groups.items():
            sx = torch.sin(2 * math.pi * torch.arange(nx, dtype=torch.float64, device=DEVICE) / nx)[:, None]
            sy = torch.sin(2 * math.pi * torch.arange(ny, dtype=torch.float64, device=DEVICE) / ny)[None, :]
            for at in range(0, len(ids), 16):  # sixteen of one size at a time
                some = ids[at:at + 16]
                along = torch.tensor([inst[i]["direction"] == "x" for i in some], device=DEVICE)[:, None, None]
                a = torch.tensor([inst[i]["amplitude"] for i in some], dtype=torch.float64, device=DEVICE)
                om = torch.tensor([inst[i]["omega"] for i in some], dtype=torch.float64, device=DEVICE)
                shape = torch.where(along, sy, sx).expand(len(some), nx, ny)
                wave = a[:, None, None] * shape
                f = _eq(torch.ones_like(wave), torch.where(along, wave, 0.0), torch.where(along, 0.0, wave))

                def sample(k):
                    _, ux, uy = _moments(f)
                    v = (torch.where(along, ux, uy) * shape).sum(dim=(1, 2)) * (2 / (nx * ny))
                    amp[k, some] = v.cpu().numpy()

                sample(0)
                for k in range(1, amp.shape[0]):
                    f = _evolve(f, om[:, None, None], "periodic", 0.0, case["every"])
                    sample(k)
                d = (f - w[..., None]).permute(1, 2, 0, 3).float()
                for j, i in enumerate(some):
                    pool[i] = d[j].reshape(-1)
        return [amp, torch.cat(pool)]
    if kind == "ghost":
        dt = DTYPES[case["dtype"]]
        f = _eq(*(a.to(dt).double() for a in _flow_fields(case["nx"], case["ny"], seed)))
        for _ in range(case["steps"]):
            g = _lid_stream(f) if case["flow"] == "lid" else _canal_stream(f, _obstacle(case["nx"], case["ny"]))
            moments = _moments(g)
            f = _collide(g, _omega(seed))
        return [f.transpose(0, 1).contiguous(), list(moments)]
    params = torch.from_numpy(_unet_params(case["in_ch"], seed)).to(DEVICE).double()
    x, target = (a.double() for a in _unet_data(case, seed))
    if kind == "unet_forward":
        return _unet(params, case["in_ch"], x)
    params.requires_grad_(True)
    loss = ((_unet(params, case["in_ch"], x) - target) ** 2).mean()
    loss.backward()
    with torch.no_grad():
        g = params.grad
        # Adam's first step: both moments are the gradient's own
        return [loss.detach().reshape(1), g, params - 1e-4 * g / (g.abs() + 1e-8)]
