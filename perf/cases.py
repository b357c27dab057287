"""Timed workloads of the shallow-water DG framework, each through its public entry points.

A case is a dict of plain values.  Its "kind" says which call a program makes:

  loop      steps of the device-resident time loop (DeviceIntegrator, captured into a graph),
            then the state in cell order (what a coupled code or an output step reads)
  ensemble  the same loop over several operators of different degree, one launch per stage
            (EnsembleIntegrator)
  ark       one additive (IMEX) step, stage by stage (AdditiveRungeKuttaIntegrator)
  apply     dst = M^-1 L(src) of one state
  monitor   what a time loop asks for between steps: velocity field, CFL speed, mass
  train     one training step of the closure network that also looks at its gradient

Flows: "vortex", a travelling vortex in balance over a flat bed on the periodic domain
[0, 2] x [0, 1]; "channel", [0, 25] x [0, 1] with discharge inflow, fixed outflow level,
walls, Manning friction and a bed with a bump and seeded ripples stored at every quadrature
point.  "split" is the fraction of the cells refined once more (hanging faces).  The mesh
depends on the case alone; initial state, bed, network and samples depend on the seed.

`exact` restates the scheme in plain torch, FP64, without the framework.
"""
import math

import numpy as np
import torch

G = 9.81
WETDRY = 0.1
MANNING = 0.02
DISCHARGE = 4.42
LEVEL = 2.0
SWEEPS = 15

# a + b per scheme: rows of the Butcher tableau, the weights last
RK4 = [[0.5], [0.0, 0.5], [0.0, 0.0, 1.0], [1 / 6, 1 / 3, 1 / 3, 1 / 6]]


# ------------------------------------------------------------------------------ cases
def listed():
    return [
        # latency of a small resident job: the smallest vortex configuration, 12,800 cells
        dict(name="vortex_p1_12k_fp64", kind="loop", flow="vortex", degree=1, nx=160, ny=80,
             split=0.0, precision="fp64", viscosity=0.0, closure=False, steps=5),
        # one coarse channel run (boundary conditions, friction, stored bed), 2,500 cells
        dict(name="channel_p2_2k_fp64", kind="loop", flow="channel", degree=2, nx=250, ny=10,
             split=0.0, precision="fp64", viscosity=0.0, closure=False, steps=5),
        # the same channel coupled to a learned closure, mixed precision
        dict(name="channel_p2_2k_closure", kind="loop", flow="channel", degree=2, nx=250,
             ny=10, split=0.0, precision="mixed", viscosity=0.0, closure=True, steps=5),
        # the headline mesh: degree 3, 30 % of 51,200 cells split, both precisions
        dict(name="vortex_p3_97k_mixed", kind="loop", flow="vortex", degree=3, nx=320, ny=160,
             split=0.3, precision="mixed", viscosity=0.0, closure=False, steps=5),
        dict(name="vortex_p3_97k_fp64", kind="loop", flow="vortex", degree=3, nx=320, ny=160,
             split=0.3, precision="fp64", viscosity=0.0, closure=False, steps=5),
        # a large low-order run, well past the caches
        dict(name="vortex_p1_819k_mixed", kind="loop", flow="vortex", degree=1, nx=1280,
             ny=640, split=0.0, precision="mixed", viscosity=0.0, closure=False, steps=2),
        # horizontal viscosity: the diffusive flux and the velocity update of every step
        dict(name="vortex_p2_51k_viscous", kind="loop", flow="vortex", degree=2, nx=320,
             ny=160, split=0.0, precision="fp64", viscosity=1e-3, closure=False, steps=5),
        # several uneven instances of degree 1 to 4 advanced together
        dict(name="ensemble_p1234_mixed", kind="ensemble", instances=3, cells=6000,
             precision="mixed", steps=2),
        # stiff friction treated implicitly, a refined channel
        dict(name="channel_p2_64k_ark", kind="ark", flow="channel", degree=2, nx=1264, ny=51,
             split=0.0, precision="fp64"),
        # the spatial operator alone, highest degree
        dict(name="apply_p4_25k_fp64", kind="apply", flow="vortex", degree=4, nx=226, ny=113,
             split=0.0, precision="fp64"),
        # between steps: velocity for output, CFL speed, mass check
        dict(name="monitor_p2_102k", kind="monitor", flow="vortex", degree=2, nx=452, ny=226,
             split=0.0, precision="fp64"),
        # closure training at the batch size of the training loop
        dict(name="train_4096", kind="train", rows=4096),
    ]


def draw(rng):
    """another case of the same ranges: 1,000 to about 100,000 cells, every degree, both
    precisions, with and without hanging faces, viscosity and closure"""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["loop", "loop", "loop", "loop", "ensemble", "ark", "apply", "monitor",
                       "train"])
    if kind == "train":
        return dict(kind=kind, rows=spread(500, 20000))
    if kind == "ensemble":
        return dict(kind=kind, instances=rng.randint(1, 3), cells=spread(1000, 8000),
                    precision=rng.choice(["fp64", "mixed"]), steps=rng.randint(1, 3))
    degree = rng.randint(1, 4)
    cells = spread(1000, 160000 / (degree + 1))
    flow = rng.choice(["vortex", "channel"])
    aspect = 2.0 if flow == "vortex" else 25.0
    ny = max(3, int(round(math.sqrt(cells / aspect))))
    nx = max(7, cells // ny)
    case = dict(kind=kind, flow=flow, degree=degree, nx=nx, ny=ny, split=0.0,
                precision=rng.choice(["fp64", "mixed"]))
    if kind == "loop":
        if flow == "vortex" and rng.random() < 0.5:
            case["split"] = round(rng.uniform(0.05, 0.5), 3)
        case.update(viscosity=1e-3 if flow == "vortex" and rng.random() < 0.2 else 0.0,
                    closure=flow == "channel" and degree <= 2 and rng.random() < 0.4,
                    steps=rng.randint(1, 5))
    return case


# ---------------------------------------------------------------------- meshes and flows
class Grid:
    """nx x ny cells on [0, lx] x [0, 1], a fraction of them split in four (at random, fixed
    seed), in the arrays OceanoOperator takes; periodic, or boundary ids 1 (x = 0), 2
    (x = lx), 0 (walls)"""

    def __init__(self, nx, ny, lx, split, periodic):
        hx, hy = lx / nx, 1.0 / ny
        flag = np.zeros(nx * ny, bool)
        n_split = int(round(split * nx * ny))
        flag[np.random.default_rng(20261202).permutation(nx * ny)[:n_split]] = True
        start = np.concatenate([[0], np.cumsum(np.where(flag, 4, 1))])
        self.n_cells = int(start[-1])
        base = np.repeat(np.arange(nx * ny), np.where(flag, 4, 1))
        child = np.arange(self.n_cells) - start[base]
        fine = flag[base]
        scale = np.where(fine, 0.5, 1.0)
        self.geom = np.ascontiguousarray(np.stack(
            [(base % nx + 0.5 * (child % 2)) * hx, (base // nx + 0.5 * (child // 2)) * hy,
             scale * hx, scale * hy], 1))
        faces = []

        def join(a, b, axis):
            """faces between base cells a and b (b on the upper side along `axis`)"""
            fm, fp = 2 * axis + 1, 2 * axis
            lo = [0, 2] if axis == 0 else [0, 1]  # children on the lower side of a cell
            hi = [1, 3] if axis == 0 else [2, 3]
            fa, fb = flag[a], flag[b]
            m = ~fa & ~fb
            faces.append((start[a[m]], fm, -1, start[b[m]], fp, -1))
            for s in range(2):
                m = fa & fb
                faces.append((start[a[m]] + hi[s], fm, -1, start[b[m]] + lo[s], fp, -1))
                m = ~fa & fb
                faces.append((start[a[m]], fm, s, start[b[m]] + lo[s], fp, -1))
                m = fa & ~fb
                faces.append((start[a[m]] + hi[s], fm, -1, start[b[m]], fp, s))

        ij = np.arange(nx * ny)
        i, j = ij % nx, ij // nx
        right, up = (i + 1) % nx + nx * j, i + nx * ((j + 1) % ny)
        join(ij if periodic else ij[i < nx - 1], right if periodic else right[i < nx - 1], 0)
        join(ij if periodic else ij[j < ny - 1], up if periodic else up[j < ny - 1], 1)
        s = start[ij[flag]]
        for a, b, axis in ((0, 1, 0), (2, 3, 0), (0, 2, 1), (1, 3, 1)):
            faces.append((s + a, 2 * axis + 1, -1, s + b, 2 * axis, -1))
        rows = [np.stack([np.broadcast_to(np.asarray(c), np.shape(f[0])) for c in f], 1)
                for f in faces]
        self.inner = np.ascontiguousarray(np.concatenate(rows), np.int32)
        edges = []
        if not periodic:  # the channel, whose cells are not split
            for cells, f, bid in ((ij[i == 0], 0, 1), (ij[i == nx - 1], 1, 2),
                                  (ij[j == 0], 2, 0), (ij[j == ny - 1], 3, 0)):
                edges.append(np.stack([cells, np.full_like(cells, f),
                                       np.full_like(cells, bid)], 1))
        self.boundary = np.ascontiguousarray(
            np.concatenate(edges) if edges else np.zeros((0, 3)), np.int32)


class Union:
    """disjoint union of grids (the instances of one degree of an ensemble)"""

    def __init__(self, grids):
        off = np.concatenate([[0], np.cumsum([g.n_cells for g in grids])])
        self.n_cells = int(off[-1])
        self.geom = np.concatenate([g.geom for g in grids])
        shift = np.array([1, 0, 0, 1, 0, 0])
        self.inner = np.ascontiguousarray(np.concatenate(
            [g.inner + o * shift for g, o in zip(grids, off)]), np.int32)
        self.boundary = np.zeros((0, 3), np.int32)


def _rng(seed):
    return np.random.default_rng([seed, 17])


def _lobatto(n):
    """n Gauss-Lobatto points and weights on [0, 1]"""
    c = np.zeros(n)
    c[-1] = 1.0
    x = np.concatenate([[-1.0], np.sort(np.polynomial.legendre.legroots(
        np.polynomial.legendre.legder(c)).real), [1.0]])
    p = np.polynomial.legendre.legval(x, c)
    return 0.5 * (x + 1.0), 1.0 / (n * (n - 1) * p * p)


def _gauss(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1.0), 0.5 * w


def _basis(n1, x):
    """values and slopes [len(x), n1] of the Lagrange basis on the n1 Gauss-Lobatto nodes"""
    nodes = _lobatto(n1)[0]
    c = np.linalg.inv(np.vander(nodes, increasing=True))  # column i: l_i's coefficients
    V = np.vander(x, n1, increasing=True)
    D = np.zeros_like(V)
    D[:, 1:] = V[:, :-1] * np.arange(1, n1)
    return V @ c, D @ c


def _nodes(geom, n1):
    """node coordinates of every cell, [n_cells, n1 * n1] each"""
    t = _lobatto(n1)[0]
    x = geom[:, :1] + geom[:, 2:3] * np.tile(t, n1)
    y = geom[:, 1:2] + geom[:, 3:4] * np.repeat(t, n1)
    return x, y


def _vortex(rng, geom, n1):
    """a swirl v = V (r/R)(1 - r^2/R^2)^2 in balance with its depression, carried by (1, 0);
    nodal free surface and discharges, cell-major [n_cells, nd], [n_cells, 2, nd]"""
    x, y = _nodes(geom, n1)
    cx, cy = rng.uniform(0.5, 1.5), rng.uniform(0.4, 0.6)
    R, drop = rng.uniform(0.2, 0.35), rng.uniform(0.05, 0.15)
    V = math.sqrt(10.0 * G * drop)
    dx, dy = (x - cx + 1.0) % 2.0 - 1.0, (y - cy + 0.5) % 1.0 - 0.5
    s = np.clip(1.0 - (dx * dx + dy * dy) / (R * R), 0.0, None)
    zeta = 1.0 - drop * s ** 5
    return zeta, np.stack([zeta * (1.0 - V / R * s * s * dy), zeta * (V / R * s * s * dx)], 1)


class Bed:
    """z_b = -b of the channel: a parabolic bump and 5 to 15 ripples"""

    def __init__(self, rng):
        n = int(rng.integers(5, 16))
        self.a = rng.uniform(0.02, 0.05, n)
        self.w = rng.uniform(0.2, 0.5, n)
        self.x = rng.uniform(1.0, 24.0, n)

    def __call__(self, x):
        b = np.where(np.abs(x - 10.0) < 2.0, 0.2 - 0.05 * (x - 10.0) ** 2, 0.0)
        for a, w, c in zip(self.a, self.w, self.x):
            b = b + a * np.exp(-((x - c) / w) ** 2)
        return -b


def _channel(rng, bed, geom, n1):
    x, y = _nodes(geom, n1)
    k, ph = rng.uniform(0.3, 1.0), rng.uniform(0.0, 2 * np.pi)
    zeta = LEVEL + 0.01 * np.sin(k * x + ph) * np.cos(np.pi * y)
    return zeta, np.stack([DISCHARGE + 0.02 * np.cos(k * x + ph),
                           0.01 * np.sin(np.pi * y) * np.sin(k * x)], 1)


def _input(case, seed):
    """mesh, bed (None = flat) and initial state of a case"""
    rng = _rng(seed)
    n1 = case["degree"] + 1
    if case["flow"] == "vortex":
        mesh = Grid(case["nx"], case["ny"], 2.0, case["split"], True)
        return mesh, None, *_vortex(rng, mesh.geom, n1)
    mesh = Grid(case["nx"], case["ny"], 25.0, 0.0, False)
    bed = Bed(rng)
    return mesh, bed, *_channel(rng, bed, mesh.geom, n1)


def _members(case, seed):
    """per degree: mesh of the union and initial state of an ensemble's instances"""
    sizes = np.random.default_rng(case["cells"] + case["instances"])
    rng, out = _rng(seed), []
    for degree in range(1, 5):
        grids = []
        for _ in range(case["instances"]):
            m = max(5, int(round(math.sqrt(case["cells"] * sizes.uniform(0.2, 1.8) / 2))))
            grids.append(Grid(2 * m, m, 2.0, 0.0, True))
        states = [_vortex(rng, g.geom, degree + 1) for g in grids]
        out.append((degree, Union(grids), np.concatenate([s[0] for s in states]),
                    np.concatenate([s[1] for s in states])))
    return out


def _time_step(mesh, degree, bed):
    """CFL 0.15 / (p + 1) on the smallest cell; over a bed 0.075 at degree 2 (the channel's)"""
    speed = math.sqrt(G * (1.0 if bed is None else 2.2)) + (2.0 if bed is None else 2.6)
    h = float(mesh.geom[:, 2:].min())
    return (0.15 if bed is None else 0.225) / (degree + 1) * h / speed


# ------------------------------------------------------------------ the closure network
HID, WIDE = 64, 32


def _network(rng, n_in, n_out):
    """weights of the closure network, [fan_in, fan_out] per layer, with their biases"""
    shape = [n_in, HID, HID, HID, n_out]
    return [(rng.uniform(-1, 1, (a, b)) * math.sqrt(6.0 / (a + b)), 0.1 * rng.normal(size=b))
            for a, b in zip(shape[:-1], shape[1:])]


def _packed(layers):
    """the layers in oc_mlp_set_params' order (32 inputs, 32 outputs, pads zero)"""
    out = []
    for l, (W, b) in enumerate(layers):
        P = np.zeros((WIDE if l == 0 else HID, WIDE if l == 3 else HID))
        P[:W.shape[0], :W.shape[1]] = W
        q = np.zeros(P.shape[1])
        q[:b.size] = b
        out += [P.reshape(-1), q]
    return np.concatenate(out).astype(np.float32)


def _modal(n1):
    """nodal -> modal (orthonormal Legendre) matrix of one direction, on [0, 1]"""
    t = _lobatto(n1)[0]
    V = np.stack([math.sqrt(2 * a + 1) * np.polynomial.legendre.legval(
        2 * t - 1, np.eye(n1)[a]) for a in range(n1)], 1)
    return np.linalg.inv(V)


def _closure(seed, n_cells, degree):
    """a network, its normalisation and the cells' sub-grid statistics"""
    nd = (degree + 1) ** 2
    rng = np.random.default_rng([seed, 23])
    mean = np.concatenate([np.zeros(3 * nd), [-0.025, 5e-4, 0.0]])
    mean[0], mean[nd] = LEVEL, DISCHARGE
    std = np.concatenate([np.full(3 * nd, 0.05), [0.015, 3e-4, 0.6]])
    stats = np.stack([rng.uniform(-0.05, 0.0, n_cells), rng.uniform(1e-5, 1e-3, n_cells),
                      rng.uniform(-1, 1, n_cells)], 1)
    return _network(rng, 3 * nd + 3, 2 * nd), mean, std, np.full(2 * nd, 1e-3), stats


def _samples(case, seed):
    """rows of normalised-scale features and targets of a degree-2 closure"""
    rng = np.random.default_rng([seed, 29])
    X = rng.normal(size=(case["rows"], 30)).astype(np.float32)
    A = rng.normal(size=(30, 18)) / math.sqrt(30)
    T = np.tanh(X @ A) + 0.1 * rng.normal(size=(case["rows"], 18))
    return X, T.astype(np.float32), _network(rng, 30, 18)


# ---------------------------------------------------------------------- prepare and run
def _operator(mesh, degree, bed, zeta, q, precision, viscosity=0.0):
    from oceano_amd.operator import OceanoOperator
    bcs = {} if bed is None else {0: "wall", 1: "discharge_inflow", 2: "height_inflow"}

    def problem_data(xy):
        out = np.zeros((xy.shape[0], 5))
        if bed is not None:
            out[:, 0], out[:, 1] = bed(xy[:, 0]), MANNING
        return out

    op = OceanoOperator(mesh, degree, g=G, threshold_wetdry=WETDRY, viscosity=viscosity,
                        precision=precision, boundary_conditions=bcs)
    op.initialize_data_at_quadrature(problem_data)
    if bed is not None:
        values = np.zeros((op.n_boundary, op.n_q_points_1d, 3))
        values[:, :, 0], values[:, :, 1] = LEVEL, DISCHARGE
        op.set_boundary_values(values)
    return op, op.pack(zeta.reshape(-1), 1), op.pack(q.reshape(-1), 2)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "train":
        from oceano_amd.mlp import ClosureNetwork
        X, T, layers = _samples(case, seed)
        s["net"] = ClosureNetwork(30, 18)
        s["net"].set_params(_packed(layers))
        s["x"], s["t"] = torch.tensor(X, device="cuda"), torch.tensor(T, device="cuda")
        return s
    if kind == "ensemble":
        from oceano_amd.integrator import EnsembleIntegrator
        s["ops"], s["w_h"], s["w_q"], dts = [], [], [], []
        for degree, mesh, zeta, q in _members(case, seed):
            op, h, w = _operator(mesh, degree, None, zeta, q, case["precision"])
            s["ops"].append(op)
            s["w_h"].append(h)
            s["w_q"].append(w)
            dts.append(_time_step(mesh, degree, None))
        s["loop"] = EnsembleIntegrator(s["ops"])
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            s["loop"].capture(dts, s["w_h"], s["w_q"], n_steps=case["steps"])
        return s
    mesh, bed, zeta, q = _input(case, seed)
    op, s["h"], s["q"] = _operator(mesh, case["degree"], bed, zeta, q, case["precision"],
                                   case.get("viscosity", 0.0))
    s["op"], s["dt"] = op, _time_step(mesh, case["degree"], bed)
    if kind == "loop":
        from oceano_amd.integrator import DeviceIntegrator
        if case["closure"]:
            from oceano_amd.mlp import ClosureNetwork
            layers, mean, std, scale, stats = _closure(seed, mesh.n_cells, case["degree"])
            net = ClosureNetwork(mean.size, scale.size)
            net.set_params(_packed(layers))
            net.set_normalization(mean, std, np.zeros(scale.size), scale)
            op.set_subgrid_stats(stats)
            op.set_closure(net)
        vel = op.velocity(s["h"], s["q"]) if case["viscosity"] else None
        s["loop"], s["vel"] = DeviceIntegrator(op), vel
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            s["loop"].capture(s["dt"], s["h"], s["q"], vel, n_steps=case["steps"])
    elif kind == "ark":
        from oceano_amd.integrator import AdditiveRungeKuttaIntegrator
        s["loop"] = AdditiveRungeKuttaIntegrator()
        s["loop"].reinit(op)
    elif kind == "apply":
        s["dst"] = [op.initialize_vector(0), op.initialize_vector(1)]
    return s


def run(s):
    kind = s["kind"]
    if kind == "train":
        loss, grad = s["net"].gradients(s["x"], s["t"])
        s["net"].adam(1e-4)
        return {"loss": loss, "gradient": grad}
    if kind == "ensemble":
        s["loop"].replay(1)
        return [[op.unpack(h, 1), op.unpack(q, 2)]
                for op, h, q in zip(s["ops"], s["w_h"], s["w_q"])]
    op = s["op"]
    if kind == "loop":
        s["loop"].replay(1)
        return [op.unpack(s["h"], 1), op.unpack(s["q"], 2)]
    if kind == "ark":
        s["loop"].perform_time_step(op, 0.0, s["dt"], s["h"], s["q"])
        return [op.unpack(s["h"], 1), op.unpack(s["q"], 2)]
    if kind == "apply":
        op.apply(0.0, [s["h"], s["q"]], s["dst"])
        return [op.unpack(s["dst"][0], 1), op.unpack(s["dst"][1], 2)]
    return {"velocity": op.unpack(op.velocity(s["h"], s["q"]), 2),
            "speed": op.transport_speed(s["h"], s["q"]), "volume": op.volume(s["h"])}


# --------------------------------------------------------------------------------- work
def _stage_flops(degree, viscosity):
    """additions and multiplications of one evaluation of L on one cell, sum-factorised, a
    face counted half to each of its cells, with the depth solve and the inverse mass"""
    n1, nq, ng = degree + 1, (3 * degree) // 2 + 1, degree + 2
    tensor = 2 * (n1 * n1 * nq + n1 * nq * nq)  # one field to (or from) the Gauss points
    cell = 3 * tensor + 2 * tensor + 40 * nq * nq + 2 * 2 * tensor + 2 * tensor
    if viscosity:
        cell += 4 * tensor
    face = 2 * (9 * 2 * n1 * ng + 70 * ng)
    solve = 4 * (n1 * n1 * ng + n1 * ng * ng) + 2 * n1 ** 4
    return cell + face + solve + 2 * 8 * n1 ** 3


def work(case):
    kind = case["kind"]
    if kind == "train":
        n = case["rows"]
        macs = 30 * HID + 2 * HID * HID + HID * 18
        return {"bytes": 4 * n * 48 + 3 * 4 * macs, "flops": 6 * n * macs}
    if kind == "ensemble":
        b = f = 0
        sizes = np.random.default_rng(case["cells"] + case["instances"])
        for degree in range(1, 5):
            for _ in range(case["instances"]):
                m = max(5, int(round(math.sqrt(case["cells"] * sizes.uniform(0.2, 1.8) / 2))))
                b += 2 * 24 * 2 * m * m * (degree + 1) ** 2
                f += 4 * case["steps"] * 2 * m * m * _stage_flops(degree, 0)
        return {"bytes": b, "flops": f}
    n = case["nx"] * case["ny"]
    n += 3 * int(round(case["split"] * n))
    degree = case["degree"]
    nd, nq, ng = (degree + 1) ** 2, (3 * degree) // 2 + 1, degree + 2
    state, geometry = 24 * nd * n, 48 * n
    bed = 8 * n * (nq * nq + ng * ng + 2 * ng) if case["flow"] == "channel" else 0
    flops = n * _stage_flops(degree, case.get("viscosity", 0.0))
    if kind == "loop":
        return {"bytes": 2 * state + geometry + bed, "flops": 4 * case["steps"] * flops}
    if kind == "ark":
        return {"bytes": 2 * state + geometry + bed, "flops": 3 * 1.5 * flops}
    if kind == "apply":
        return {"bytes": 2 * state + geometry + bed, "flops": flops}
    bed = 8 * n * (nd + ng * ng) if case["flow"] == "channel" else 0
    return {"bytes": state + 16 * nd * n + geometry + bed,
            "flops": n * (5 * 4 * nd * (degree + 1) + 4 * 4 * ng * ng * ng + 30 * ng * ng)}


# ----------------------------------------------------------- the scheme in plain FP64
def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a),
                           device="cuda" if torch.cuda.is_available() else "cpu")


def _depth(z, zb):
    return torch.clamp(z + zb, min=1e-12)


def _inv_depth(h):
    h4 = h ** 4
    return math.sqrt(2.0) * h / torch.sqrt(h4 + torch.clamp(h4, min=WETDRY ** 4))


class Scheme:
    """the semi-discrete operator, the depth solve and the steps of one problem; states are
    cell-major: zeta [n, nd], q [n, 2, nd]"""

    def __init__(self, mesh, degree, bed, viscosity=0.0):
        n1 = degree + 1
        self.n1, self.nd, self.nu, self.mesh = n1, n1 * n1, viscosity, mesh
        xq, wq = _gauss((3 * degree) // 2 + 1)
        xg, wg = _lobatto(degree + 2)
        xn, wn = _gauss(n1)
        (Sq, Dq), (Sg, _), (Sn, _) = _basis(n1, xq), _basis(n1, xg), _basis(n1, xn)
        self.Bq, self.Bx, self.By = (_t(np.kron(a, b)) for a, b in
                                     ((Sq, Sq), (Sq, Dq), (Dq, Sq)))
        self.wq2, self.Bg, self.wg2 = _t(np.kron(wq, wq)), _t(np.kron(Sg, Sg)), \
            _t(np.kron(wg, wg))
        self.Bn, self.wn2 = _t(np.kron(Sn, Sn)), _t(np.kron(wn, wn))
        self.Bni = torch.linalg.inv(self.Bn)
        self.minv = torch.linalg.inv(self.Bn.T @ (self.wn2[:, None] * self.Bn))
        self.lump = self.Bg.T @ self.wg2
        self.geom = g = _t(mesh.geom)
        self.hx, self.hy, self.area = g[:, 2:3], g[:, 3:4], g[:, 2:3] * g[:, 3:4]
        flat = bed is None
        self.manning = 0.0 if flat else MANNING

        def at(x1):  # z_b at the tensor points x1 x x1 of every cell
            if flat:
                return 0.0
            x = mesh.geom[:, :1] + mesh.geom[:, 2:3] * np.tile(x1, len(x1))
            return _t(bed(x))

        self.zq, self.zg, self.zn = at(xq), at(xg), at(xn)
        node = np.arange(self.nd).reshape(n1, n1)  # [j][i]
        dofs = [node[:, 0], node[:, -1], node[0, :], node[-1, :]]
        half = [_basis(n1, 0.5 * (xg + s))[0] for s in range(2)]
        self.faces = []
        inner = mesh.inner
        for fm in (1, 3):
            for sm in (-1, 0, 1):
                for sp in (-1, 0, 1):
                    F = inner[(inner[:, 1] == fm) & (inner[:, 2] == sm) & (inner[:, 5] == sp)]
                    if not len(F):
                        continue
                    cm, cp = F[:, 0], F[:, 3]
                    length = mesh.geom[cm, 3 if fm == 1 else 2] * (0.5 if sm >= 0 else 1.0)
                    if flat:
                        zb = 0.0
                    else:
                        x = (mesh.geom[cm, :1] + mesh.geom[cm, 2:3] if fm == 1 else
                             mesh.geom[cm, :1] + mesh.geom[cm, 2:3] * xg)
                        zb = _t(bed(np.broadcast_to(x, (len(F), len(xg)))))
                    self.faces.append((fm, _t(cm).long(), _t(cp).long(), _t(dofs[fm]),
                                       _t(dofs[fm - 1]), _t(Sg if sm < 0 else half[sm]),
                                       _t(Sg if sp < 0 else half[sp]),
                                       _t(length[:, None] * wg), zb))
        self.sides = []
        for f in range(4):
            B = mesh.boundary[mesh.boundary[:, 1] == f]
            if len(B):
                c = B[:, 0]
                x = (mesh.geom[c, :1] + (mesh.geom[c, 2:3] if f == 1 else 0.0) if f < 2 else
                     mesh.geom[c, :1] + mesh.geom[c, 2:3] * xq)
                self.sides.append((f, int(B[0, 2]), _t(c).long(), _t(dofs[f]), _t(Sq),
                                   _t(mesh.geom[c, 3 if f < 2 else 2][:, None] * wq),
                                   _t(bed(np.broadcast_to(x, (len(B), len(xq)))))))

    # fluxes through a face with unit normal along +axis: mass, momentum [.., 2], pressure
    def flux(self, axis, zm, qm, zp, qp, zb):
        out = []
        for z, q in ((zm, qm), (zp, qp)):
            h = _depth(z, zb)
            v = [c * _inv_depth(h) for c in q]
            out.append((h, v, v[axis].abs() + torch.sqrt(G * h),
                        torch.maximum(z, torch.as_tensor(-zb, dtype=z.dtype,
                                                         device=z.device))))
        (hm, vm, lm, cm), (hp, vp, lp, cp) = out
        lam = torch.maximum(lm, lp)
        mass = 0.5 * (hm * vm[axis] + hp * vp[axis]) + 0.5 * lam * (cm - cp)
        um, up = [hm * v for v in vm], [hp * v for v in vp]
        wm, wp = um[axis] * _inv_depth(hm), up[axis] * _inv_depth(hp)
        mom = [0.5 * (a * wm + b * wp) + 0.5 * lam * (a - b) for a, b in zip(um, up)]
        return mass, mom, 0.25 * G * (hm + hp) * (cp - cm)

    def friction(self, h, v):
        return G * self.manning ** 2 / torch.exp(torch.log(h) * 0.33333333333) \
            * torch.sqrt(v[0] ** 2 + v[1] ** 2)

    def integrals(self, zeta, q, vel=None, friction=True):
        """L_zeta, L_q: the cell and face integrals against the basis"""
        qx, qy = q[:, 0], q[:, 1]
        z, ax, ay = zeta @ self.Bq.T, qx @ self.Bq.T, qy @ self.Bq.T
        h = _depth(z, self.zq)
        s = _inv_depth(h)
        v = [ax * s, ay * s]
        JxW = self.wq2 * self.area
        Rz = ((ax * JxW) @ self.Bx) / self.hx + ((ay * JxW) @ self.By) / self.hy
        F = [[ax * v[0], ax * v[1]], [ay * v[0], ay * v[1]]]
        if vel is not None:
            Gr = [[h * (vel[:, e] @ self.Bx.T) / self.hx, h * (vel[:, e] @ self.By.T) / self.hy]
                  for e in range(2)]
            div = Gr[0][0] + Gr[1][1]
            for e in range(2):
                for d in range(2):
                    F[e][d] = F[e][d] - self.nu * (Gr[e][d] + Gr[d][e]) \
                        + (self.nu * div if e == d else 0.0)
        grad = [(zeta @ self.Bx.T) / self.hx, (zeta @ self.By.T) / self.hy]
        Rq = torch.zeros_like(q)
        for e in range(2):
            S = -G * h * grad[e]
            if self.manning and friction:
                S = S - self.friction(h, v) * v[e]
            Rq[:, e] = (S * JxW) @ self.Bq + ((F[e][0] * JxW) @ self.Bx) / self.hx \
                + ((F[e][1] * JxW) @ self.By) / self.hy
        for f, cm, cp, dm, dp, Sm, Sp, JxW, zb in self.faces:
            axis = 0 if f == 1 else 1

            def trace(c, d, S):
                return zeta[c][:, d] @ S.T, [q[c, e][:, d] @ S.T for e in range(2)]

            (zm, qm), (zp, qp) = trace(cm, dm, Sm), trace(cp, dp, Sp)
            mass, mom, pres = self.flux(axis, zm, qm, zp, qp, zb)
            for c, d, S, sign in ((cm, dm, Sm, -1.0), (cp, dp, Sp, 1.0)):
                Rz.index_put_((c[:, None], d[None]), sign * (mass * JxW) @ S, accumulate=True)
                for e in range(2):
                    # the pressure jump is centred: its value is the same seen from each side
                    # up to the sign that the orientation already carries
                    val = sign * mom[e] + (-pres if e == axis else 0.0)
                    Rq[:, e].index_put_((c[:, None], d[None]), (val * JxW) @ S,
                                        accumulate=True)
        for f, bid, c, d, S, JxW, zb in self.sides:
            axis, n = f // 2, (-1.0 if f % 2 == 0 else 1.0)
            z, w = zeta[c][:, d] @ S.T, [q[c, e][:, d] @ S.T for e in range(2)]
            ze, we = z, list(w)
            if bid == 0:
                we[axis] = -w[axis]
            elif bid == 1:
                we = [torch.zeros_like(z), torch.zeros_like(z)]
                we[axis] = torch.full_like(z, -n * DISCHARGE)
            else:
                ze = torch.full_like(z, LEVEL)
            lo, hi = ((z, w), (ze, we)) if n > 0 else ((ze, we), (z, w))
            mass, mom, pres = self.flux(axis, *lo, *hi, zb)
            Rz.index_put_((c[:, None], d[None]), -n * (mass * JxW) @ S, accumulate=True)
            for e in range(2):
                val = -n * mom[e] + (-pres if e == axis else 0.0)
                Rq[:, e].index_put_((c[:, None], d[None]), (val * JxW) @ S, accumulate=True)
        return Rz, Rq

    def apply(self, zeta, q):
        Rz, Rq = self.integrals(zeta, q)
        return (Rz @ self.minv) / self.area, (Rq @ self.minv) / self.area[:, :, None]

    def depth_solve(self, zeta, rhs):
        """the capped lumped Jacobi iteration of M h(zeta') = M h(zeta) + rhs, wet cells"""
        JxW = self.wg2 * self.area
        front = rhs + (_depth(zeta @ self.Bg.T, self.zg) * JxW) @ self.Bg
        z, on = zeta.clone(), torch.ones(len(zeta), dtype=torch.bool, device=zeta.device)
        for _ in range(SWEEPS):
            r = front - (_depth(z @ self.Bg.T, self.zg) * JxW) @ self.Bg
            d = r / (self.lump * self.area) * on[:, None]
            z = z + d
            on = on & (d.abs().sum(1) > 1e-12)
        return z

    def velocity(self, zeta, q):
        s = _inv_depth(_depth(zeta @ self.Bn.T, self.zn))
        return ((q @ self.Bn.T) * s[:, None]) @ self.Bni.T

    def step(self, zeta, q, dt, vel=None, source=None):
        kz, kq, rz, rq = [], [], zeta, q
        for row in RK4:
            Rz, Rq = self.integrals(rz, rq, vel)
            kz.append(Rz)
            kq.append((Rq @ self.minv) / self.area[:, :, None])
            if source is not None:
                kq[-1] = kq[-1] + source(rz, rq)
            rhs = sum(dt * a * k for a, k in zip(row, kz))
            nz = self.depth_solve(zeta, rhs)
            rz, rq = nz, q + sum(dt * a * k for a, k in zip(row, kq))
        return rz, rq

    def ark_step(self, zeta, q, dt):
        """three-stage second-order additive scheme, friction implicit"""
        chi = 2.0 - math.sqrt(2.0)
        b = [0.5 - chi / 4, 0.5 - chi / 4, chi / 2]
        a = [[chi], [0.5, 0.5], b]
        at = [[chi / 2], [0.5 / math.sqrt(2.0)] * 2]
        d = [chi / 2, 1.0 - 1.0 / math.sqrt(2.0)]
        kz, kex, kim, rz, rq = [], [], [], zeta, q
        for s in range(3):
            last = s == 2
            Rz, Rq = self.integrals(rz, rq, friction=last)
            kz.append(Rz)
            kex.append(Rq)
            nz = self.depth_solve(zeta, sum(dt * c * k for c, k in zip(a[s], kz)))
            if last:
                F = dt * b[0] * kex[0] + sum(dt * b[j] * kex[j] + dt * b[j - 1] * kim[j - 1]
                                             for j in (1, 2))
                return nz, q + (F @ self.minv) / self.area[:, :, None]
            h = _depth(rz @ self.Bq.T, self.zq)
            v = [(rq[:, e] @ self.Bq.T) * _inv_depth(h) for e in range(2)]
            JxW = self.wq2 * self.area
            kim.append(torch.stack([(-self.friction(h, v) * v[e] * JxW) @ self.Bq
                                    for e in range(2)], 1))
            W = (self.wn2 * self.area)[:, None]
            F = sum(dt * a[s][j] * kex[j] + dt * at[s][j] * kim[j] for j in range(s + 1)) \
                + ((q @ self.Bn.T) * W) @ self.Bn
            h = _depth(rz @ self.Bn.T, self.zn)
            v = [(rq[:, e] @ self.Bn.T) * _inv_depth(h) for e in range(2)]
            J = G * self.manning ** 2 / torch.exp(torch.log(h) * 1.33333333333) \
                * torch.sqrt(v[0] ** 2 + v[1] ** 2)
            rq = ((F @ self.Bni) / (W * (1.0 + dt * d[s] * J[:, None]))) @ self.Bni.T
            rz = nz


def _forward(layers, x):
    """network output and the pre-activations of its hidden layers"""
    zs = []
    for l, (W, b) in enumerate(layers):
        z = x @ W + b
        if l == 3:
            return z, zs
        zs.append((x, z))
        x = 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0)))


def _tensors(layers):
    return [(_t(W.astype(np.float32).astype(np.float64)),
             _t(b.astype(np.float32).astype(np.float64))) for W, b in layers]


def _gradient(case, seed):
    X, T, layers = _samples(case, seed)
    x, t = _t(X.astype(np.float64)), _t(T.astype(np.float64))
    L = [(W.requires_grad_(), b.requires_grad_()) for W, b in _tensors(layers)]
    loss = ((_forward(L, x)[0] - t) ** 2).mean()
    loss.backward()
    with torch.no_grad():
        grads = [(W.grad.cpu().numpy(), b.grad.cpu().numpy()) for W, b in L]
    out = []
    for l, (W, b) in enumerate(grads):
        P = np.zeros((WIDE if l == 0 else HID, WIDE if l == 3 else HID))
        P[:W.shape[0], :W.shape[1]] = W
        q = np.zeros(P.shape[1])
        q[:b.size] = b
        out += [P.reshape(-1), q]
    return {"loss": float(loss), "gradient": np.concatenate(out)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _gradient(case, seed)
    if kind == "ensemble":
        out = []
        for degree, mesh, zeta, q in _members(case, seed):
            S, z, w = Scheme(mesh, degree, None), _t(zeta), _t(q)
            for _ in range(case["steps"]):
                z, w = S.step(z, w, _time_step(mesh, degree, None))
            out.append([z.reshape(-1), w.reshape(-1)])
        return out
    mesh, bed, zeta, q = _input(case, seed)
    S = Scheme(mesh, case["degree"], bed, case.get("viscosity", 0.0))
    z, w = _t(zeta), _t(q)
    dt = _time_step(mesh, case["degree"], bed)
    if kind == "apply":
        a, b = S.apply(z, w)
        return [a.reshape(-1), b.reshape(-1)]
    if kind == "ark":
        z, w = S.ark_step(z, w, dt)
        return [z.reshape(-1), w.reshape(-1)]
    if kind == "monitor":
        xg = S.Bg
        h = _depth(z @ xg.T, S.zg)
        v = [(w[:, e] @ xg.T) * _inv_depth(h) for e in range(2)]
        # the largest eigenvalue of J^-T J^-1 as the framework's scheme estimates it: five
        # power iterations from (1, 1)
        ij = 1.0 / S.geom[:, 2:]
        e = torch.ones_like(ij)
        for _ in range(5):
            e = ij * ij * e
            e = e / e.abs().amax(1, keepdim=True)
        lam = torch.sqrt(((ij * e) ** 2).sum(1) / (e ** 2).sum(1))
        speed = lam[:, None] * torch.sqrt(G * h) + torch.maximum(
            v[0].abs() * ij[:, :1], v[1].abs() * ij[:, 1:])
        return {"velocity": S.velocity(z, w).reshape(-1), "speed": float(speed.max()),
                "volume": float((h * S.wg2 * S.area).sum())}
    source = None
    if case["closure"]:
        layers, mean, std, scale, stats = _closure(seed, mesh.n_cells, case["degree"])
        L, M = _tensors(layers), _modal(case["degree"] + 1)
        M2 = _t(np.kron(M, M))
        V2 = torch.linalg.inv(M2)

        def source(rz, rq):
            f = torch.cat([rz @ M2.T, rq[:, 0] @ M2.T, rq[:, 1] @ M2.T, _t(stats)], 1)
            y = _forward(L, (f - _t(mean)) / _t(std))[0] * _t(scale)
            return y.reshape(len(rz), 2, -1) @ V2.T
    vel = S.velocity(z, w) if case["viscosity"] else None
    for _ in range(case["steps"]):
        z, w = S.step(z, w, dt, vel, source)
        if vel is not None:
            vel = S.velocity(z, w)
    return [z.reshape(-1), w.reshape(-1)]
