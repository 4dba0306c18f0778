"""The work whose speed counts in this repository: what a program that uses the
solver has it do, over the range of sizes, options and directions in use.

Four paths, each through entry points a program can call:

  substep  a frame of the simulation: the state goes in as host arrays
           (sph_upload_state), a frame's worth of substeps runs (10 at
           dt = 1/300 s is one frame at 30 FPS), the state comes out
           (sph_download_state).  `calls` says how: "fused" sph_step, "staged"
           the reference driver's own sequence of stage calls, "warm" sph_step
           with the trained warm-start network.
  batch    the same for many independent scenes in one context.
  train    Adam steps of the warm-start network, then its weights.
  eval     the network's FP32 forward pass and BF16 inference over rows.
  sort     SortByKey and the cell bounds on device arrays.
  collide  the obstacle push on device arrays.

A pass starts from the same uploaded state every time, so that it can be
repeated.  `exact` restates every path in 64 bits with plain torch.
"""
import ctypes
import functools
import math
import os

import numpy as np
import torch

import sphpc_amd as sa
from sphpc_amd import workloads

DT, GRAVITY, RHO0 = 1.0 / 300.0, 9.81, 1000.0
MAX_NB = 60
NET_FILE = os.path.join(os.path.dirname(sa.__file__), "data", "warm_net_s0.008.bin")
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def substep_case(name, dims, box, spacing, obstacle="none", blocks=1, iterations=4, tolerance=0.0,
                 terms=True, model=1, calls="fused", graph=False, substeps=10):
    return dict(name=name, path="substep", nx=dims[0], ny=dims[1], nz=dims[2], blocks=blocks,
                box_x=box[0], box_y=box[1], box_z=box[2], spacing=spacing, obstacle=obstacle,
                iterations=iterations, tolerance=tolerance, terms=terms, model=model, calls=calls,
                graph=graph, substeps=substeps)


def listed():
    return [
        # the smallest scene in use (the smoke scene): launches and latency are all there is
        substep_case("small_4k", (16, 16, 16), (1.0, 1.0, 1.0), 0.02, iterations=3),
        # the reference's CPU-sized plain dam break, replayed from a graph
        substep_case("dam_32k_graph", (32, 32, 32), (2.0, 1.0, 1.0), 0.02, iterations=3,
                     terms=False, graph=True),
        # the reference driver's call order and its 10 iterations, an odd-sized block
        substep_case("staged_65k", (61, 37, 29), (2.0, 1.0, 1.0), 0.02, iterations=10,
                     calls="staged"),
        # the double dam break at a quarter of its lattice, solved to a tolerance
        substep_case("dams_131k_tol", (64, 32, 32), (6.0, 2.0, 2.0), 0.008, "torus_box", 2,
                     iterations=10, tolerance=1e-3),
        # the held-out 3/8-scale dam break, warm-started by the trained network
        substep_case("dams_442k_warm", (96, 48, 48), (6.0, 2.0, 2.0), 0.008, "torus_box", 2,
                     iterations=10, tolerance=1e-3, calls="warm"),
        # a block of a million particles beside a sphere, replayed from a graph
        substep_case("block_1m_graph", (128, 128, 64), (4.0, 2.0, 2.0), 0.01, "sphere", 1,
                     graph=True),
        # the headline workload: 8,388,608 particles, replayed from a graph
        substep_case("dams_8m_graph", (256, 128, 128), (6.0, 2.0, 2.0), 0.008, "torus_box", 2,
                     graph=True),
        # independent scenes of 2k to 128k particles in one context
        dict(name="batch_96", path="batch", scenes=96, scene_seed=4, n_min=2000, n_max=128000,
             spacing=0.01, iterations=4, substeps=10, graph=True),
        # the trainer's mini-batch, ten steps between two looks at the loss
        dict(name="train_65536", path="train", rows=1000003, batch=65536, steps=10, lr=2e-3),
        # the network over a validation set, in FP32 and as the solver runs it
        dict(name="eval_1m", path="eval", rows=1000003),
        # the native sort and bounds of the reference's boundary, keys of a hash grid
        dict(name="sort_1m", path="sort", pairs=1000003, cells=600000, entry="any"),
        # the obstacle push on the reference's own FP64 arrays
        dict(name="collide_1m_f64", path="collide", points=1000003, wide=True, sdf=128),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["substep"] * 6 + ["batch", "train", "eval", "sort", "collide"])
    if path == "substep":
        n = _spread(rng, 2000, 2500000)
        a, b = rng.uniform(0.6, 2.0), rng.uniform(0.6, 1.6)
        nz = max(4, int(round((n / (a * b)) ** (1.0 / 3.0))))
        nx, ny = max(4, int(round(a * nz))), max(4, int(round(b * nz)))
        spacing = rng.choice([0.008, 0.01, 0.02])
        obstacle = rng.choice(["none", "sphere"])
        box = tuple(round(c * spacing * rng.uniform(1.2, 3.0) + 2.0 * spacing, 3)
                    for c in (nx, ny, nz))
        calls = rng.choice(["fused", "fused", "staged", "warm"])
        tolerance = rng.choice([0.0, 0.0, 1e-3]) if calls != "staged" else 0.0
        substeps = rng.choice([1, 5, 10])
        # the reference's own vorticity formula (model 0) runs away at these spacings
        # within a few substeps
        model = rng.choice([0, 1]) if substeps == 1 else 1
        c = substep_case("", (nx, ny, nz), box, spacing, obstacle, 1, rng.choice([3, 4, 7, 10]),
                         tolerance, rng.random() < 0.8, model, calls,
                         calls == "fused" and rng.random() < 0.5, substeps)
        del c["name"]
        return c
    if path == "batch":
        return dict(path="batch", scenes=_spread(rng, 3, 64), scene_seed=rng.randrange(1000),
                    n_min=2000, n_max=_spread(rng, 8000, 64000), spacing=rng.choice([0.01, 0.02]),
                    iterations=rng.choice([3, 4]), substeps=rng.choice([1, 10]),
                    graph=rng.random() < 0.5)
    if path == "train":
        rows = _spread(rng, 5000, 3000000)
        return dict(path="train", rows=rows, batch=_spread(rng, 100, min(rows, 131072)),
                    steps=rng.choice([1, 10]), lr=2e-3)
    if path == "eval":
        return dict(path="eval", rows=_spread(rng, 100, 4000000))
    if path == "sort":
        pairs = _spread(rng, 1000, 8000000)
        entry = rng.choice(["any", "bits"] + (["noalloc"] if pairs <= 1 << 21 else []))
        return dict(path="sort", pairs=pairs, cells=_spread(rng, 500, 6000000), entry=entry)
    return dict(path="collide", points=_spread(rng, 1000, 8000000), wide=rng.random() < 0.5,
                sdf=rng.choice([64, 100, 128]))


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------
def _params(h, spacing, case):
    terms = int(case.get("terms", True))
    return sa.default_params(h, time_step=DT, g=GRAVITY, k=0.5 * terms, c=0.01 * terms,
                             rest_density=RHO0, rest_mass=RHO0 * spacing ** 3,
                             lambda_epsilon=600.0, vorticity_epsilon=0.01,
                             vorticity_model=case.get("model", 1),
                             solve_iterations=case["iterations"],
                             density_tolerance=case.get("tolerance", 0.0),
                             surface_tension=terms, viscosity=terms, vorticity=terms)


@functools.lru_cache(maxsize=4)
def _obstacle(kind, box, dim):
    """(sdf, dims, spacing, wmin, wmax) of a scene's obstacle, or None."""
    if kind == "none":
        return None
    if kind == "torus_box":  # the double dam break's own obstacle
        dims, wmin, wmax = (dim,) * 3, (2.2, 0.2, 0.0), (3.8, 1.8, 1.6)
        shapes = [sa.torus((3.0, 0.75, 0.12), 0.4, 0.12, axis=2),
                  sa.box_shape((3.0, 1.45, 0.25), (0.25, 0.2, 0.25))]
    else:  # a sphere in the middle of the box, where the block's far edge reaches it
        r = 0.15 * min(box)
        c = tuple(0.5 * b for b in box)
        dims = (dim,) * 3
        wmin, wmax = tuple(v - 1.3 * r for v in c), tuple(v + 1.3 * r for v in c)
        shapes = [sa.sphere(c, r)]
    sdf = sa.sdf_sample_shapes(shapes, dims, wmin, wmax)
    return sdf, dims, (wmax[0] - wmin[0]) / dims[0], wmin, wmax


def _motion(pos, seed):
    """Velocities of a fluid in motion: a smooth flow and a little noise."""
    r = np.random.default_rng([seed, 7])
    vel = r.standard_normal(pos.shape, dtype=np.float32) * np.float32(0.02)
    for a in range(3):
        for b in range(3):
            k, phase = r.uniform(1.0, 4.0), r.uniform(0.0, 6.28)
            vel[:, a] += (0.25 * np.sin(np.float32(k) * pos[:, b] + np.float32(phase))).astype(
                np.float32)
    return vel


def _columns(pos, vel):
    return [np.ascontiguousarray(a[:, i], dtype=np.float32) for a in (pos, vel) for i in range(3)]


def _scene(case, seed):
    s = float(np.float32(case["spacing"]))
    box = (case["box_x"], case["box_y"], case["box_z"])
    d = (case["nx"], case["ny"], case["nz"])
    if case["blocks"] == 2:  # at the two x-ends, centred in y
        y0 = (box[1] - d[1] * s) / 2.0
        blocks = [sa.Block(*d, 0.0, y0, 0.0), sa.Block(*d, box[0] - d[0] * s, y0, 0.0)]
    else:
        blocks = [sa.Block(*d, 0.0, 0.0, 0.0)]
    pos = sa.scene_lattice(blocks, s, jitter=0.02, seed=seed)
    dim = 256 if case["obstacle"] == "torus_box" else 128
    return s, box, pos, _motion(pos, seed), _obstacle(case["obstacle"], box, dim)


@functools.lru_cache(maxsize=2)
def _batch_scenes(count, seed, n_min, n_max, spacing):
    return workloads.batched_scenes(count, seed=seed, spacing=spacing, n_min=n_min, n_max=n_max)


def _batch_state(case, seed):
    s, scenes, pos = _batch_scenes(case["scenes"], case["scene_seed"], case["n_min"],
                                   case["n_max"], case["spacing"])
    r = np.random.default_rng([seed, 3])
    pos = pos + (r.random(pos.shape, dtype=np.float32) - np.float32(0.5)) * np.float32(0.02 * s)
    return s, scenes, np.maximum(pos, np.float32(0.0)), _motion(pos, seed)


# ---------------------------------------------------------------------------
# Network rows, keys and points
# ---------------------------------------------------------------------------
# offsets and deviations of the features as the solver logs them in a dam break
_FEATURE_MEAN = [0.9, 0.0, 0.02, 0.75, 0.0, 3.6, 0.0, 0.0, 0.05, 0.0, 0.0, 0.0]
_FEATURE_STD = [0.12, 0.06, 0.05, 0.1, 0.02, 0.9, 0.15, 0.15, 0.2, 0.05, 0.05, 0.05]


def _rows(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    n = case["rows"]
    x = torch.zeros(n, sa.MLP_STRIDE, device=DEV)
    x[:, :12] = (torch.randn(n, 12, device=DEV, generator=g) *
                 torch.tensor(_FEATURE_STD, device=DEV) + torch.tensor(_FEATURE_MEAN, device=DEV))
    t = (0.8 * x[:, 1] + 0.3 * x[:, 2] - x[:, 4]).clamp_min(0.0) + \
        0.005 * torch.randn(n, device=DEV, generator=g).abs()
    w = torch.zeros(sa.MLP_PARAMS, dtype=torch.float64)
    c = torch.Generator().manual_seed(seed)
    for first, rows, fan in ((0, 12 * 64, 12), (1088, 4096, 64), (5248, 64, 64)):
        w[first:first + rows] = (torch.rand(rows, generator=c) * 2 - 1) * math.sqrt(3.0 / fan)
    mean = (x[:, :12].double().mean(0).float().cpu().numpy(), x[:, :12].double().std(
        0, unbiased=False).float().cpu().numpy(), float(t.mean()), float(t.std()))
    return x, t, w.float().numpy(), mean


def _sort_inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    # particles in the order of an earlier sort: keys near their place, most of them moved
    n, cells = case["pairs"], case["cells"]
    base = torch.arange(n, device=DEV) * cells // n
    moved = torch.randint(-cells // 50 - 2, cells // 50 + 3, (n,), device=DEV, generator=g)
    keys = (base + moved).clamp_(0, cells - 1).to(torch.int32)
    return keys, torch.arange(n, device=DEV, dtype=torch.int32)


def _points(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind = torch.float64 if case["wide"] else torch.float32
    p = torch.rand(3, case["points"], device=DEV, dtype=torch.float64, generator=g)
    return [(p[i] * (2.0 if i == 0 else 1.0)).to(kind) for i in range(3)]


# ---------------------------------------------------------------------------
# The measured passes
# ---------------------------------------------------------------------------
def prepare(case, seed):
    path = case["path"]
    if path == "substep":
        s, box, pos, vel, ob = _scene(case, seed)
        ctx = sa.Context(_params(2.0 * s, s, case), box, len(pos))
        if ob is not None:
            ctx.set_obstacle(*ob)
        state = dict(case=case, ctx=ctx, n=len(pos), columns=_columns(pos, vel))
        if case["calls"] == "warm":
            state["net"] = sa.Mlp()
            state["net"].load(NET_FILE)
            ctx.set_warm_start(state["net"])
        ctx.set_graph(case["graph"])
    elif path == "batch":
        s, scenes, pos, vel = _batch_state(case, seed)
        ctx = sa.BatchContext(_params(2.0 * s, s, case), scenes)
        ctx.set_graph(case["graph"])
        state = dict(case=case, ctx=ctx, n=len(pos), columns=_columns(pos, vel))
    elif path in ("train", "eval"):
        x, t, w, mean = _rows(case, seed)
        net = sa.Mlp()
        net.set_weights(w)
        net.reset_optimizer()
        net.set_normalization(*mean)
        state = dict(case=case, net=net, x=x, t=t, seed=seed)
        if path == "eval":
            state["y"] = torch.empty(case["rows"], device=DEV)
            state["z"] = torch.empty(case["rows"], device=DEV)
        torch.cuda.synchronize()  # the network works on a stream of its own
    elif path == "sort":
        keys, values = _sort_inputs(case, seed)
        cells = case["cells"]
        state = dict(case=case, keys=keys, values=values, k=torch.empty_like(keys),
                     v=torch.empty_like(values),
                     lower=torch.empty(cells, device=DEV, dtype=torch.int32),
                     upper=torch.empty(cells, device=DEV, dtype=torch.int32))
    else:
        pts = _points(case, seed)
        sdf, dims, dx, wmin, wmax = _obstacle("sphere", (2.0, 1.0, 1.0), case["sdf"])
        d = sa.ObstacleDesc(*dims, dx, sa.AABB(wmin[0], wmax[0], wmin[1], wmax[1], wmin[2],
                                               wmax[2]), sdf.ctypes.data)
        handle = ctypes.c_void_p()
        sa.check(sa.lib().sph_sdf_create(ctypes.byref(d), ctypes.byref(handle)))
        state = dict(case=case, points=pts, moved=[torch.empty_like(p) for p in pts],
                     sdf=handle)
    if "columns" in state:
        state["out"] = [np.empty_like(c) for c in state["columns"]]
        state["in_ptrs"] = [sa._fptr(c) for c in state["columns"]]
        state["out_ptrs"] = [sa._fptr(c) for c in state["out"]]
    return state


def _staged_substep(ctx, iterations, terms):
    """The loop body of the reference driver (simulation.c:59-108)."""
    ctx.apply_gravity()
    ctx.predict_positions()
    ctx.find_all_neighbors()
    for it in range(iterations):
        ctx.compute_densities()
        ctx.compute_lambda()
        ctx.update_dps(it)
        ctx.update_position_stars()
    ctx.update_velocities()
    if terms:
        ctx.compute_surface_tension()
        ctx.apply_viscosity()
        ctx.compute_vorticity()
        ctx.apply_vorticity_confinement()
    ctx.update_positions()


def run(state):
    case = state["case"]
    path, L = case["path"], sa.lib()
    if path in ("substep", "batch"):
        ctx = state["ctx"]
        sa.check(L.sph_upload_state(ctx.handle, state["n"], *state["in_ptrs"]))
        if case.get("calls") == "staged":
            for _ in range(case["substeps"]):
                _staged_substep(ctx, case["iterations"], case["terms"])
        else:
            ctx.step(case["substeps"])
        sa.check(L.sph_download_state(ctx.handle, *state["out_ptrs"]))
        return state["out"]
    if path == "train":
        net, x, t = state["net"], state["x"].data_ptr(), state["t"].data_ptr()
        for k in range(case["steps"]):
            loss = ctypes.c_float() if k == case["steps"] - 1 else None
            sa.check(L.sph_mlp_train_step(net.handle, x, t, case["rows"], case["batch"],
                                          case["lr"], state["seed"] * 1000003 + k, loss))
        return {"loss": np.float32(loss.value), "weights": net.weights()}
    if path == "eval":
        net, x = state["net"], state["x"].data_ptr()
        sa.check(L.sph_mlp_forward(net.handle, x, case["rows"], state["y"].data_ptr()))
        sa.check(L.sph_mlp_infer_bf16(net.handle, x, case["rows"], state["z"].data_ptr()))
        return {"fp32": state["y"], "bf16": state["z"]}
    stream = torch.cuda.current_stream().cuda_stream
    if path == "sort":
        k, v, n, cells = state["k"], state["v"], case["pairs"], case["cells"]
        k.copy_(state["keys"])  # the sort is in place
        v.copy_(state["values"])
        if case["entry"] == "any":
            sa.check(L.sph_sort_by_key(k.data_ptr(), v.data_ptr(), n, stream))
        else:
            entry = (L.sph_sort_by_key_bits if case["entry"] == "bits" else
                     L.sph_sort_by_key_bits_noalloc)
            sa.check(entry(k.data_ptr(), v.data_ptr(), n, (cells - 1).bit_length(), stream))
        sa.check(L.sph_find_lower_bounds(k.data_ptr(), n, cells, state["lower"].data_ptr(), stream))
        sa.check(L.sph_find_upper_bounds(k.data_ptr(), n, cells, state["upper"].data_ptr(), stream))
        return {"keys": k, "values": v, "lower": state["lower"], "upper": state["upper"]}
    moved = state["moved"]
    for a, b in zip(moved, state["points"]):  # the push is in place
        a.copy_(b)
    entry = (L.sph_calculate_particle_collisions_f64 if case["wide"] else
             L.sph_calculate_particle_collisions)
    sa.check(entry(*[p.data_ptr() for p in moved], case["points"], state["sdf"], stream))
    return moved


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    path = case["path"]
    if path in ("substep", "batch"):
        if path == "batch":
            n = len(_batch_scenes(case["scenes"], case["scene_seed"], case["n_min"],
                                  case["n_max"], case["spacing"])[2])
        else:
            n = case["nx"] * case["ny"] * case["nz"] * case["blocks"]
        # x and v read and written by each substep, and by the transfers; 29
        # neighbours in the lattice: about 27 operations a pair in density and
        # lambda, 22 in delta p, 120 in the five velocity passes
        pair = 49 * case["iterations"] + (120 if case.get("terms", True) else 0)
        return {"bytes": 48.0 * n * (case["substeps"] + 1),
                "flops": 29.0 * n * pair * case["substeps"]}
    if path == "train":
        rows = case["batch"] * case["steps"]
        return {"bytes": rows * 52.0 + case["steps"] * 7.0 * 4 * sa.MLP_PARAMS,
                "flops": rows * 6.0 * (12 * 64 + 64 * 64 + 64)}
    if path == "eval":
        return {"bytes": case["rows"] * (48.0 + 8.0),
                "flops": case["rows"] * 4.0 * (12 * 64 + 64 * 64 + 64)}
    if path == "sort":
        return {"bytes": 24.0 * case["pairs"] + 8.0 * case["cells"], "flops": 0.0}
    size = 8.0 if case["wide"] else 4.0
    return {"bytes": 12.0 * size * case["points"] + 4.0 * case["sdf"] ** 3, "flops": 0.0}


# ---------------------------------------------------------------------------
# 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    path = case["path"]
    if path == "substep":
        # the warm-started solve is accepted or taken back by a test on values of
        # a BF16 network: it has no value in 64 bits
        if case["calls"] == "warm":
            return None
        s, box, pos, vel, ob = _scene(case, seed)
        return _exact_frame(case, s, [box], [len(pos)], [ob], pos, vel)
    if path == "batch":
        s, scenes, pos, vel = _batch_state(case, seed)
        grids = [(o["sdf"], o["dims"], o["spacing"], o["wmin"], o["wmax"]) if o else None
                 for o in (sc["sdf"] for sc in scenes)]
        return _exact_frame(case, s, [sc["size"] for sc in scenes],
                            [sc["particles"] for sc in scenes], grids, pos, vel)
    if path in ("train", "eval"):
        x, t, w, mean = _rows(case, seed)
        return _exact_train(case, seed, x, t, w, mean) if path == "train" else \
            _exact_eval(x, w, mean)
    if path == "sort":
        return None  # whole numbers
    sdf, dims, dx, wmin, wmax = _obstacle("sphere", (2.0, 1.0, 1.0), case["sdf"])
    p = torch.stack([q.double() for q in _points(case, seed)], 1)
    grid = _Grids([(sdf, dims, dx, wmin, wmax)], p.device)
    out = grid.push(p, torch.zeros(len(p), dtype=torch.long, device=p.device))
    return [out[:, i].contiguous().to(torch.float64) for i in range(3)]


class _Grids:
    """Obstacle grids of the scenes (all of one size; None: no obstacle)."""

    def __init__(self, grids, device):
        some = next((g for g in grids if g is not None), None)
        self.any = some is not None
        if not self.any:
            return
        none = (np.ones_like(some[0]), some[1], 1.0, (1e30,) * 3, (2e30,) * 3)
        full = [g if g is not None else none for g in grids]
        self.dims = some[1]
        self.data = torch.from_numpy(np.stack([g[0].ravel() for g in full])).to(device).double()
        self.lo = torch.tensor([g[3] for g in full], device=device, dtype=torch.float64)
        self.hi = torch.tensor([g[4] for g in full], device=device, dtype=torch.float64)
        self.texel = torch.tensor([g[2] for g in full], device=device, dtype=torch.float64)

    def sample(self, scene, u):
        """Trilinear, texel centres at (i + 1/2) / dim, clamped at the edges."""
        nx, ny, nz = self.dims
        c = u * torch.tensor(self.dims, device=u.device, dtype=torch.float64) - 0.5
        f = torch.floor(c)
        a, i = c - f, f.long()
        total = 0.0
        for corner in range(8):
            at, wgt = [], 1.0
            for ax, dim in enumerate((nx, ny, nz)):
                up = corner >> ax & 1
                at.append((i[:, ax] + up).clamp(0, dim - 1))
                wgt = wgt * (a[:, ax] if up else 1.0 - a[:, ax])
            total = total + wgt * self.data[scene, at[0] + nx * (at[1] + ny * at[2])]
        return total

    def push(self, p, scene):
        if not self.any:
            return p
        inside = ((p > self.lo[scene]) & (p < self.hi[scene])).all(1).nonzero()[:, 0]
        if not len(inside):
            return p
        q, sc = p[inside], scene[inside]
        span = self.hi[sc] - self.lo[sc]
        u = (q - self.lo[sc]) / span
        d = self.sample(sc, u)
        grad = []
        for ax in range(3):
            e = torch.zeros(3, device=p.device, dtype=torch.float64)
            e[ax] = 1.0 / self.dims[ax]
            grad.append(self.sample(sc, u + e) - self.sample(sc, u - e))
        grad = torch.stack(grad, 1)
        norm = grad.square().sum(1).sqrt()
        move = (d < 0) & (norm > 0)
        scale = span[:, 0] / (self.dims[0] * self.texel[sc])
        step = (d.abs() * scale / norm.clamp_min(1e-300))[:, None] * grad
        out = p.clone()
        out[inside] = torch.where(move[:, None], q + step, q)
        return out


def _pairs(xs, key, key_id, base, dims, h, rows=1 << 18):
    """Neighbour pairs (i, j) in cell order: the first 60 of each particle within
    h, rows of three cells by (dz, dy), then (cell, id)."""
    dev, n = xs.device, len(xs)
    cells = int((base + dims[:, 0] * dims[:, 1] * dims[:, 2]).max()) + 1
    start = torch.searchsorted(key, torch.arange(cells + 1, device=dev))
    rel = key - base
    nx, ny, nz = dims[:, 0], dims[:, 1], dims[:, 2]
    cz = rel // (nx * ny)
    cy = (rel - cz * nx * ny) // nx
    cx = rel % nx
    out_i, out_j = [], []
    for first in range(0, n, rows):
        sl = slice(first, min(first + rows, n))
        me = torch.arange(sl.start, sl.stop, device=dev)
        bx, by, bz = nx[sl], ny[sl], nz[sl]
        part_i, part_j = [], []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                z, y = cz[sl] + dz, cy[sl] + dy
                ok = (z >= 0) & (z < bz) & (y >= 0) & (y < by)
                row = base[sl] + (z * by + y) * bx
                row = torch.where(ok, row, base[sl])
                lo = start[row + (cx[sl] - 1).clamp_min(0)]
                hi = start[row + torch.minimum(cx[sl] + 1, bx - 1) + 1]
                cnt = torch.where(ok, hi - lo, torch.zeros_like(lo))
                i = torch.repeat_interleave(me, cnt)
                j = torch.arange(len(i), device=dev) + torch.repeat_interleave(
                    lo - torch.cumsum(cnt, 0) + cnt, cnt)
                hit = ((xs[i] - xs[j]).square().sum(1) < h * h) & (i != j)
                part_i.append(i[hit])
                part_j.append(j[hit])
        i, j = torch.cat(part_i), torch.cat(part_j)
        order = torch.argsort(i, stable=True)
        i, j = i[order], j[order]
        rank = torch.arange(len(i), device=dev) - torch.searchsorted(i, i)
        out_i.append(i[rank < MAX_NB])
        out_j.append(j[rank < MAX_NB])
    return torch.cat(out_i), torch.cat(out_j)


def _exact_frame(case, s, boxes, counts, grids, pos, vel):
    n = len(pos)
    if n * case["substeps"] > 40000000:
        return None  # minutes of 64-bit arithmetic
    f64 = dict(device=DEV, dtype=torch.float64)
    h = 2.0 * s
    p = _params(h, s, case)
    mass, iters, tol = p.rest_mass, case["iterations"], case.get("tolerance", 0.0)
    terms, model = case.get("terms", True), case.get("model", 1)
    scene = torch.repeat_interleave(torch.arange(len(boxes), device=DEV),
                                    torch.tensor(counts, device=DEV))
    size = torch.tensor(boxes, **f64)
    dims_s = torch.ceil(size / h).long() + 1
    base_s = torch.cumsum(dims_s.prod(1), 0) - dims_s.prod(1)
    grid = _Grids(grids, torch.device(DEV))
    x = torch.from_numpy(np.ascontiguousarray(pos)).to(**f64)
    v = torch.from_numpy(np.ascontiguousarray(vel)).to(**f64)
    w_norm = 315.0 / (64.0 * math.pi * h ** 9)
    d_poly = -6.0 * w_norm
    d_spiky = -45.0 / (math.pi * h ** 6)
    c_norm = 32.0 / (math.pi * h ** 9)
    rmin = 1e-4 * h

    def walls(q, top):
        q = torch.where(q < 0.0, torch.zeros_like(q), q)
        return torch.where(q >= top, top - 1e-4 * h, q)

    for _ in range(case["substeps"]):
        v[:, 2] -= GRAVITY * DT
        xs = walls(x + DT * v, size[scene])
        g = torch.floor(xs / h).long()
        g = torch.minimum(g, dims_s[scene] - 1)
        key = base_s[scene] + (g[:, 2] * dims_s[scene, 1] + g[:, 1]) * dims_s[scene, 0] + g[:, 0]
        key, ids = torch.sort(key, stable=True)
        q, xo, sc = xs[ids], x[ids], scene[ids]
        i, j = _pairs(q, key, ids, base_s[sc], dims_s[sc], h)
        top = size[sc]

        def add(values):
            out = torch.zeros((n,) + values.shape[1:], **f64)
            return out.index_add_(0, i, values)

        def apart():
            d = q[i] - q[j]
            r2 = d.square().sum(1)
            return d, r2, r2.clamp_min(rmin * rmin)

        def density(r2):
            return mass * w_norm * (h ** 6 + add((h * h - r2).clamp_min(0.0) ** 3))

        rho = torch.zeros(n, **f64)
        done = False
        for it in range(iters):
            d, r2, r2c = apart()
            rho = density(r2)
            con = rho / RHO0 - 1.0
            if tol > 0.0 and float(con.clamp_min(0.0).max()) <= tol:
                done = True
                break
            r = r2c.sqrt()
            gr = (h - r).clamp_min(0.0) ** 2 / r
            own = add(gr[:, None] * d).square().sum(1)
            k2 = (mass * d_spiky / RHO0) ** 2
            lam = -con.clamp_min(0.0) / (k2 * (add(gr * gr * r2) + own) + 600.0)
            stiff = 1.0 if it == 0 else 1.0 - (1.0 - p.stiffness_k) ** (1.0 / it)
            dp = stiff * mass * d_spiky / RHO0 * add(((lam[i] + lam[j]) * gr)[:, None] * d)
            q = grid.push(walls(q + dp, top), sc)
        if tol > 0.0 and not done:
            rho = density(apart()[1])
        vs = ((q - xo) / DT).clamp(-p.v_max, p.v_max)
        if terms:
            d, r2, r2c = apart()
            r = r2c.sqrt()
            u2 = (h * h - r2c).clamp_min(0.0) ** 2
            normal = h * mass * d_poly * add((u2 / rho[j])[:, None] * d)
            t3 = ((h - r).clamp_min(0.0) * r) ** 3
            spline = torch.where(r <= 0.5 * h, 2.0 * t3 - h ** 6 / 64.0, t3)
            coh = -20.0 * p.k * mass * mass * c_norm * spline / r
            kk = 2.0 * RHO0 / (rho[i] + rho[j])
            force = add(kk[:, None] * (coh[:, None] * d - p.k * mass * (normal[i] - normal[j])))
            vs = vs + (DT / rho)[:, None] * force
            # the viscosity's distance keeps the reference's dx^2 + dy^2 dz^2
            typo = (h * h - (d[:, 0] ** 2 + d[:, 1] ** 2 * d[:, 2] ** 2)).clamp_min(0.0) ** 3
            vs = vs + p.c * mass * w_norm * add((typo / rho[j])[:, None] * (vs[j] - vs[i]))
            gr = (h - r).clamp_min(0.0) ** 2 / r
            weight = gr / rho[j] * mass if model == 1 else gr
            omega = d_spiky * add(torch.linalg.cross(vs[j] - vs[i], weight[:, None] * d))
            size_w = omega.square().sum(1).sqrt()
            eta = d_spiky * add((size_w[j] * gr)[:, None] * d)
            eta = eta / eta.square().sum(1).sqrt().clamp_min(rmin)[:, None]
            conf = DT * 0.01 / (1.0 if model == 1 else mass)
            vs = vs + conf * torch.linalg.cross(eta, omega)
        x, v = torch.empty_like(q), torch.empty_like(vs)
        x[ids], v[ids] = q, vs
    return [a[:, k].contiguous() for a in (x, v) for k in range(3)]


def _unpack(w):
    return (w[:1024].view(16, 64)[:12], w[1024:1088], w[1088:5184].view(64, 64), w[5184:5248],
            w[5248:5312], w[5312:5313])


def _normalised(x, mean):
    mu, sd = (torch.from_numpy(a).to(x.device).double() for a in mean[:2])
    return (x[:, :12].double() - mu) / sd


def _forward(w, xn):
    w1, b1, w2, b2, w3, b3 = w
    silu = torch.nn.functional.silu
    return silu(silu(xn @ w1 + b1) @ w2 + b2) @ w3 + b3


def _exact_eval(x, w, mean):
    w = _unpack(torch.from_numpy(w).to(x.device).double())
    y = torch.cat([_forward(w, _normalised(part, mean)) for part in x.split(1 << 20)])
    y = y * mean[3] + mean[2]
    return {"fp32": y, "bf16": y}


def _mix64(x):
    """splitmix64 (Steele, Lea, Flood 2014), by which the trainer draws rows."""
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))


def _exact_train(case, seed, x, t, w, mean):
    w = torch.from_numpy(w).to(x.device).double()
    m, vv, loss = torch.zeros_like(w), torch.zeros_like(w), None
    for k in range(case["steps"]):
        step_seed = np.uint64(seed * 1000003 + k)
        rows = _mix64(step_seed ^ _mix64(np.arange(case["batch"], dtype=np.uint64))) % \
            np.uint64(case["rows"])
        rows = torch.from_numpy(rows.astype(np.int64)).to(x.device)
        leaf = w.clone().requires_grad_(True)
        r = _forward(_unpack(leaf), _normalised(x[rows], mean)) - \
            (t[rows].double() - mean[2]) / mean[3]
        loss = 0.5 * r.square().mean()
        (g,) = torch.autograd.grad(loss, leaf)
        m, vv = 0.9 * m + 0.1 * g, 0.999 * vv + 0.001 * g * g
        w = w - case["lr"] * (m / (1 - 0.9 ** (k + 1))) / \
            ((vv / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return {"loss": loss.detach(), "weights": w}
