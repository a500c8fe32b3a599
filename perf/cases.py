"""The work a user of this library has it do, as timed cases.

Each case goes through the public Python entry points (simuverse_amd.lbm):
interactive frames in the reference's semantics, channels past obstacles,
periodic porous boxes, batches of uneven domains, the learned collision and
its training, and the three-dimensional lattice, from calls of a few
microseconds of device work to lattices of 67 million cells, in binary32 and
binary16 storage, with the tile shape tuned by the program and left alone.

  listed()             the cases, each a dict of plain values with a name
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call
  run(state)           one pass, and its outputs
  work(case)           bytes and operations a pass cannot do without
  exact(case, seed)    the outputs in binary64, from plain torch
"""
import math

import numpy as np
import torch

from simuverse_amd import lbm as L

DEV = "cuda"

# D2Q9 in the reference's numbering: 6 2 5 / 3 0 1 / 7 4 8, y grows downwards.
EX = (0, 1, 0, -1, 0, 1, -1, -1, 1)
EY = (0, 0, -1, 0, 1, -1, -1, 1, 1)
INV = (0, 3, 4, 1, 2, 7, 8, 5, 6)
WEIGHT = (4 / 9,) + (1 / 9,) * 4 + (1 / 36,) * 4
# the reference's truncated weights and post-collision caps (frames)
W_REF = tuple(float(np.float32(v)) for v in (0.444444,) + (0.111111,) * 4 + (0.0277777,) * 4)
MAX_REF = tuple(float(np.float32(v)) for v in (0.6,) + (0.2222,) * 4 + (0.1111,) * 4)
# D3Q19: rest, faces, edges, opposite directions adjacent (include/lbm3d.h).
E3 = ((0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1),
      (1, 1, 0), (-1, -1, 0), (1, -1, 0), (-1, 1, 0), (1, 0, 1), (-1, 0, -1), (1, 0, -1), (-1, 0, 1),
      (0, 1, 1), (0, -1, -1), (0, 1, -1), (0, -1, 1))
INV3 = (0,) + tuple(i + 1 if i % 2 else i - 1 for i in range(1, 19))
WEIGHT3 = (1 / 3,) + (1 / 18,) * 6 + (1 / 36,) * 12

HIDDEN, NPARAMS = 64, 64 * 9 + 64 + 64 * 64 + 64 + 9 * 64 + 9


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # One displayed frame of the reference's own default scene (600 x 375
        # lattice, two steps, the velocity texture read back): launches and
        # latency count.
        {"name": "frame_600x375", "kind": "frame", "nx": 600, "ny": 375, "tau": 0.56},
        # The 256 x 256 channel past a cylinder, 1000 steps, shape not tuned:
        # a small lattice that lives in the caches.
        {"name": "channel_256", "kind": "channel", "nx": 256, "ny": 256, "tau": 0.6, "ux": 0.05, "storage": "f32",
         "steps": 1000, "tuned": False},
        # A channel of odd sizes as a program without tuning runs it.
        {"name": "channel_1531x1037", "kind": "channel", "nx": 1531, "ny": 1037, "tau": 0.7, "ux": 0.04,
         "storage": "f32", "steps": 400, "tuned": False},
        # The benchmark's default lattice: periodic box of disks with a body
        # force, tuned.
        {"name": "disks_4096", "kind": "disks", "nx": 4096, "ny": 4096, "tau": 0.55, "storage": "f32", "steps": 1000,
         "tuned": True},
        # The largest lattice in use, in binary16 storage, tuned.
        {"name": "disks_8192_f16", "kind": "disks", "nx": 8192, "ny": 8192, "tau": 0.55, "storage": "f16",
         "steps": 400, "tuned": True},
        # A parameter sweep: uneven channel domains stepped together, in both
        # storages.
        {"name": "batch_20", "kind": "batch", "count": 20, "size_min": 64, "size_max": 1024, "storage": "f32",
         "steps": 300},
        {"name": "batch_20_f16", "kind": "batch", "count": 20, "size_min": 64, "size_max": 1024, "storage": "f16",
         "steps": 300},
        # The learned collision on the coarse lattice of the learned workload
        # (bf16 operands, the default).
        {"name": "learned_2048", "kind": "learned", "nx": 2048, "ny": 2048, "operands": "bf16", "steps": 100},
        # Its training: Adam steps of a million samples each.
        {"name": "train_1m", "kind": "train", "samples": 2000000, "batch": 1000000, "steps": 4},
        # One loss and gradient of a small batch of host samples (a training
        # loop of the user's own).
        {"name": "grad_4096", "kind": "grad", "n": 4096},
        # Three dimensions: the benchmark's cube, tuned, and an uneven box in
        # binary16 as a program without tuning runs it.
        {"name": "d3q19_256", "kind": "d3", "nx": 256, "ny": 256, "nz": 256, "tau": 0.6, "storage": "f32",
         "steps": 200, "tuned": True},
        {"name": "d3q19_200x144x90_f16", "kind": "d3", "nx": 200, "ny": 144, "nz": 90, "tau": 0.7, "storage": "f16",
         "steps": 200, "tuned": False},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def tau():
        return round(rng.uniform(0.55, 0.9), 3)

    kind = rng.choice(["frame", "channel", "disks", "batch", "learned", "train", "grad", "d3"])
    storage = rng.choice(["f32", "f16"])
    if kind == "frame":
        return {"kind": kind, "nx": log(64, 2048), "ny": log(64, 1536), "tau": round(rng.uniform(0.52, 0.8), 3)}
    if kind == "channel":
        return {"kind": kind, "nx": log(64, 2048), "ny": log(64, 2048), "tau": round(rng.uniform(0.6, 0.9), 3),
                "ux": round(rng.uniform(0.02, 0.06), 3), "storage": storage, "steps": log(50, 1000),
                "tuned": rng.random() < 0.5}
    if kind == "disks":
        return {"kind": kind, "nx": log(256, 8192), "ny": log(256, 4096), "tau": tau(), "storage": storage,
                "steps": log(60, 500), "tuned": rng.random() < 0.75}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 20), "size_min": 64, "size_max": 32 * rng.randint(8, 32),
                "storage": storage, "steps": log(60, 300)}
    if kind == "learned":
        return {"kind": kind, "nx": log(128, 2048), "ny": log(128, 2048),
                "operands": rng.choice(["bf16", "f16"]), "steps": log(20, 100)}
    if kind == "train":
        b = log(1000, 1000000)
        return {"kind": kind, "samples": 2 * b + rng.randint(0, 999), "batch": b, "steps": rng.randint(2, 4)}
    if kind == "grad":
        return {"kind": kind, "n": log(100, 16384)}
    return {"kind": kind, "nx": log(24, 256), "ny": log(24, 256), "nz": log(24, 256), "tau": tau(),
            "storage": storage, "steps": log(20, 200), "tuned": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# Inputs, made from the case and the seed alone
# ---------------------------------------------------------------------------

def _storage(case):
    return L.STORAGE_F16_DEV if case["storage"] == "f16" else L.STORAGE_F32


def _materials(solid):
    """Solid cells are obstacles (4), the rest bulk (1)."""
    return torch.where(solid, 4, 1).to(torch.uint8).cpu().numpy()


def _disks(nx, ny, rng):
    """About 5 % of a periodic box in non-overlapping disks of radius 4..24:
    one in each square of about 112 cells, at a place of its own."""
    bx, by = max(1, nx // 112), max(1, ny // 112)
    wx, wy = nx / bx, ny / by
    r = rng.integers(4, min(25, max(5, int(min(wx, wy) / 2) - 1)), (by, bx))
    cx = (np.arange(bx) + 0.5)[None, :] * wx + (rng.random((by, bx)) - 0.5) * (wx - 2 * r - 2)
    cy = (np.arange(by) + 0.5)[:, None] * wy + (rng.random((by, bx)) - 0.5) * (wy - 2 * r - 2)
    cx, cy, r = (torch.from_numpy(np.floor(v).astype(np.float32)).to(DEV) for v in (cx, cy, r))
    x = torch.arange(nx, device=DEV)
    y = torch.arange(ny, device=DEV)
    kx = (x / wx).long().clamp_(max=bx - 1)
    ky = (y / wy).long().clamp_(max=by - 1)
    solid = torch.empty((ny, nx), dtype=torch.bool, device=DEV)
    for a in range(0, ny, 1024):  # bands of rows: small temporaries
        q = ky[a:a + 1024, None]
        dx = x[None, :] - cx[q, kx[None, :]]
        dy = y[a:a + 1024, None] - cy[q, kx[None, :]]
        solid[a:a + 1024] = dx * dx + dy * dy <= r[q, kx[None, :]] ** 2
    return solid


def _flow(nx, ny, u0, rng):
    """A smooth flow around u0 with eddies of a few sizes, and its density."""
    x = torch.arange(nx, device=DEV, dtype=torch.float32)[None, :] * (2 * math.pi / nx)
    y = torch.arange(ny, device=DEV, dtype=torch.float32)[:, None] * (2 * math.pi / ny)
    ux = torch.full((ny, nx), float(u0[0]), device=DEV)
    uy = torch.full((ny, nx), float(u0[1]), device=DEV)
    rho = torch.ones((ny, nx), device=DEV)
    for _ in range(4):
        k, m = (int(v) for v in rng.integers(1, 6, 2))
        p, q = (float(v) for v in rng.random(2) * 2 * math.pi)
        amp = 0.006 * float(rng.uniform(0.5, 1.5))
        ux += amp * torch.sin(m * y + p) * torch.cos(k * x + q)
        uy -= amp * (k * ny / (m * nx)) * min(1.0, m * nx / (k * ny)) * torch.cos(m * y + p) * torch.sin(k * x + q)
        rho += 0.002 * torch.cos(k * x + p) * torch.cos(m * y + q)
    return rho, ux, uy


def _feq(rho, ux, uy, w=WEIGHT):
    usq = 1.5 * (ux * ux + uy * uy)
    f = torch.empty((9,) + tuple(rho.shape), dtype=rho.dtype, device=rho.device)
    for i in range(9):
        eu = EX[i] * ux + EY[i] * uy
        f[i] = w[i] * rho * (1.0 + 3.0 * eu + 4.5 * eu * eu - usq)
    return f


def _channel_scene(nx, ny, rng, obstacles=1):
    """Walls on the first and last row and disks away from the ends."""
    x = torch.arange(nx, device=DEV)[None, :]
    y = torch.arange(ny, device=DEV)[:, None]
    solid = ((y == 0) | (y == ny - 1)).expand(ny, nx).clone()
    for _ in range(obstacles):
        r = int(rng.integers(2, max(3, min(nx, ny) // 12)))
        cx = int(rng.integers(r + 4, max(r + 5, nx // 2)))
        cy = int(rng.integers(r + 2, max(r + 3, ny - r - 3)))
        solid |= (x - cx) ** 2 + (y - cy) ** 2 <= r * r
    return solid


def _domain_inputs(case, seed):
    """(solid, populations) of a single 2-D lattice in physics mode."""
    rng = np.random.default_rng([seed, 2])
    nx, ny = case["nx"], case["ny"]
    if case["kind"] == "channel":
        solid = _channel_scene(nx, ny, rng)
        rho, ux, uy = _flow(nx, ny, (case["ux"], 0.0), rng)
    elif case["kind"] == "disks":
        solid = _disks(nx, ny, rng)
        rho, ux, uy = _flow(nx, ny, (0.04, 0.03), rng)
    else:
        solid = _disks(nx, ny, rng)
        rho, ux, uy = _flow(nx, ny, (0.03, 0.02), rng)
    f = _feq(rho, ux, uy)
    f[:, solid] = 0.0
    return solid, f


FORCE = (1e-6, 0.0)      # body force of the periodic boxes
FORCE3 = (1e-6, 0.0, 0.0)


def _batch_domains(case, seed):
    rng = np.random.default_rng([seed, 3])
    # the sizes are the case's own (the same for every seed), spread evenly
    # over its range and paired unevenly
    sizes = np.linspace(case["size_min"], case["size_max"], case["count"])
    sizes = [int(v) // 32 * 32 for v in sizes]
    out = []
    for d in range(case["count"]):
        nx, ny = sizes[d], sizes[(7 * d + 3) % case["count"]]
        solid = _channel_scene(nx, ny, rng, int(rng.integers(0, 9)))
        out.append({"nx": nx, "ny": ny, "tau": float(np.float32(rng.uniform(0.6, 1.0))), "x_edge": L.X_INLET_OUTLET,
                    "inlet_ux": float(np.float32(rng.uniform(0.02, 0.06))), "solid": solid})
    return out


def _network(seed):
    """Glorot-like weights, small biases: (parameters, input scale, output
    scale) of a network as training leaves it."""
    rng = np.random.default_rng([seed, 4])
    p = np.concatenate([
        rng.uniform(-1, 1, 64 * 9) * math.sqrt(6 / 73), 0.1 * rng.standard_normal(64),
        rng.uniform(-1, 1, 64 * 64) * math.sqrt(6 / 128), 0.1 * rng.standard_normal(64),
        rng.uniform(-1, 1, 9 * 64) * math.sqrt(6 / 73), 0.02 * rng.standard_normal(9)]).astype(np.float32)
    return p, float(np.float32(2e-4)), float(np.float32(4e-3))


def _samples(n, seed):
    """Order-one inputs and targets, as normalised training samples are: the
    targets depend on the inputs, with noise; outputs 3..8 train to zero."""
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + n)
    x = torch.randn((n, 9), generator=g, device=DEV)
    t = torch.zeros((n, 9), device=DEV)
    t[:, 0] = 0.6 * torch.tanh(x[:, 1] - x[:, 3]) + 0.8 * torch.randn(n, generator=g, device=DEV)
    t[:, 1] = 0.5 * x[:, 5] * x[:, 7] + 0.8 * torch.randn(n, generator=g, device=DEV)
    t[:, 2] = 0.4 * x[:, 2] + 0.9 * torch.randn(n, generator=g, device=DEV)
    return x, t


def _box_inputs(case, seed):
    """Solid cells and populations of a 3-D box with spheres (about 5 %)."""
    rng = np.random.default_rng([seed, 5])
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    ax = [torch.arange(n, device=DEV, dtype=torch.float32) for n in (nx, ny, nz)]
    X, Y, Z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    solid = torch.zeros((nz, ny, nx), dtype=torch.bool, device=DEV)
    for kz in range(max(1, nz // 32)):
        for ky in range(max(1, ny // 32)):
            for kx in range(max(1, nx // 32)):
                r = int(rng.integers(3, 11))
                c = [32 * k + 16 + int(rng.integers(-4, 5)) for k in (kx, ky, kz)]
                lo = [max(0, v - r) for v in c]
                sl = tuple(slice(a, v + r + 1) for a, v in zip(lo[::-1], c[::-1]))
                solid[sl] |= ((X[..., lo[0]:c[0] + r + 1] - c[0]) ** 2 + (Y[:, lo[1]:c[1] + r + 1] - c[1]) ** 2
                              + (Z[lo[2]:c[2] + r + 1] - c[2]) ** 2) <= r * r
    ph = rng.random(6) * 2 * math.pi
    kx, ky, kz = (2 * math.pi / n for n in (nx, ny, nz))
    one = torch.ones((nz, ny, nx), device=DEV)
    u = (0.04 + 0.01 * torch.sin(ky * Y + ph[0]) * torch.cos(kz * Z + ph[1]) * one,
         0.01 * torch.sin(2 * kz * Z + ph[2]) * torch.cos(kx * X + ph[3]) * one,
         0.01 * torch.sin(kx * X + ph[4]) * torch.cos(2 * ky * Y + ph[5]) * one)
    rho = one + 0.002 * torch.cos(kx * X + ph[0]) * torch.cos(ky * Y + ph[5])
    usq = 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
    f = torch.empty((19, nz, ny, nx), device=DEV)
    for i in range(19):
        eu = E3[i][0] * u[0] + E3[i][1] * u[1] + E3[i][2] * u[2]
        f[i] = WEIGHT3[i] * rho * (1.0 + 3.0 * eu + 4.5 * eu * eu - usq)
    f[:, solid] = 0.0
    return solid, f


def _frame_scene(case, seed):
    """The reference's default scene (walls, ghost columns, an accelerating
    inlet column, an outlet column, three disks) and one obstacle that the
    user has placed."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng([seed, 6])
    y, x = np.mgrid[0:ny, 0:nx]
    mat = np.full((ny, nx), 1, np.int32)
    mat[:, nx - 2] = 5
    mat[:, 1] = 3
    mat[:, [0, nx - 1]] = 7
    inner = (x > 1) & (x < nx - 2) & (y > 0) & (y < ny - 1)
    r = min(28.0, min(nx, ny) / 12.0)
    spots = [(nx / 7 - r, ny / 2), (nx / 5, ny / 4), (nx / 5, ny * 0.75),
             (nx * rng.uniform(0.35, 0.8), ny * rng.uniform(0.2, 0.8))]
    for cx, cy in spots:
        mat[inner & ((x - cx) ** 2 + (y - cy) ** 2 <= r * r)] = 4
    mat[[0, ny - 1], :] = 2
    info = np.zeros((ny, nx), L.LATTICE_INFO_DTYPE)
    info["material"], info["block_iter"] = mat, -1
    info["vx"] = np.where(mat == 3, np.float32(0.12), np.float32(0.0))
    return info


def prepare(case, seed):
    kind = case["kind"]
    if kind == "frame":
        lat = L.Lattice(case["nx"], case["ny"], case["tau"], mode=L.MODE_PARITY_WGSL, fluid_ty=0)
        lat.write_lattice_info(_frame_scene(case, seed))
        lat.reset()
        return {"kind": kind, "lat": lat}
    if kind in ("channel", "disks", "learned"):
        solid, f = _domain_inputs(case, seed)
        if kind == "channel":
            lat = L.Lattice(case["nx"], case["ny"], case["tau"], storage=_storage(case), x_edge=L.X_INLET_OUTLET,
                            inlet_ux=case["ux"])
        elif kind == "disks":
            lat = L.Lattice(case["nx"], case["ny"], case["tau"], storage=_storage(case), force=FORCE)
        else:
            lat = L.Lattice(case["nx"], case["ny"], 0.505, force=FORCE)
        lat.write_materials(_materials(solid))
        lat.write_populations(f.cpu().numpy())
        state = {"kind": kind, "lat": lat, "steps": case["steps"]}
        if kind == "learned":
            params, s_in, s_out = _network(seed)
            net = L.Network(seed=1)
            net.set_params(params)
            net.set_scales(s_in, s_out)
            lat.set_learned_collision(net)
            lat.set_learned_precision(L.MLP_F16 if case["operands"] == "f16" else L.MLP_BF16)
        elif case["tuned"]:
            lat.autotune(steps=20)
        return state
    if kind == "batch":
        doms = _batch_domains(case, seed)
        batch = L.Batch([{k: v for k, v in d.items() if k != "solid"} for d in doms], storage=_storage(case))
        for k, d in enumerate(doms):
            batch.write_materials(k, _materials(d["solid"]))
        batch.reset()
        batch.autotune(steps=10)
        return {"kind": kind, "batch": batch, "count": len(doms), "steps": case["steps"]}
    if kind == "train":
        x, t = _samples(case["samples"], seed)
        params, _, _ = _network(seed)
        net = L.Network(seed=1, capacity=case["samples"])
        net.set_params(params)
        net.add_samples(x.cpu().numpy(), t.cpu().numpy())
        return {"kind": kind, "net": net, "steps": case["steps"], "batch": case["batch"], "seed": seed & 0xFFFF}
    if kind == "grad":
        x, t = _samples(case["n"], seed)
        params, _, _ = _network(seed)
        net = L.Network(seed=1)
        net.set_params(params)
        return {"kind": kind, "net": net, "x": x.cpu().numpy(), "t": t.cpu().numpy()}
    solid, f = _box_inputs(case, seed)
    lat = L.Lattice3D(case["nx"], case["ny"], case["nz"], case["tau"], storage=_storage(case), force=FORCE3)
    lat.write_materials(_materials(solid))
    lat.write_populations(f.cpu().numpy())
    if case["tuned"]:
        lat.autotune(steps=10)
    return {"kind": kind, "lat": lat, "steps": case["steps"]}


LEARNING_RATE = 2e-3


def run(state):
    kind = state["kind"]
    if kind == "frame":
        state["lat"].run(2, export_macro=True)
        return state["lat"].read_macro_rgba16f()
    if kind == "batch":
        state["batch"].run(state["steps"])
        return [state["batch"].macro(d) for d in range(state["count"])]
    if kind == "train":
        loss = state["net"].train(steps=state["steps"], batch=state["batch"], lr=LEARNING_RATE, seed=state["seed"])
        return loss, state["net"].params()
    if kind == "grad":
        return state["net"].loss_grad(state["x"], state["t"])
    state["lat"].run(state["steps"])
    return state["lat"].macro()


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

# Operations of one cell's step (a fused multiply-add counts two): moments,
# equilibrium, relaxation and force, with what opposite directions share.
FLOPS_2D, FLOPS_3D = 130, 280
# 9 -> 64 -> 64 -> 9 forward; backward is twice that less the input gradient.
FLOPS_NET = 2 * (9 * 64 + 64 * 64 + 64 * 9)
FLOPS_NET_TRAIN = 3 * FLOPS_NET - 2 * 9 * 64


def work(case):
    """Bytes: the state read and written once, and the fields handed out."""
    kind = case["kind"]
    if kind == "train":
        n = case["batch"] * case["steps"]
        return {"bytes": 72.0 * n, "flops": float(FLOPS_NET_TRAIN) * n}
    if kind == "grad":
        return {"bytes": 72.0 * case["n"] + 8.0 * NPARAMS, "flops": float(FLOPS_NET_TRAIN) * case["n"]}
    elem = 2 if case.get("storage") == "f16" else 4
    if kind == "d3":
        cells = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": cells * (2.0 * 19 * elem + 1 / 8 + 16), "flops": float(FLOPS_3D) * cells * case["steps"]}
    if kind == "batch":
        sizes = [int(v) // 32 * 32 for v in np.linspace(case["size_min"], case["size_max"], case["count"])]
        cells = sum(sizes[d] * sizes[(7 * d + 3) % len(sizes)] for d in range(len(sizes)))
    else:
        cells = case["nx"] * case["ny"]
    if kind == "frame":
        return {"bytes": cells * (2.0 * 36 + 1 + 8), "flops": 2.0 * FLOPS_2D * cells}
    per = FLOPS_2D + (FLOPS_NET if kind == "learned" else 0)
    return {"bytes": cells * (2.0 * 9 * elem + 1 / 8 + 12), "flops": float(per) * cells * case["steps"]}


# ---------------------------------------------------------------------------
# The same in binary64, from plain torch
# ---------------------------------------------------------------------------

def _roll(a, ex, ey):
    """Value at (x, y) of a at (x - ex, y - ey), periodic."""
    return torch.roll(a, (ey, ex), (-2, -1)) if ex or ey else a


class _Plane:
    """D2Q9 BGK with Guo force, half-way bounce-back, and the Zou-He inlet
    and zero-gradient outlet where `inlet` is given, in binary64."""

    def __init__(self, f, solid, tau, force=(0.0, 0.0), inlet=None):
        self.f, self.solid, self.inlet = f, solid, inlet
        self.omega = 1.0 / float(np.float32(tau))
        self.g = tuple(float(np.float32(v)) for v in force)
        self.own = []  # where direction i comes from the cell itself
        for i in range(9):
            m = _roll(solid, EX[i], EY[i]).clone()
            if inlet is not None and EX[i]:
                m[:, 0 if EX[i] > 0 else -1] = True
            self.own.append(m)
        if inlet is not None:
            self.out_rows = ~solid[:, -2]

    def gather(self):
        p = torch.empty_like(self.f)
        for i in range(9):
            torch.where(self.own[i], self.f[INV[i]], _roll(self.f[i], EX[i], EY[i]), out=p[i])
        if self.inlet is not None:
            p[:, self.out_rows, -1] = p[:, self.out_rows, -2]
            c = p[:, :, 0]
            u0 = self.inlet
            rho = (c[0] + c[2] + c[4] + 2.0 * (c[3] + c[6] + c[7])) / (1.0 - u0)
            h = 0.5 * (c[4] - c[2])
            c1, c5, c8 = c[3] + 2.0 / 3.0 * rho * u0, c[7] + h + rho * u0 / 6.0, c[6] - h + rho * u0 / 6.0
            c[1], c[5], c[8] = c1, c5, c8
        return p

    def moments(self, p):
        rho = p.sum(0)
        ux = (p[1] - p[3] + p[5] - p[6] - p[7] + p[8] + 0.5 * self.g[0]) / rho
        uy = (p[4] - p[2] + p[7] - p[5] + p[8] - p[6] + 0.5 * self.g[1]) / rho
        return rho, ux, uy

    def step(self, correct=None):
        p = self.gather()
        rho, ux, uy = self.moments(p)
        usq = 1.5 * (ux * ux + uy * uy)
        gx, gy = self.g
        ug = ux * gx + uy * gy if gx or gy else None
        extra = correct(p, rho, ux, uy) if correct else None
        for i in range(9):
            eu = EX[i] * ux + EY[i] * uy
            feq = (eu * (3.0 + 4.5 * eu)).sub_(usq).add_(1.0).mul_(rho).mul_(WEIGHT[i])
            out = p[i].add_(feq.sub_(p[i]).mul_(self.omega))
            if ug is not None:
                eg = EX[i] * gx + EY[i] * gy
                out += (1.0 - 0.5 * self.omega) * WEIGHT[i] * (3.0 * (eg - ug) + 9.0 * eg * eu)
            if extra is not None:
                out += extra[i]
        self.f = p

    def macro(self):
        rho, ux, uy = self.moments(self.gather())
        return [torch.where(self.solid, torch.zeros((), dtype=torch.float64, device=DEV), v).cpu().numpy()
                for v in (rho, ux, uy)]


def _net64(params, x):
    """The network in binary64: (y, pre-activations, activations)."""
    p = torch.from_numpy(params.astype(np.float64)).to(DEV) if isinstance(params, np.ndarray) else params
    w1, b1, w2, b2, w3, b3 = p.split([576, 64, 4096, 64, 576, 9])
    a1 = torch.addmm(b1, x, w1.view(64, 9).t())
    h1 = torch.nn.functional.gelu(a1)
    a2 = torch.addmm(b2, h1, w2.view(64, 64).t())
    h2 = torch.nn.functional.gelu(a2)
    return torch.addmm(b3, h2, w3.view(9, 64).t()), (a1, h1, a2, h2)


# rows of the energy and the two stress moments of the orthogonal basis
M_E = (-4, -1, -1, -1, -1, 2, 2, 2, 2)
M_XX = tuple(EX[i] ** 2 - EY[i] ** 2 for i in range(9))
M_XY = tuple(EX[i] * EY[i] for i in range(9))


def _learned_correction(params, s_in, s_out, solid, omega):
    near = torch.zeros_like(solid)
    for dy in (-1, 0, 1):
        for dx in (-1, 0, 1):
            near |= _roll(solid, dx, dy)
    cells = (~near).view(-1).nonzero().view(-1)
    bound = min(0.5 * (2.0 - omega), 0.5 * omega)
    p64 = torch.from_numpy(params.astype(np.float64)).to(DEV)

    def correct(p, rho, ux, uy):
        q = p - _feq(rho, ux, uy)
        flat = q.view(9, -1)
        corr = torch.zeros_like(flat)
        scale = torch.tensor([1.0 / (w * s_in) for w in WEIGHT], dtype=torch.float64, device=DEV)
        for a in range(0, cells.numel(), 1 << 20):
            c = cells[a:a + (1 << 20)]
            qc = flat[:, c]
            y, _ = _net64(p64, (qc.t() * scale).contiguous())
            for k, (m, norm) in enumerate(((M_E, 36.0), (M_XX, 4.0), (M_XY, 4.0))):
                row = torch.tensor(m, dtype=torch.float64, device=DEV)
                d = (s_out * y[:, k]).clamp_(-bound, bound) * (row[:, None] * qc).sum(0) / norm
                corr[:, c] += row[:, None] * d[None, :]
        return corr.view_as(q)

    return correct


def _exact_frame(case, seed):
    info = _frame_scene(case, seed)
    nx, ny = case["nx"], case["ny"]
    mat = torch.from_numpy(info["material"].copy()).to(DEV)
    solid, accel = (mat == 2) | (mat == 4), mat == 3
    vx = torch.from_numpy(info["vx"].astype(np.float64)).to(DEV)
    f = torch.tensor(W_REF, dtype=torch.float64, device=DEV)[:, None, None].repeat(1, ny, nx)
    f[1] = W_REF[1] + 0.5 * W_REF[3]
    f[3] = 0.5 * W_REF[3]
    f[:, solid] = 0.0
    omega = 1.0 / float(np.float32(case["tau"]))
    inside = torch.zeros_like(solid)
    inside[1:-1, 1:-1] = True
    for _ in range(2):
        p = torch.stack([_roll(f[i], EX[i], EY[i]) for i in range(9)])
        rho = p.sum(0).clamp_(0.8, 1.2)
        ux = sum(EX[i] * p[i] for i in range(9)) / rho
        uy = sum(EY[i] * p[i] for i in range(9)) / rho
        ux = torch.where(accel, 0.5 * vx / rho, ux)
        uy = torch.where(accel, torch.zeros_like(uy), uy)
        feq = _feq(rho, ux, uy, W_REF)
        new = torch.zeros_like(f)
        for i in range(9):
            t = p[i] - omega * (p[i] - feq[i]) + torch.where(accel, W_REF[i] * 3.0 * EX[i] * vx, torch.zeros_like(vx))
            new[i] = t.clamp_(0.0, MAX_REF[i])
        new[:, solid] = 0.0
        back = torch.zeros_like(f)
        for i in range(1, 9):
            hit = ~solid & inside & _roll(solid, -EX[i], -EY[i])
            back[INV[i]] += _roll(torch.where(hit, new[i], torch.zeros_like(new[i])), EX[i], EY[i])
            new[i][hit] = 0.0
        f = new + back
    one = (~solid).double()
    return torch.stack([ux * one, uy * one, rho * one, one], -1).cpu().numpy()


class _Box:
    """D3Q19 BGK with Guo force and half-way bounce-back, periodic."""

    def __init__(self, f, solid, tau, force):
        self.f, self.solid = f, solid
        self.omega = 1.0 / float(np.float32(tau))
        self.g = tuple(float(np.float32(v)) for v in force)
        self.own = [torch.roll(solid, E3[i][::-1], (0, 1, 2)) for i in range(19)]

    def gather(self):
        p = torch.empty_like(self.f)
        for i in range(19):
            torch.where(self.own[i], self.f[INV3[i]], torch.roll(self.f[i], E3[i][::-1], (0, 1, 2)), out=p[i])
        return p

    def moments(self, p):
        rho = p.sum(0)
        u = [sum(p[i] * E3[i][a] for i in range(19) if E3[i][a]).add_(0.5 * self.g[a]).div_(rho) for a in range(3)]
        return rho, u

    def step(self):
        p = self.gather()
        rho, u = self.moments(p)
        usq = 1.5 * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
        ug = sum(self.g[a] * u[a] for a in range(3))
        for i in range(19):
            eu = E3[i][0] * u[0] + E3[i][1] * u[1] + E3[i][2] * u[2]
            feq = (eu * (3.0 + 4.5 * eu)).sub_(usq).add_(1.0).mul_(rho).mul_(WEIGHT3[i])
            eg = sum(E3[i][a] * self.g[a] for a in range(3))
            p[i].add_(feq.sub_(p[i]).mul_(self.omega))
            p[i].add_((9.0 * eg * eu + 3.0 * (eg - ug)).mul_((1.0 - 0.5 * self.omega) * WEIGHT3[i]))
        self.f = p

    def macro(self):
        rho, u = self.moments(self.gather())
        zero = torch.zeros((), dtype=torch.float64, device=DEV)
        rho, *u = (torch.where(self.solid, zero, v) for v in (rho, *u))
        return rho.cpu().numpy(), torch.stack(u).cpu().numpy()


def _mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _loss_grad64(p, x, t):
    """Loss 1/(9 n) sum (y - t)^2 and its gradient, in binary64."""
    n = x.shape[0]
    loss, grad = 0.0, torch.zeros(NPARAMS, dtype=torch.float64, device=DEV)
    for a in range(0, n, 1 << 18):
        q = p.clone().requires_grad_(True)
        y, _ = _net64(q, x[a:a + (1 << 18)].double())
        part = (y - t[a:a + (1 << 18)].double()).square().sum() / (9.0 * n)
        part.backward()
        loss += float(part.detach())
        grad += q.grad
    return loss, grad


def _exact_train(case, seed):
    x, t = _samples(case["samples"], seed)
    p = torch.from_numpy(_network(seed)[0].astype(np.float64)).to(DEV)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    golden, turn = 0x9E3779B97F4A7C15, 0xD1B54A32D192ED03
    loss = 0.0
    for s in range(case["steps"]):
        base = ((seed & 0xFFFF) + turn * (s + 1)) % (1 << 64)
        with np.errstate(over="ignore"):
            k = np.uint64(base) + np.uint64(golden) * np.arange(1, case["batch"] + 1, dtype=np.uint64)
            index = (_mix64(k) % np.uint64(case["samples"])).astype(np.int64)
        index = torch.from_numpy(index).to(DEV)
        loss, g = _loss_grad64(p, x[index], t[index])
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - LEARNING_RATE * (m / (1 - 0.9 ** (s + 1))) / ((v / (1 - 0.999 ** (s + 1))).sqrt() + 1e-8)
    return loss, p.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        return _exact_frame(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "grad":
        x, t = _samples(case["n"], seed)
        p = torch.from_numpy(_network(seed)[0].astype(np.float64)).to(DEV)
        loss, g = _loss_grad64(p, x, t)
        return loss, g.cpu().numpy()
    if kind == "batch":
        out = []
        for d in _batch_domains(case, seed):
            ny, nx = d["solid"].shape
            f = torch.tensor(WEIGHT, dtype=torch.float64, device=DEV)[:, None, None].repeat(1, ny, nx)
            plane = _Plane(f, d["solid"], d["tau"], inlet=d["inlet_ux"])
            for _ in range(case["steps"]):
                plane.step()
            out.append(plane.macro())
        return out
    if kind == "d3":
        if case["nx"] * case["ny"] * case["nz"] * case["steps"] > 4e9:
            return None
        solid, f = _box_inputs(case, seed)
        box = _Box(f.double(), solid, case["tau"], FORCE3)
        for _ in range(case["steps"]):
            box.step()
        return box.macro()
    if case["nx"] * case["ny"] * case["steps"] > 3e10 or (kind == "learned" and
                                                          case["nx"] * case["ny"] * case["steps"] > 5e8):
        return None
    solid, f = _domain_inputs(case, seed)
    if kind == "channel":
        plane = _Plane(f.double(), solid, case["tau"], inlet=float(np.float32(case["ux"])))
    elif kind == "disks":
        plane = _Plane(f.double(), solid, case["tau"], force=FORCE)
    else:
        plane = _Plane(f.double(), solid, 0.505, force=FORCE)
    correct = None
    if kind == "learned":
        correct = _learned_correction(*_network(seed), solid, plane.omega)
    for _ in range(case["steps"]):
        plane.step(correct)
    return plane.macro()
