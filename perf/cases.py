"""The work that users of this library have it do, as timed cases.

Every case goes through the package's public entry points: `Volume3` (the
projection, the surface step), `project_batch` and `learned.Network`. Sizes,
options and input distributions are those of the repository's own workloads,
tests and benchmark: free-surface tanks with solid spheres and smooth 16-mode
velocities, a closed box of independent faces, a bottom cut into the grid
with fractional apertures, a level-set pool, a sloshing basin, uneven patches
and the convolutional preconditioner's training step.

`exact` solves the same discrete systems in 64 bits with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from fluidisim_amd import _lib
from fluidisim_amd.learned import Network
from fluidisim_amd.volume import Domain3, Volume3, project_batch

MAX_ITERS = 4000
EDGES = (32, 48, 64, 96, 128)
EDGE_WEIGHTS = (0.3, 0.25, 0.2, 0.15, 0.1)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # The smallest patch of the patch workload on its own: one call in a
        # frame, where latency and launches count.
        dict(name="patch_32", kind="tank", nx=32, ny=32, nz=32, storage="f32"),
        # A pure-Neumann closed box of noise: the three-level V-cycle and the
        # gauge of the singular problem.
        dict(name="closed_box_64", kind="box", nx=64, ny=64, nz=64),
        # A basin whose rows do not split into groups of four cells and whose
        # edges halve once only: a size that nobody chose for the machine.
        dict(name="ragged_tank_90x70x54", kind="tank", nx=90, ny=70, nz=54, storage="f32"),
        # A bottom cut into the grid (fractional apertures) with the default
        # options (damped Jacobi, re-discretised coarse levels) and physical
        # units: the settings a host switching to the library starts from.
        dict(name="cut_bottom_128x64x96", kind="cut", nx=128, ny=64, nz=96),
        # A liquid given by labels and a level set (pool, drop, solid block).
        dict(name="level_set_128x96x80", kind="levelset", nx=128, ny=96, nz=80),
        # An ordinary tank, one projection from rest.
        dict(name="tank_128", kind="tank", nx=128, ny=128, nz=128, storage="f32"),
        # The large tank (8.4 M cells), and the same with the V-cycle's
        # vectors in bfloat16 and the residual replaced every 50 iterations.
        dict(name="tank_256x256x128", kind="tank", nx=256, ny=256, nz=128, storage="f32"),
        dict(name="tank_256x256x128_bf16", kind="tank", nx=256, ny=256, nz=128, storage="bf16"),
        # Sixteen uneven patches of a scene projected together.
        dict(name="batch_16_patches", kind="batch", count=16, edges_seed=1),
        # One step of the moving surface in a large basin: advection, warm
        # projection, extrapolation, transport.
        dict(name="surface_step_256x256x128", kind="step", nx=256, ny=256, nz=128),
        # Flexible CG with the network as the V-cycle's initial guess (the
        # network's forward pass in the loop).
        dict(name="learned_fcg_256x256x128", kind="learned", nx=256, ny=256, nz=128),
        # Loss and gradients of the network at its training size (forward and
        # backward).
        dict(name="network_gradients_128", kind="train", nx=128, ny=128, nz=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_mult(rng, m, lo, hi):
    return max(lo, min(hi, m * int(round(_log_int(rng, lo, hi) / m))))


def draw(rng):
    kind = rng.choice(("tank", "tank", "ragged", "ragged", "box", "cut", "levelset", "batch", "step", "learned", "train"))
    if kind == "tank":
        nx, ny, nz = _log_mult(rng, 8, 32, 256), _log_mult(rng, 8, 32, 256), _log_mult(rng, 8, 32, 128)
        return dict(kind="tank", nx=nx, ny=ny, nz=nz, storage=rng.choice(("f32", "f32", "bf16")))
    if kind == "ragged":
        if rng.random() < 0.5:  # odd edges: no coarse level at all
            return dict(kind="tank", nx=_log_int(rng, 17, 72), ny=_log_int(rng, 17, 72), nz=_log_int(rng, 17, 64),
                        storage="f32")
        return dict(kind="tank", nx=4 * _log_int(rng, 6, 40) + 2, ny=2 * _log_int(rng, 12, 64),
                    nz=2 * _log_int(rng, 12, 40), storage="f32")
    if kind == "box":
        n = _log_mult(rng, 4, 32, 128)
        return dict(kind="box", nx=n, ny=n, nz=n)
    if kind == "cut":
        n = rng.choice((32, 48, 64, 80, 96, 128))
        return dict(kind="cut", nx=n, ny=n // 2, nz=3 * n // 4)
    if kind == "levelset":
        return dict(kind="levelset", nx=_log_mult(rng, 4, 32, 160), ny=_log_mult(rng, 2, 24, 128),
                    nz=_log_mult(rng, 2, 32, 96))
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(4, 16), edges_seed=rng.randint(2, 10000))
    if kind == "step":
        return dict(kind="step", nx=_log_mult(rng, 8, 32, 256), ny=_log_mult(rng, 8, 32, 256),
                    nz=_log_mult(rng, 8, 32, 128))
    if kind == "learned":
        return dict(kind="learned", nx=rng.choice((64, 128, 192, 256)), ny=_log_mult(rng, 4, 32, 256),
                    nz=_log_mult(rng, 4, 32, 128))
    return dict(kind="train", nx=rng.choice((64, 128)), ny=_log_mult(rng, 4, 32, 128), nz=_log_mult(rng, 4, 32, 128))


def _patch_sizes(case):
    r = np.random.default_rng(case["edges_seed"])
    return [tuple(int(v) for v in r.choice(EDGES, size=3, p=EDGE_WEIGHTS)) for _ in range(case["count"])]


def _work_of(nx, ny, nz):
    n, cols = nx * ny * nz, nx * ny
    faces = (nx + 1) * ny * nz + nx * (ny + 1) * nz + nx * ny * (nz + 1)
    # predicted faces in, corrected faces out, pressure out, cell classes and
    # heights in; one operator application and one gradient per cell
    return 8 * faces + 5 * n + 4 * cols, 30 * n


def work(case):
    if case["kind"] == "batch":
        parts = [_work_of(*s) for s in _patch_sizes(case)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["kind"] == "train":
        n = nx * ny * nz
        # binary16 features (4 channels), target, wet flags; weight products
        # of the forward pass, of the data gradients and of the weight
        # gradients (27 taps, levels at 1, 1/8 and 1/64 of the cells)
        macs = 27 * sum(ci * co * n >> (3 * level) for level, ci, co in _layer_sizes())
        return {"bytes": 13 * n + 8 * 80729, "flops": 3 * 2 * macs}
    b, f = _work_of(nx, ny, nz)
    if case["kind"] == "step":
        b += 4 * nx * ny * nz + 12 * nx * ny  # the warm pressure in, heights and their roundoff out
    if case["kind"] == "learned":
        # one application of the network is the least that this path does
        f += 2 * 27 * sum(ci * co * nx * ny * nz >> (3 * level) for level, ci, co in _layer_sizes())
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------- inputs
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _smooth_faces(rng, nx, ny, nz):
    """u, v, w faces of a sum of 16 Fourier modes of amplitude ~ 1/|k|^2, RMS
    about 1, divergence and all."""
    dev = _dev()
    comp = [-4, -3, -2, -1, 1, 2, 3, 4]
    k = rng.choice(comp, size=(16, 3)).astype(np.float64)
    amp = 1.0 / (k * k).sum(1)
    amp /= math.sqrt(0.5 * (amp * amp).sum() / 3.0)
    z, t = rng.uniform(-1, 1, 16), rng.uniform(0, 2 * math.pi, 16)
    pol = np.stack([np.sqrt(1 - z * z) * np.cos(t), np.sqrt(1 - z * z) * np.sin(t), z], 1) * amp[:, None]
    phase = rng.uniform(0, 2 * math.pi, 16)

    def table(axis, count, length, half, ph=None):
        x = (np.arange(count) + (0.5 if half else 0.0)) / length
        th = 2 * math.pi * k[:, axis, None] * x[None] + (0.0 if ph is None else ph[:, None])
        return torch.from_numpy(np.exp(1j * th)).to(torch.complex64).to(dev)

    def faces(a, sizes):
        X = table(0, sizes[0], nx, a != 0, phase)
        Y = table(1, sizes[1], ny, a != 1)
        Z = table(2, sizes[2], nz, a != 2)
        P = torch.from_numpy(pol[:, a]).to(torch.complex64).to(dev)
        zy = (Z[:, :, None] * Y[:, None, :]).reshape(16, -1)  # 16 x (nz ny)
        out = zy.real.t().contiguous() @ (P[:, None] * X).real - zy.imag.t().contiguous() @ (P[:, None] * X).imag
        return out.reshape(sizes[2], sizes[1], sizes[0]).contiguous()

    return faces(0, (nx + 1, ny, nz)), faces(1, (nx, ny + 1, nz)), faces(2, (nx, ny, nz + 1))


def _close(u, v, w, solid):
    """Zero on the box walls and on faces of solid cells."""
    u[:, :, 0] = 0
    u[:, :, -1] = 0
    v[:, 0] = 0
    v[:, -1] = 0
    w[0] = 0
    w[-1] = 0
    if solid is not None:
        s = torch.from_numpy(solid.astype(np.float32)).to(u.device) == 0
        u[:, :, :-1] *= s
        u[:, :, 1:] *= s
        v[:, :-1] *= s
        v[:, 1:] *= s
        w[:-1] *= s
        w[1:] *= s
    return u, v, w


def _spheres(rng, nx, ny, nz, spheres):
    solid = np.zeros((nz, ny, nx), np.uint8)
    for cx, cy, cz, r in spheres:
        i = np.arange(nx, dtype=np.float64) + 0.5 - cx
        j = np.arange(ny, dtype=np.float64) + 0.5 - cy
        k = np.arange(nz, dtype=np.float64) + 0.5 - cz
        a, b = max(0, int(cz - r) - 1), min(nz, int(cz + r) + 2)
        if b > a:
            solid[a:b] |= (k[a:b, None, None] ** 2 + j[None, :, None] ** 2 + i[None, None, :] ** 2 < r * r)
    return solid


def _red_black(**more):
    o = dict(preconditioner=_lib.PRECOND_MULTIGRID, smoother=_lib.SMOOTH_RBGS, max_levels=-1, pre_sweeps=2,
             post_sweeps=2, coarse_sweeps=8, coarse_operator=_lib.COARSE_GALERKIN)
    o.update(more)
    return o


def _tank(nx, ny, nz, seed, **options):
    """A free surface of four sines about half the height, eight solid spheres
    in the water, a smooth velocity; p = 0 at the surface, closed lid."""
    rng = np.random.default_rng([seed, nx, ny, nz])
    s = nz / 128.0
    a, f, g, ph = rng.uniform(2, 6, 4) * s, rng.uniform(0.02, 0.15, 4), rng.uniform(0.02, 0.15, 4), rng.uniform(0, 2 * math.pi, 4)

    def height(x, y):
        return nz / 2 + sum(a[m] * np.sin(f[m] * x + g[m] * y + ph[m]) for m in range(4))

    eta = height(np.arange(nx)[None] + 0.5, np.arange(ny)[:, None] + 0.5).astype(np.float32)
    spheres = []
    for _ in range(8):
        cx, cy = rng.uniform(0, nx), rng.uniform(0, ny)
        spheres.append((cx, cy, rng.uniform(0, height(cx, cy)), rng.uniform(6, 14) * s))
    solid = _spheres(rng, nx, ny, nz, spheres)
    return dict(nx=nx, ny=ny, nz=nz, dx=1.0, rho=1.0, g=9.81, rest=nz / 2.0, eta=eta, solid=solid,
                faces=_close(*_smooth_faces(rng, nx, ny, nz), solid), homogeneous=True, closed_lid=True, scale=-1.0,
                k1=1.0, options=_red_black(**options))


def _box(nx, ny, nz, seed):
    """All fluid between six walls, independent faces in [-1, 1]."""
    rng = np.random.default_rng([seed, nx])
    f = [torch.from_numpy(rng.uniform(-1, 1, s).astype(np.float32)).to(_dev())
         for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
    return dict(nx=nx, ny=ny, nz=nz, dx=1.0, rho=1.0, g=9.81, rest=float(nz), eta=np.full((ny, nx), nz, np.float32),
                solid=None, faces=_close(*f, None), homogeneous=True, closed_lid=True, scale=-1.0, k1=1.0,
                options=_red_black(max_levels=2))


def _cut(nx, ny, nz, seed):
    """An 8 m tank, 4 m of water with a sine of about a centimetre, a smooth
    bump on the bottom cut into the grid: fractional apertures, solid cells
    below the bottom, the hydrostatic ghost values of the heights."""
    rng = np.random.default_rng([seed, nx, ny, nz])
    f32 = np.float32
    dx = f32(8.0) / f32(nx)
    d = float(dx)
    x0, y0, top = rng.uniform(2, 6), rng.uniform(0.25, 0.75) * ny * d, rng.uniform(0.4, 0.8)

    def bottom(x, y):
        return 0.4 + top * np.exp(-(((x - x0) / 1.2) ** 2 + ((y - y0) / 0.9) ** 2))

    xc, yc = (np.arange(nx) + 0.5) * d, (np.arange(ny) + 0.5) * d
    z0 = np.arange(nz)[:, None, None] * d
    level = lambda b: np.clip((z0 + d - b[None]) / d, 0.0, 1.0)  # the share of a cell height above b
    snap = lambda q: np.where(q < 0.02, 0.0, np.where(q > 0.98, 1.0, q)).astype(f32)
    solid = (level(bottom(xc[None], yc[:, None])) < 0.02).astype(np.uint8)
    ou = snap(level(bottom(np.arange(nx + 1)[None] * d, yc[:, None])))
    ov = snap(level(bottom(xc[None], np.arange(ny + 1)[:, None] * d)))
    ow = snap(np.clip((np.arange(nz + 1)[:, None, None] * d - bottom(xc[None], yc[:, None])[None]) / d + 0.5, 0, 1))
    ou[:, :, [0, nx]] = 0
    ov[:, [0, ny]] = 0
    ow[0] = 0
    free = (1 - solid).astype(f32)
    ou[:, :, :-1] *= free
    ou[:, :, 1:] *= free
    ov[:, :-1] *= free
    ov[:, 1:] *= free
    ow[:-1] *= free
    ow[1:] *= free
    amp, ph = rng.uniform(0.005, 0.02), rng.uniform(0, 2 * math.pi)
    eta = np.broadcast_to((4.0 + amp * np.sin(2 * math.pi * xc / 8.0 + ph)).astype(f32), (ny, nx)).copy()
    faces = [0.1 * q for q in _close(*_smooth_faces(rng, nx, ny, nz), solid)]
    dt = 2e-3
    return dict(nx=nx, ny=ny, nz=nz, dx=d, rho=1025.0, g=9.81, rest=4.0, eta=eta, solid=solid, opens=(ou, ov, ow),
                faces=faces, homogeneous=False, closed_lid=False, scale=float(f32(-1025.0 / dt)),
                k1=float(f32(dt / 1025.0)), options={})


def _levelset(nx, ny, nz, seed):
    """A pool of a third of the box, a drop above it, a solid block in a
    corner, noisy faces under gravity."""
    rng = np.random.default_rng([seed, nx, ny, nz])
    dx, rho, dt = 0.025, 1000.0, 0.004
    X, Y, Z = (np.arange(nx) + 0.5) * dx, (np.arange(ny) + 0.5) * dx, (np.arange(nz) + 0.5) * dx
    X, Y, Z = X[None, None], Y[None, :, None], Z[:, None, None]
    pool = Z - (nz * dx / 3 + 0.03 * np.sin(2 * math.pi * X / (nx * dx) + rng.uniform(0, 6.28))) + 0 * Y
    drop = np.sqrt((X - rng.uniform(0.4, 0.7) * nx * dx) ** 2 + (Y - rng.uniform(0.4, 0.6) * ny * dx) ** 2 +
                   (Z - 0.7 * nz * dx) ** 2) - 0.15 * nz * dx
    phi = np.minimum(pool, drop).astype(np.float32)
    label = np.where(phi < 0, _lib.LABEL_WATER, _lib.LABEL_AIR).astype(np.uint8)
    label[: int(0.25 * nz), : int(0.3 * ny), : int(0.25 * nx)] = _lib.LABEL_SOLID
    u = rng.uniform(-0.2, 0.2, (nz, ny, nx + 1)).astype(np.float32)
    v = rng.uniform(-0.2, 0.2, (nz, ny + 1, nx)).astype(np.float32)
    w = (rng.uniform(-0.2, 0.2, (nz + 1, ny, nx)) - 9.81 * dt).astype(np.float32)
    faces = _close(*(torch.from_numpy(a).to(_dev()) for a in (u, v, w)), None)
    return dict(nx=nx, ny=ny, nz=nz, dx=dx, rho=rho, g=9.81, rest=0.0, eta=None, solid=None, label=label, phi=phi,
                faces=faces, homogeneous=True, closed_lid=True, scale=-rho / dt, k1=dt / rho,
                options=_red_black(coarse_sweeps=2))


STEP_US = 1000


def _basin(nx, ny, nz, seed):
    """An 8 m basin of water two thirds full, a standing wave of 2 % with its
    own phase, four solid spheres well below the surface, already moving."""
    rng = np.random.default_rng([seed, nx, ny, nz])
    f32 = np.float32
    dx = f32(8.0) / f32(nx)
    rest = f32(nz) * dx * f32(2.0) / f32(3.0)
    a, b = rng.uniform(0.5, 1.0), rng.uniform(-0.5, 0.5)
    ci, cj = np.cos(math.pi * (np.arange(nx) + 0.5) / nx), np.cos(math.pi * (np.arange(ny) + 0.5) / ny)
    eta = (rest * (1 + 0.02 * (a * cj[:, None] * ci[None] + b * ci[None]))).astype(f32)
    spheres = []
    for _ in range(4):
        r = rng.uniform(2.0, 4.0)
        top = max(r + 1.5, float(rest) / 2 / float(dx) - r - 1)
        spheres.append((rng.uniform(r + 1, nx - r - 1), rng.uniform(r + 1, ny - r - 1), rng.uniform(r + 1, top), r))
    solid = _spheres(rng, nx, ny, nz, spheres)
    faces = [0.05 * q for q in _close(*_smooth_faces(rng, nx, ny, nz), solid)]
    dt = STEP_US * 1e-6
    return dict(nx=nx, ny=ny, nz=nz, dx=float(dx), rho=1025.0, g=9.81, rest=float(rest), eta=eta, solid=solid,
                faces=faces, homogeneous=False, closed_lid=False, scale=float(f32(-1025.0 / dt)),
                k1=float(f32(dt / 1025.0)), options=_red_black())


def _problem(case, seed):
    kind, size = case["kind"], (case["nx"], case["ny"], case["nz"])
    if kind == "tank":
        if case["storage"] == "bf16":
            return _tank(*size, seed, vcycle_storage=_lib.STORE_BF16, replace_every=50)
        return _tank(*size, seed)
    if kind == "learned":
        return _tank(*size, seed, preconditioner=_lib.PRECOND_LEARNED, learned_budget=200, learned_vcycle=1)
    return {"box": _box, "cut": _cut, "levelset": _levelset, "step": _basin}[kind](*size, seed)


def _patches(case, seed):
    return [_tank(*s, 1000 * seed + q) for q, s in enumerate(_patch_sizes(case))]


def _volume(P):
    vol = Volume3.configure(Domain3(P["nx"], P["ny"], P["nz"], P["dx"]), rho=P["rho"], g_eff=P["g"], **P["options"])
    if P.get("label") is not None:
        vol.set_level_set(P["label"].ravel(), P["phi"].ravel())
    else:
        vol.set_surface_mode(P["homogeneous"], P["closed_lid"])
        opens = P.get("opens", (None, None, None))
        flat = lambda a: None if a is None else a.ravel()
        vol.set_solid(flat(P["solid"]), *(flat(o) for o in opens))
        vol.set_free_surface(P["eta"].ravel(), P["rest"])
    return vol


# ---------------------------------------------------------------- the network's training inputs
def _layer_sizes():
    return [(0, 4, 8), (0, 8, 8), (1, 8, 16), (1, 16, 16), (2, 16, 32), (2, 32, 32), (1, 32, 16), (1, 16, 16),
            (0, 16, 8), (0, 8, 8), (0, 8, 1)]


def _weights(rng):
    """He-style weights, as a training run starts with, biases a little off 0."""
    parts = []
    for q, (_, ci, co) in enumerate(_layer_sizes()):
        parts.append(rng.standard_normal(co * 27 * ci) * math.sqrt((1.0 if co == 1 else 2.0) / (27 * ci)))
        parts.append(rng.uniform(-0.05, 0.05, co))
    return np.concatenate(parts).astype(np.float32)


def _train_inputs(case, seed):
    """Features (scaled residual, wet, ghost row, solid) of a half-full tank
    and a smooth target on its wet cells."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    rng = np.random.default_rng([seed, nx, ny, nz])
    dev = _dev()
    modes = _smooth_faces(rng, nx, ny, nz)
    noise = torch.from_numpy(rng.standard_normal((nz, ny, nx)).astype(np.float32)).to(dev)
    i, j = torch.arange(nx, device=dev), torch.arange(ny, device=dev)
    top = nz / 2 + nz / 32 * (torch.sin(0.11 * i)[None, :] + torch.cos(0.07 * j)[:, None])
    k = torch.arange(nz, device=dev)[:, None, None]
    solid = torch.from_numpy(_spheres(rng, nx, ny, nz, [(rng.uniform(0, nx), rng.uniform(0, ny), rng.uniform(0, nz / 2),
                                                         nz * rng.uniform(0.05, 0.1)) for _ in range(8)])).to(dev) != 0
    wet = (k + 0.5 < top) & ~solid
    ghost = wet & (k + 1.5 >= top)
    x = torch.stack([(modes[0][:, :, 1:] + 0.5 * noise) * wet, wet.float(), ghost.float(), solid.float()], -1)
    x = x.to(torch.float16).contiguous()
    target = (modes[2][1:] * wet).contiguous()
    return x, target, wet.to(torch.uint8).contiguous(), _weights(rng)


# ---------------------------------------------------------------- a user's program
def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        probs = _patches(case, seed)
        vols = [_volume(P) for P in probs]
        for vol, P in zip(vols, probs):
            vol.set_velocity(*P["faces"])
        return dict(case=case, vols=vols, scales=[P["scale"] for P in probs], k1s=[P["k1"] for P in probs])
    if kind == "train":
        x, target, wet, theta = _train_inputs(case, seed)
        net = Network()
        net.set_params(theta)
        return dict(case=case, net=net, x=x.view(torch.int16).reshape(-1), target=target.reshape(-1),
                    wet=wet.reshape(-1))
    P = _problem(case, seed)
    vol = _volume(P)
    state = dict(case=case, vol=vol, scale=P["scale"], k1=P["k1"])
    if kind == "step":
        vol.set_step_velocity(*P["faces"])
    else:
        vol.set_velocity(*P["faces"])
    if kind == "learned":
        state["net"] = Network()
        state["net"].load()
        state["net"].attach(vol)
    return state


def _fields(vol):
    return dict(p=vol.pressure(), u=vol.velocity_u(), v=vol.velocity_v(), w=vol.velocity_w())


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        project_batch(state["vols"], state["scales"], state["k1s"], MAX_ITERS, concurrency=8)
        return [_fields(v) for v in state["vols"]]
    if case["kind"] == "train":
        loss, grad = state["net"].loss_grad(state["x"], state["target"], state["wet"],
                                            (case["nx"], case["ny"], case["nz"]))
        return dict(loss=loss, grad=grad)
    vol = state["vol"]
    if case["kind"] == "step":
        vol.step_surface_mobile(STEP_US, MAX_ITERS)
        eta, roundoff = vol.surface()
        return dict(eta=eta, **_fields(vol))
    vol.project_mobile3(state["scale"], state["k1"], MAX_ITERS, warm=False)
    return _fields(vol)


# ---------------------------------------------------------------- 64 bits
class _System:
    """The projection's linear system of one geometry in float64: couplings
    of the three face directions, the ghost faces' part of the diagonal and
    of the right-hand side, and the gradient of the correction."""

    def __init__(self, P):
        dev = _dev()
        self.P = P
        nx, ny, nz = P["nx"], P["ny"], P["nz"]
        f64, f32 = torch.float64, torch.float32
        dx32 = torch.tensor(P["dx"], dtype=f32, device=dev)
        dx = float(np.float32(P["dx"]))
        self.dx, self.inv = dx, 1.0 / (dx * dx)
        level = P.get("label") is not None
        zc32 = (torch.arange(nz, device=dev, dtype=f32) + 0.5) * dx32
        zc = zc32.double()[:, None, None]
        shape = (nz, ny, nx)
        if level:
            label = torch.from_numpy(P["label"]).to(dev)
            phi = torch.from_numpy(P["phi"]).to(dev).double()
            solid, wet = label == _lib.LABEL_SOLID, label == _lib.LABEL_WATER
        else:
            solid = torch.zeros(shape, dtype=torch.bool, device=dev)
            if P["solid"] is not None:
                solid = torch.from_numpy(P["solid"]).to(dev) != 0
            eta32 = torch.from_numpy(np.ascontiguousarray(P["eta"])).to(dev)
            wet = ~solid & (zc32[:, None, None] < eta32[None])
            h = eta32.double()[None]
        dry = ~wet & ~solid
        cut = level or P["solid"] is not None or P["closed_lid"] or P.get("opens") is not None
        # apertures, walls included
        opens = P.get("opens")
        if opens is not None:
            ou, ov, ow = (torch.from_numpy(o).to(dev).double() for o in opens)
        else:
            ou, ov, ow = (torch.ones(s, dtype=f64, device=dev) for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)))
            if cut:
                for o, a in ((ou, 2), (ov, 1)):
                    o.select(a, 0).zero_()
                    o.select(a, -1).zero_()
                ow[0] = 0
                if P["closed_lid"]:
                    ow[-1] = 0
                if not level:
                    free = (~solid).double()
                    for o, a in ((ou, 2), (ov, 1), (ow, 0)):
                        n = o.shape[a]
                        o.narrow(a, 0, n - 1).mul_(free)
                        o.narrow(a, 1, n - 1).mul_(free)
        self.apertures = (ou, ov, ow) if cut else None
        self.solid, self.wet = solid, wet
        rho, g, rest = P["rho"], P["g"], P["rest"]
        zero = lambda: torch.zeros(shape, dtype=f64, device=dev)
        self.ghost_diag, self.ghost_rhs = zero(), zero()
        self.couple, self.gradient = [], []

        def theta(c, n, axis):
            """theta and ghost value of wet cells c against dry cells n of the same axis (slices)."""
            if level:
                fc, fa = phi[c], phi[n]
                t = (fc / (fc - fa)).clamp(min=0.01)
                return 1.0 / t, torch.zeros_like(t)
            hh = h.expand(shape)
            if axis == 0:
                t = ((hh[c] - zc.expand(shape)[c]) / dx).clamp(min=1e-3)
                val = rho * g * (hh[c] - rest)
            else:
                t = ((hh[c] - zc.expand(shape)[c]) / (hh[c] - hh[n])).clamp(min=1e-3)
                val = rho * g * (zc.expand(shape)[c] - rest)
            return 1.0 / t, torch.zeros_like(val) if P["homogeneous"] else val

        for axis, o in ((2, ou), (1, ov), (0, ow)):
            n = shape[axis]
            lo = tuple(slice(0, n - 1) if a == axis else slice(None) for a in range(3))
            hi = tuple(slice(1, n) if a == axis else slice(None) for a in range(3))
            inner = tuple(slice(1, n) if a == axis else slice(None) for a in range(3))
            ap = o[inner]
            usable = (ap != 0) & ~solid[lo] & ~solid[hi]
            both = usable & wet[lo] & wet[hi]
            self.couple.append((axis, lo, hi, torch.where(both, ap, torch.zeros_like(ap))))
            it_l, val_l = theta(lo, hi, axis)
            up = usable & wet[lo] & dry[hi]
            if axis == 0 and not level:
                down = torch.zeros_like(up)
                it_r, val_r = it_l, val_l
            else:
                it_r, val_r = theta(hi, lo, axis)
                down = usable & wet[hi] & dry[lo]
            for cell, where, it, val in ((lo, up, it_l, val_l), (hi, down, it_r, val_r)):
                d = torch.where(where, ap * it, torch.zeros_like(it))
                self.ghost_diag[cell] += d
                self.ghost_rhs[cell] += d * torch.where(where, val, torch.zeros_like(val))
            self.gradient.append((axis, lo, hi, inner, both, up, it_l, val_l, down, it_r, val_r))
        self.lid = None
        if not level:
            # the top face of a wet top cell
            c = (slice(nz - 1, nz),)
            t = ((h - zc[nz - 1]) / dx).clamp(min=1e-3)
            val = torch.zeros_like(t) if P["homogeneous"] else rho * g * (h - rest)
            where = wet[c] & (ow[nz:] != 0)
            d = torch.where(where, ow[nz:] / t, torch.zeros_like(t))
            self.ghost_diag[c] += d
            self.ghost_rhs[c] += d * val
            self.lid = (c, where, 1.0 / t, val)
        self.diag = self.ghost_diag.clone()
        for _, lo, hi, a in self.couple:
            self.diag[lo] += a
            self.diag[hi] += a
        self.active = wet & (self.diag > 0)

    def apply(self, x):
        y = self.diag * x
        for _, lo, hi, a in self.couple:
            y[lo] -= a * x[hi]
            y[hi] -= a * x[lo]
        return y

    def divergence(self, u, v, w):
        if self.apertures is not None:
            u, v, w = (o * f for o, f in zip(self.apertures, (u, v, w)))
        d = (u[:, :, 1:] - u[:, :, :-1] + v[:, 1:] - v[:, :-1] + w[1:] - w[:-1]) / self.dx
        return torch.where(self.solid, torch.zeros_like(d), d) if self.apertures is not None else d

    def solve(self, rhs):
        """Conjugate gradients with the diagonal, to 1e-13 of the right-hand side."""
        act = self.active
        b = torch.where(act, rhs, torch.zeros_like(rhs)) / self.inv
        neumann = not bool((self.ghost_diag != 0).any())
        count = int(act.sum())
        if neumann:
            b = torch.where(act, b - b.sum() / count, b)
        m = torch.where(act, 1.0 / self.diag.clamp(min=1e-300), torch.zeros_like(b))
        x, r = torch.zeros_like(b), b.clone()
        z = m * r
        d = z.clone()
        rz = (r * z).sum()
        goal = 1e-26 * float((b * b).sum())
        for it in range(20000):
            q = self.apply(d)
            alpha = rz / (d * q).sum()
            x += alpha * d
            r -= alpha * q
            z = m * r
            new = (r * z).sum()
            d.mul_(new / rz).add_(z)
            rz = new
            if it % 40 == 39 and not float((r * r).sum()) > goal:
                break
        if neumann:
            x = torch.where(act, x - x.sum() / count, x)
        return x

    def project(self, u, v, w):
        """(p, u, v, w) of predicted float64 faces."""
        P = self.P
        rhs = P["scale"] * self.divergence(u, v, w) + self.ghost_rhs * self.inv
        p = self.solve(torch.where(self.wet, rhs, torch.zeros_like(rhs)))
        out = [f.clone() for f in (u, v, w)]
        k1 = P["k1"] / self.dx
        for (axis, lo, hi, inner, both, up, it_l, val_l, down, it_r, val_r), f in zip(self.gradient, out):
            g = torch.where(both, p[hi] - p[lo], torch.zeros_like(it_l))
            g = torch.where(up, (val_l - p[lo]) * it_l, g)
            g = torch.where(down, (p[hi] - val_r) * it_r, g)
            f[inner] -= k1 * g
        if self.lid is not None:
            c, where, it, val = self.lid
            out[2][-1:] -= torch.where(where, k1 * (val - p[c]) * it, torch.zeros_like(it))
        return p, out


def _flat(p, faces):
    return dict(p=p.reshape(-1), **{n: f.reshape(-1) for n, f in zip("uvw", faces)})


def _advect(P, u, v, w):
    """The moving surface's predicted faces: central differences of each
    component along and across, closed and wall faces unchanged."""
    S = _System(P)
    dt, h = STEP_US * 1e-6, 0.5 / S.dx
    out = []
    f3 = (u, v, w)
    for c in range(3):
        f = f3[c]
        own = 2 - c  # array axis of the component's direction
        grad = []
        for axis in range(3):
            n = f.shape[axis]
            a = torch.cat([f.narrow(axis, 1, n - 1), f.narrow(axis, n - 1, 1)], axis)
            b = torch.cat([f.narrow(axis, 0, 1), f.narrow(axis, 0, n - 1)], axis)
            grad.append((a - b) * h)
        adv = f * grad[own]
        for o in range(3):
            if o == c:
                continue
            ax = 2 - o
            q = f3[o]
            # mean of the four faces of the other component about this face
            q = q.narrow(ax, 0, q.shape[ax] - 1) + q.narrow(ax, 1, q.shape[ax] - 1)
            mean = torch.zeros_like(f)
            m = q.shape[own]
            mean.narrow(own, 1, m - 1).copy_(0.25 * (q.narrow(own, 0, m - 1) + q.narrow(own, 1, m - 1)))
            adv = adv + mean * grad[ax]
        new = f - dt * adv
        n = f.shape[own]
        keep = S.apertures[c] == 0
        keep.narrow(own, 0, 1).fill_(True)
        keep.narrow(own, n - 1, 1).fill_(True)
        out.append(torch.where(keep, f, new))
    return S, out


def _step(P):
    u, v, w = (f.double() for f in P["faces"])
    S, pred = _advect(P, u, v, w)
    p, faces = S.project(*pred)
    nx, ny, nz = P["nx"], P["ny"], P["nz"]
    # extrapolation up the columns: the last solved face carried over the dry ones
    wet, solid = S.wet, S.solid
    u, v, w = faces
    solved_u, solved_v, solved_w = (torch.zeros(f.shape, dtype=torch.bool, device=f.device) for f in faces)
    either = lambda lo, hi: ~solid[lo] & ~solid[hi] & (wet[lo] | wet[hi])
    a = slice(None)
    solved_u[:, :, 1:-1] = either((a, a, slice(0, nx - 1)), (a, a, slice(1, nx)))
    solved_v[:, 1:-1] = either((a, slice(0, ny - 1)), (a, slice(1, ny)))
    solved_w[1:] = wet
    for c, (f, solved, o) in enumerate(((u, solved_u, S.apertures[0]), (v, solved_v, S.apertures[1]), (w, solved_w, S.apertures[2]))):
        last, have = torch.zeros_like(f[0]), torch.zeros_like(solved[0])
        for k in range(1 if c == 2 else 0, f.shape[0]):
            opened = o[k] != 0
            take = opened & solved[k]
            last, have = torch.where(take, f[k], last), have | take
            f[k] = torch.where(opened & ~solved[k] & have, last, f[k])
    # heights from the wetted discharges
    eta = torch.from_numpy(P["eta"]).to(u.device).double()
    dx, dt = S.dx, STEP_US * 1e-6
    flux = []
    for c, f in ((0, u), (1, v)):
        o = S.apertures[c]
        q = torch.zeros_like(f[0])
        surf = 0.5 * (eta[:, :-1] + eta[:, 1:]) if c == 0 else 0.5 * (eta[:-1] + eta[1:])
        for k in range(nz):
            wetted = ((surf - k * dx) / dx).clamp(0, 1)
            if c == 0:
                q[:, 1:-1] += (o[k] * f[k])[:, 1:-1] * dx * wetted
            else:
                q[1:-1] += (o[k] * f[k])[1:-1] * dx * wetted
        flux.append(q)
    eta = eta - dt / dx * (flux[0][:, 1:] - flux[0][:, :-1] + flux[1][1:] - flux[1][:-1])
    return dict(eta=eta.reshape(-1), **_flat(p, (u, v, w)))


def _network(theta, x):
    """The 3-level encoder-decoder in float64; x is channels first."""
    pad = torch.nn.functional.pad
    at = 0
    acts, h = {}, x
    names = ("e1a", "e1b", "e2a", "e2b", "e3a", "e3b", "d2a", "d2b", "d1a", "d1b", "head")
    for name, (_, ci, co) in zip(names, _layer_sizes()):
        W = theta[at: at + co * 27 * ci].reshape(co, 27, ci)
        b = theta[at + co * 27 * ci: at + co * 27 * ci + co]
        at += co * 27 * ci + co
        if name in ("e2a", "e3a"):
            c, z, y, q = h.shape
            h = h.reshape(c, z // 2, 2, y // 2, 2, q // 2, 2).mean((2, 4, 6))
        if name in ("d2a", "d1a"):
            h = h.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)
        _, nz, ny, nx = h.shape
        hp = pad(h, (1, 1, 1, 1, 1, 1))
        out = b[:, None].expand(co, nz * ny * nx)
        for t in range(27):
            z, y, q = t // 9, t // 3 % 3, t % 3
            out = out + W[:, t] @ hp[:, z: z + nz, y: y + ny, q: q + nx].reshape(ci, -1)
        out = out.reshape(co, nz, ny, nx)
        if name in ("d2a", "d1a"):
            out = out + acts["e2b" if name == "d2a" else "e1b"]
        h = out if name == "head" else torch.relu(out)
        acts[name] = h
    return h[0]


def _gradients(case, seed):
    x, target, wet, theta = _train_inputs(case, seed)
    t = torch.from_numpy(theta).to(x.device).double().requires_grad_(True)
    y = _network(t, x.double().permute(3, 0, 1, 2).contiguous())
    d = (y - target.double()) * wet
    loss = (d * d).sum() / max(int(wet.sum()), 1)
    loss.backward()
    return dict(loss=float(loss.detach()), grad=t.grad.detach().cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _gradients(case, seed)
    if kind == "batch":
        return [_flat(*_System(P).project(*(f.double() for f in P["faces"]))) for P in _patches(case, seed)]
    P = _problem(case, seed)
    if kind == "step":
        return _step(P)
    return _flat(*_System(P).project(*(f.double() for f in P["faces"])))
