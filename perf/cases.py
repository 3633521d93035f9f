"""The work that programs on this library have it do, as cases to be timed.

A case is a dict of plain values.  `prepare` makes what a program holds before
the call (a terrain or a batch with its state in device memory, a host
gradient, torch tensors), `run` is one pass through the public entry points,
`work` says what a pass cannot do without and `exact` gives its outputs in
64-bit torch arithmetic, without the library.

Kinds:
  grid       hg_step_grid: `steps` erosion steps on an n x n terrain whose
             state stays on the device; the planes are handed on as device
             buffers (hg_plane_device_ptr).
  frame      one step and the HEIGHT channel read back, what a host-side
             renderer does per frame.
  batch      `steps` steps of many uneven terrains from a captured graph, then
             the heights and water read back (making a data set).
  adjoint    hg_adjoint_rollout with host gradients.
  autograd   hydrogen.autograd.rollout, forward and backward.
  droplets   hg_step_particle on a resident terrain, and a snapshot of it (one
             tensor: single planes differ from run to run, since concurrent
             droplets meet in no fixed order).
  particles  hg_step_particle_reference, the reference's particle mode, and a
             snapshot of the terrain and its water.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "hydro-gen_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hydrogen as hg  # noqa: E402
from hydrogen import autograd as hg_autograd  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
STATE = ("rock", "dirt", "water", "flux_l", "flux_r", "flux_t", "flux_b", "sed_rock", "sed_dirt")
WARM = 3            # steps that give a new terrain its running water before the timed work

# Coefficients: the benchmark's, and the reference's own grid defaults.
BENCH = dict(Kc=0.05, Ks=(0.02, 0.02), Kd=(0.02, 0.02), Ke=0.01, Kalpha=(math.radians(35.0),) * 2,
             Kspeed=(0.1, 0.1), G=9.81, dt=0.005, Kconv=0.001, E=1.0)
REFERENCE = dict(Kc=0.2, Ks=(0.03, 0.09), Kd=(0.01, 0.03), Ke=0.03, Kalpha=(1.3, 0.6), Kspeed=(0.5, 2.0),
                 G=1.0, dt=0.001, Kconv=0.001, E=1.0)


def listed() -> list:
    return [
        # one step per call on the smallest map in the tests: an interactive
        # preview, where launches and latency are everything
        dict(name="grid-64", kind="grid", n=64, steps=1, coef="bench", rain="uniform", tune=False),
        # the plain 512^2 configuration, a few steps per call
        dict(name="grid-512", kind="grid", n=512, steps=8, coef="bench", rain="uniform", tune=False),
        # a side that no tile width divides, the reference's coefficients, rain off
        dict(name="grid-1000", kind="grid", n=1000, steps=4, coef="reference", rain="off", tune=False),
        # the reference's default map size
        dict(name="grid-1024", kind="grid", n=1024, steps=16, coef="bench", rain="uniform", tune=False),
        # the headline size, tiles tuned beforehand as the benchmark does
        dict(name="grid-4096", kind="grid", n=4096, steps=4, coef="bench", rain="uniform", tune=True),
        # a host-side renderer's frame at the default map size
        dict(name="frame-1024", kind="frame", n=1024, steps=1, coef="bench", rain="constant", tune=False),
        # uneven terrains with their own coefficients, the batched configuration's sides
        dict(name="batch-20", kind="batch", count=20, smallest=256, largest=2048, steps=96),
        # the differentiable-rollout configuration, two checkpoint segments of it
        dict(name="adjoint-1024", kind="adjoint", n=1024, steps=32, k_ckpt=16),
        # an optimiser's step on a small map, through torch
        dict(name="autograd-256", kind="autograd", n=256, steps=32, k_ckpt=16),
        # the particle configuration's size: 2^20 droplets of 64 steps
        dict(name="droplets-2048", kind="droplets", n=2048, count=1 << 20, life=64, passes=False),
        # a small map with few droplets, thermal and smoothing after each iteration
        dict(name="droplets-512", kind="droplets", n=512, count=20000, life=30, passes=True),
        # the reference's particle mode with its default particle count
        dict(name="particles-2048", kind="particles", n=2048, count=262144, steps=4),
    ]


def _log(rng, lo: float, hi: float) -> float:
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _side(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, 8 * round(_log(rng, lo, hi) / 8)))


def draw(rng) -> dict:
    kind = rng.choice(["grid"] * 5 + ["frame", "batch", "adjoint", "autograd", "droplets", "particles"])
    if kind == "grid":
        n = _side(rng, 64, 4096)
        return dict(kind=kind, n=n, steps=max(1, min(rng.randint(1, 32), (4 * 4096 * 4096) // (n * n))),
                    coef=rng.choice(["bench", "bench", "reference"]),
                    rain=rng.choice(["uniform", "uniform", "constant", "off"]), tune=n >= 2048 and rng.random() < 0.5)
    if kind == "frame":
        return dict(kind=kind, n=_side(rng, 128, 2048), steps=rng.randint(1, 4), coef=rng.choice(["bench", "reference"]),
                    rain=rng.choice(["uniform", "constant"]), tune=False)
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 20), smallest=_side(rng, 64, 256), largest=_side(rng, 512, 2048),
                    steps=2 * rng.randint(4, 48))
    if kind == "adjoint":
        return dict(kind=kind, n=_side(rng, 128, 1024), steps=rng.randint(5, 32), k_ckpt=rng.choice([4, 8, 16, 32]))
    if kind == "autograd":
        return dict(kind=kind, n=_side(rng, 64, 512), steps=rng.randint(4, 32), k_ckpt=rng.choice([8, 16]))
    if kind == "droplets":
        return dict(kind=kind, n=_side(rng, 256, 2048), count=int(_log(rng, 4096, 1 << 20)), life=rng.randint(20, 64),
                    passes=rng.random() < 0.5)
    return dict(kind=kind, n=_side(rng, 256, 2048), count=int(_log(rng, 8192, 262144)), steps=rng.randint(1, 8))


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------

def _noise(n: int, wave: float, gen: torch.Generator, octaves: int = 6) -> torch.Tensor:
    """fBm of bicubic lattice noise in [0, 1], features of about `wave` cells."""
    out = torch.zeros(n, n, dtype=torch.float32, device=DEV)
    for o in range(octaves):
        m = max(2, round(n / wave * 2 ** o)) + 1
        if m > n:
            break
        g = torch.rand(1, 1, m, m, generator=gen, dtype=torch.float32).to(DEV)
        out += 0.5 ** o * F.interpolate(g, size=(n, n), mode="bicubic", align_corners=True)[0, 0]
    lo, hi = out.min(), out.max()
    return (out - lo) / (hi - lo)


def _terrain_planes(n: int, seed: int, coef: dict, rain: str, dtype=torch.float32) -> torch.Tensor:
    """The 9 state planes of an n x n terrain some steps into an erosion run."""
    gen = torch.Generator().manual_seed(int(seed) * 7919 + n)
    wave = min(1024.0, max(32.0, n / 4))
    st = torch.zeros(9, n, n, dtype=torch.float64, device=DEV)
    st[0] = _noise(n, wave, gen).double() * (wave / 2)
    st[1] = (_noise(n, wave / 2, gen).double() * 3.0 - 1.0).clamp_min(0.0)
    st[2] = (_noise(n, wave, gen).double() - 0.5).clamp_min(0.0) * 0.4 + 0.01
    st = st.float().double()
    p = _coef64(coef)
    for s in range(WARM):
        st = torch.stack(_step64(list(st), p, _rain64(n, rain, 0.02, seed, s)))
    return st.to(dtype)


def _heights(n: int, seed: int, hi: float) -> torch.Tensor:
    gen = torch.Generator().manual_seed(int(seed) * 7919 + n)
    return (_noise(n, min(512.0, max(32.0, n / 4)), gen) * hi).float()


def _settings(coef: dict):
    s = hg.erosion_settings(Kc=coef["Kc"], Ke=coef["Ke"], G=coef["G"], dt=coef["dt"], Kconv=coef["Kconv"], E=coef["E"])
    for f in ("Ks", "Kd", "Kalpha", "Kspeed"):
        for layer in range(2):
            getattr(s, f)[layer] = coef[f][layer]
    return s


RAIN = {"off": hg.RAIN_OFF, "constant": hg.RAIN_CONSTANT, "uniform": hg.RAIN_UNIFORM}


def _coef(case: dict) -> dict:
    return REFERENCE if case.get("coef") == "reference" else BENCH


def _terrain(n: int, coef: dict, rain: str, seed: int, planes: torch.Tensor | None, step: int) -> "hg.Terrain":
    t = hg.Terrain(n)
    t.set_erosion(_settings(coef))
    t.set_rain(RAIN[rain], amount=0.02, seed=int(seed))
    if planes is not None:
        t.write_state(planes.cpu().numpy())
    t.step = step
    return t


class _Buffer:
    """A plane of a terrain in device memory, for torch.as_tensor; keeps the
    terrain alive as long as the tensor."""

    def __init__(self, terrain, ptr: int):
        self.terrain = terrain
        self.__cuda_array_interface__ = {"shape": (terrain.n, terrain.n), "typestr": "<f4", "data": (ptr, False),
                                         "version": 2, "strides": None}


def _planes(state: dict, which) -> dict:
    """The current device buffers of the planes, as tensors (each buffer is
    wrapped the first time it is met)."""
    t, known, out = state["terrain"], state["views"], {}
    for name, p in which:
        ptr = t.device_ptr(p)
        v = known.get(ptr)
        if v is None:
            v = known[ptr] = torch.as_tensor(_Buffer(t, ptr), device=DEV)
        out[name] = v
    return out


def _snapshot(state: dict, which) -> torch.Tensor:
    """The planes stacked into one tensor, copied on the terrain's own stream."""
    planes = _planes(state, which)
    if "stream" not in state:
        state["stream"] = torch.cuda.ExternalStream(state["terrain"].stream())
    with torch.cuda.stream(state["stream"]):
        return torch.stack(tuple(planes.values()))


ALL_PLANES = tuple((name, p) for p, name in enumerate(STATE))
HEIGHTS = ALL_PLANES[:2]
SURFACE = ALL_PLANES[:3]


def _sides(case: dict) -> list:
    """The batch's sides: multiples of 8 from smallest to largest, spread by
    their logarithm and dealt out of order as a user's terrains come."""
    c, lo, hi = case["count"], case["smallest"], case["largest"]
    s = [8 * round(lo * (hi / lo) ** (((i * 7) % c) / max(1, c - 1)) / 8) for i in range(c)]
    return [max(lo, min(hi, v)) for v in s]


def _batch_coef(case: dict, seed: int) -> list:
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["count"]):
        ks, kd, a = float(rng.uniform(0.01, 0.05)), float(rng.uniform(0.01, 0.05)), math.radians(rng.uniform(30, 45))
        out.append(dict(BENCH, Kc=float(rng.uniform(0.02, 0.1)), Ks=(ks, ks), Kd=(kd, kd),
                        Ke=float(rng.uniform(0.005, 0.02)), Kalpha=(a, a)))
    return out


def _loss_gradient(n: int, seed: int) -> torch.Tensor:
    """Gradient of a mean squared height error with respect to the heights."""
    gen = torch.Generator().manual_seed(int(seed) * 104729 + n)
    return ((_noise(n, max(16.0, n / 8), gen) - 0.5) * (2.0 / (n * n))).float()


def prepare(case: dict, seed: int) -> dict:
    kind, st = case["kind"], {"case": case, "views": {}}
    if kind in ("grid", "frame"):
        coef = _coef(case)
        planes = _terrain_planes(case["n"], seed, coef, case["rain"])
        st["terrain"] = _terrain(case["n"], coef, case["rain"], seed, planes, WARM)
        if case["tune"]:
            st["terrain"].autotune()
    elif kind == "batch":
        sides, coefs = _sides(case), _batch_coef(case, seed)
        b = st["batch"] = hg.Batch(sides)
        b.set_rain(hg.RAIN_UNIFORM, amount=0.02, seed=int(seed))
        for i, n in enumerate(sides):
            b.set_erosion(_settings(coefs[i]), terrain=i)
            b.write_state(i, _terrain_planes(n, seed + i, coefs[i], "uniform").cpu().numpy())
        b.autotune()
        b.capture(case["steps"])
    elif kind == "adjoint":
        st["planes"] = _terrain_planes(case["n"], seed, BENCH, "constant").cpu().numpy()
        st["terrain"] = _terrain(case["n"], BENCH, "constant", seed, None, 0)
        st["gradient"] = _loss_gradient(case["n"], seed).cpu().numpy()
    elif kind == "autograd":
        n = case["n"]
        st["terrain"] = _terrain(n, BENCH, "constant", seed, None, 0)
        st["h0"] = _heights(n, seed, 32.0).requires_grad_(True)
        st["coef"] = torch.tensor([0.05, 0.02, 0.02, 0.01], device=DEV, requires_grad=True)
        st["gradient"] = _loss_gradient(n, seed)
    elif kind == "droplets":
        n = case["n"]
        planes = torch.zeros(2, n, n, dtype=torch.float32, device=DEV)
        planes[0] = _heights(n, seed, min(128.0, n / 16))
        st["terrain"] = t = _terrain(n, BENCH, "off", seed, planes, 0)
        # light strokes: at the default strength two runs of the same droplets
        # end up on visibly different terrains
        t.set_droplets(hg.droplet_settings(count=case["count"], max_lifetime=case["life"], capacity=1.0, erosion=0.05,
                                           deposition=0.05, seed=int(seed)))
    else:
        n = case["n"]
        t = st["terrain"] = hg.Terrain(n)
        t.write_plane(hg.P_ROCK, _heights(n, seed, min(256.0, n / 8)).cpu().numpy())
        t.set_erosion(hg.reference_particle_settings(case["count"]))
        t.ref_particles_init(case["count"])
        t.dispatch_particle_reference(2, True, float(seed % 1000), 1.0 / 60)
        st["time"] = float(seed % 1000) + 2.0 / 60
    if "terrain" in st:
        st["terrain"].sync()
    return st


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "grid":
        state["terrain"].dispatch_grid(case["steps"])
        return _planes(state, ALL_PLANES)
    if kind == "frame":
        t = state["terrain"]
        t.dispatch_grid(case["steps"])
        return t.read(hg.CH_HEIGHT)
    if kind == "batch":
        b = state["batch"]
        b.run()
        return [b.read_plane(i, p) for i in range(len(b.sizes)) for p in (hg.P_ROCK, hg.P_DIRT, hg.P_WATER)]
    if kind == "adjoint":
        t = state["terrain"]
        t.write_state(state["planes"])
        t.step = WARM
        grad_h0, grad_coef = t.adjoint_rollout(case["steps"], case["k_ckpt"], state["gradient"])
        return {"grad_h0": grad_h0, "grad_coef": grad_coef, **_planes(state, ALL_PLANES)}
    if kind == "autograd":
        h0, coef = state["h0"], state["coef"]
        h = hg_autograd.rollout(h0, coef, state["terrain"], case["steps"], case["k_ckpt"])
        grads = torch.autograd.grad(h, (h0, coef), state["gradient"])
        return {"height": h.detach(), "grad_h0": grads[0], "grad_coef": grads[1]}
    if kind == "droplets":
        state["terrain"].dispatch_particle(1, hg.STEP_THERMAL | hg.STEP_SMOOTH if case["passes"] else 0)
        return _snapshot(state, HEIGHTS)
    state["terrain"].dispatch_particle_reference(case["steps"], True, state["time"], 1.0 / 60)
    state["time"] += case["steps"] / 60.0
    return _snapshot(state, SURFACE)


def work(case: dict) -> dict:
    """Bytes and FP32 operations of a pass.  A step reads and writes the 9
    planes (72 B per cell) and takes about 330 operations per cell; its
    adjoint reads the step's start state and the adjoint planes and writes the
    latter (108 B), at about three times the operations."""
    kind = case["kind"]
    if kind in ("grid", "frame"):
        c = case["n"] ** 2
        return {"bytes": 72.0 * c * case["steps"] + (16.0 * c if kind == "frame" else 0.0), "flops": 330.0 * c * case["steps"]}
    if kind == "batch":
        c = sum(n * n for n in _sides(case))
        return {"bytes": 72.0 * c * case["steps"] + 12.0 * c, "flops": 330.0 * c * case["steps"]}
    if kind in ("adjoint", "autograd"):
        c = case["n"] ** 2
        return {"bytes": 180.0 * c * case["steps"] + 8.0 * c, "flops": 1320.0 * c * case["steps"]}
    if kind == "droplets":
        # about 100 operations per droplet step and 6 per cell of the 29-cell brush
        return {"bytes": 16.0 * case["n"] ** 2 * (2 if case["passes"] else 1),
                "flops": 274.0 * case["count"] * case["life"] + (220.0 * case["n"] ** 2 if case["passes"] else 0.0)}
    # 96 B per particle; heights, water and momentum map read and written
    return {"bytes": (96.0 * case["count"] + (16.0 + 40.0) * case["n"] ** 2) * case["steps"],
            "flops": (500.0 * case["count"] + 230.0 * case["n"] ** 2) * case["steps"]}


# ---------------------------------------------------------------------------
# the erosion step in 64 bits, differentiable by torch
# ---------------------------------------------------------------------------

def _coef64(coef: dict) -> dict:
    f = lambda v: float(np.float32(v))  # noqa: E731
    return {k: tuple(f(x) for x in v) if isinstance(v, tuple) else f(v) for k, v in coef.items()}


def _rain64(n: int, rain: str, amount: float, seed: int, step: int, terrain: int = 0):
    """What rain adds in one step: a number, or n x n uniform draws of Philox4x32-10."""
    a = float(np.float32(amount))
    if rain != "uniform":
        return a if rain == "constant" else 0.0
    m32 = 0xFFFFFFFF
    quads = (n + 3) // 4
    c0 = torch.arange(quads, dtype=torch.int64, device=DEV).expand(n, quads)
    c1 = torch.arange(n, dtype=torch.int64, device=DEV)[:, None].expand(n, quads)
    c2 = torch.full((n, quads), int(step), dtype=torch.int64, device=DEV)
    c3 = torch.full((n, quads), int(terrain), dtype=torch.int64, device=DEV)
    k0, k1 = int(seed) & m32, (int(seed) >> 32) & m32

    def mul(m, c):          # high and low words of a 32 x 32 bit product
        lo, hi = m * (c & 0xFFFF), m * (c >> 16)
        return (hi + (lo >> 16)) >> 16, (((hi & 0xFFFF) << 16) + lo) & m32

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    words = torch.stack((c0, c1, c2, c3), dim=-1).reshape(n, 4 * quads)[:, :n]
    return a * ((words >> 8).double() / 16777216.0)


OOB = float(np.float32(999999999999.0))
DIRS = ((-1, 0), (1, 0), (0, 1), (0, -1), (-1, 1), (1, 1), (-1, -1), (1, -1))   # L R T B LT RT LB RB


def _around(a: torch.Tensor, fill: float, count: int) -> list:
    n = a.shape[0]
    p = F.pad(a, (1, 1, 1, 1), value=fill)
    return [p[1 + dy:1 + dy + n, 1 + dx:1 + dx + n] for dx, dy in DIRS[:count]]


def _layer_thermal(total, height, layer, p):
    """Height change of one layer: each cell sends g * D towards the neighbours
    it stands above by more than the talus angle."""
    ta = math.tan(p["Kalpha"][layer])
    thr = [ta] * 4 + [math.sqrt(2.0) * ta] * 4
    D = [total - q for q in _around(total, 2 * OOB, 8)]
    zero = torch.zeros_like(total)
    bk = sum(torch.where(D[k] > thr[k], D[k], zero) for k in range(8))
    mc = torch.maximum(torch.maximum(D[0], D[1]), torch.maximum(D[2], D[3]))
    md = torch.maximum(torch.maximum(D[4], D[5]), torch.maximum(D[6], D[7]))
    some = bk > 0
    H = torch.minimum(height, torch.relu(torch.maximum(mc, md)))
    rmax = torch.where(some, torch.maximum(mc, md * math.sqrt(0.5)), zero)
    sharp = 1.0 + torch.relu(torch.atan(rmax) - p["Kalpha"][layer])
    S = (p["dt"] * p["Kspeed"][layer] * 0.5) * sharp ** 3 * H
    g = torch.where(some, S / torch.where(some, bk, torch.ones_like(bk)), zero)
    gn = _around(g, 0.0, 8)
    change = zero
    for k in range(8):
        change = change - D[k] * torch.where(D[k] > thr[k], g, torch.where(-D[k] > thr[k], gn[k], zero))
    return change


def _smooth64(r, d, m):
    if r.shape[0] < 3:
        return r, d
    lr, rr, tr, br = (q[1:-1, 1:-1] for q in _around(r, 0.0, 4))
    lg, rg, tg, bg = (q[1:-1, 1:-1] for q in _around(d, 0.0, 4))
    r0, d0 = r[1:-1, 1:-1], d[1:-1, 1:-1]

    def extremum(a, b, c, e):
        h = ((a + b + c + e) * 0.25).abs()
        return (((-a > h) | (-b > h)) & (a * b > 0)) | (((-c > h) | (-e > h)) & (c * e > 0))

    dl, dr, dt, db = r0 - lr, r0 - rr, r0 - tr, r0 - br
    er = extremum(dl, dr, dt, db)
    eg = extremum(d0 - lg + dl, d0 - rg + dr, d0 - tg + dt, d0 - bg + db)
    nr = torch.where(er, r0 + m * ((r0 + lr + rr + tr + br) * 0.2 - r0), r0)
    nd = torch.where(eg, d0 + m * ((d0 + lg + rg + tg + bg) * 0.2 - d0), d0)

    def inner(a, v):
        return torch.cat((a[:1], torch.cat((a[1:-1, :1], v, a[1:-1, -1:]), 1), a[-1:]), 0)

    return inner(r, nr), inner(d, nd)


def _step64(st, p, rain):
    """One step of the virtual-pipe model, both thermal layers and smoothing."""
    r, d, b, fl, fr, ft, fb, s0, s1 = st
    n, dt = r.shape[0], p["dt"]
    zero, one = torch.zeros_like(r), torch.ones_like(r)
    b = b + rain
    # outflow flux; the map's edge is a wall
    w = r + d + b
    old = (fl, fr, ft, fb)
    f = [torch.relu(p["E"] * old[i] + dt * p["G"] * (w - q)) for i, q in enumerate(_around(w, OOB, 4))]
    fin = (_around(fr, 0.0, 4)[0], _around(fl, 0.0, 4)[1], _around(fb, 0.0, 4)[2], _around(ft, 0.0, 4)[3])
    out = f[0] + f[1] + f[2] + f[3]
    some = out > 0
    q = torch.where(some, b / torch.where(some, out * dt, one), one)
    K = torch.where(q < 1, q, one)
    f = [x * K for x in f]
    d2 = torch.relu(b + dt * (fin[0] + fin[1] + fin[2] + fin[3] - out * K))
    depth = b + d2
    wet = depth > 0
    inv = torch.where(wet, 1.0 / torch.where(wet, depth, one), zero)
    vx = (fin[0] - fl + fr - fin[1]) * inv
    vy = (fin[3] - fb + ft - fin[2]) * inv
    # dissolving and deposition
    v2 = vx * vx + vy * vy
    moving = v2 > 0
    ero = torch.where(moving, torch.sqrt(torch.where(moving, v2, one)), zero)
    t = ((torch.clamp_min(depth, 5e-4) - 1e-3) / (5e-4 - 1e-3)).clamp(0.0, 1.0)
    ero = torch.where(depth < 1e-3, ero * (1.0 - t * t * (3.0 - 2.0 * t)), ero)
    hl, hr, ht, hb = _around(r + d, 0.0, 4)
    g2 = (hr - hl) ** 2 + (ht - hb) ** 2
    steep = g2 > 0
    sin_a = torch.where(steep, torch.sqrt(torch.where(steep, g2, one) / (g2 + 4.0)), zero)
    cap = p["Kc"] * torch.clamp_min(sin_a, float(np.float32(0.02))) * ero

    def layer(h, s, c, Ks, Kd):
        take = c > s
        a = torch.where(take, dt * Ks * (c - s), -dt * Kd * (s - c))
        h1, sd = h - a, s + a
        empty = take & (h1 < 0)
        return torch.where(empty, zero, h1), torch.where(empty, sd + h1, sd), take & ~empty, empty

    c1 = torch.relu(cap)
    dn, s1n, stop, empty = layer(d, s1, c1, p["Ks"][1], p["Kd"][1])
    c0 = torch.relu(cap - torch.where(empty, d, zero))
    rn, s0n, _, _ = layer(r, s0, c0, p["Ks"][0], p["Kd"][0])
    r, s0 = torch.where(stop, r, rn), torch.where(stop, s0, s0n)
    d = dn
    conv = s0 * (p["Kconv"] * dt)
    s1, s0 = s1n + conv, s0 - conv
    # semi-Lagrangian transport of the sediment
    x = torch.arange(n, dtype=r.dtype, device=r.device)
    px, py = (x[None, :] - vx * dt).clamp(0.0, n - 1.0), (x[:, None] - vy * dt).clamp(0.0, n - 1.0)
    ix, iy = px.detach().long(), py.detach().long()
    ax, ay = px - ix, py - iy
    ix1, iy1 = torch.clamp_max(ix + 1, n - 1), torch.clamp_max(iy + 1, n - 1)

    def sample(s):
        s = s.reshape(-1)
        top = s[iy * n + ix] * (1 - ax) + s[iy * n + ix1] * ax
        return top * (1 - ay) + (s[iy1 * n + ix] * (1 - ax) + s[iy1 * n + ix1] * ax) * ay

    s0, s1 = sample(s0), sample(s1)
    b = d2 * (1.0 - p["Ke"] * dt)
    # slippage of both layers, smoothing
    r = r + _layer_thermal(r, r, 0, p)
    d = d + _layer_thermal(r + d, d, 1, p)
    r, d = _smooth64(r, d, min(1.0, max(0.0, p["Kspeed"][1] * dt)))
    return [r, d, b, f[0], f[1], f[2], f[3], s0, s1]


def _forward64(st, p, n, rain, amount, seed, step, steps, terrain=0):
    for s in range(steps):
        st = _step64(st, p, _rain64(n, rain, amount, seed, step + s, terrain))
    return st


def _gradient64(st, p, case, rain_amount, grad):
    """Heights after the rollout and the gradients with respect to the initial
    rock and to (Kc, Ks, Kd, Ke), step by step from kept start states."""
    steps, kept = case["steps"], []
    with torch.no_grad():
        for s in range(steps):
            kept.append(st)
            st = _step64(st, p, rain_amount)
    final = st
    lam = [grad, grad] + [torch.zeros_like(grad) for _ in range(7)]
    total = torch.zeros(4, dtype=torch.float64, device=DEV)
    for s in reversed(range(steps)):
        x = [v.detach().requires_grad_(True) for v in kept.pop()]
        c = torch.tensor([p["Kc"], p["Ks"][0], p["Kd"][0], p["Ke"]], dtype=torch.float64, device=DEV, requires_grad=True)
        q = dict(p, Kc=c[0], Ks=(c[1], c[1]), Kd=(c[2], c[2]), Ke=c[3])
        g = torch.autograd.grad(_step64(x, q, rain_amount), x + [c], lam, allow_unused=True)
        lam = [torch.zeros_like(v) if e is None else e for v, e in zip(x, g[:9])]
        total += g[9]
    return final, lam[0], total


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("droplets", "particles"):
        return None           # the outcome depends on the order in which concurrent particles meet
    if kind == "batch":
        out = []
        for i, (n, coef) in enumerate(zip(_sides(case), _batch_coef(case, seed))):
            st = list(_terrain_planes(n, seed + i, coef, "uniform").double())
            out += _forward64(st, _coef64(coef), n, "uniform", 0.02, seed, 0, case["steps"], i)[:3]
        return out
    n = case["n"]
    if kind in ("grid", "frame"):
        coef = _coef(case)
        st = list(_terrain_planes(n, seed, coef, case["rain"]).double())
        st = _forward64(st, _coef64(coef), n, case["rain"], 0.02, seed, WARM, case["steps"])
        if kind == "grid":
            return dict(zip(STATE, st))
        return torch.stack((st[0], st[1], st[2], st[0] + st[1] + st[2]), dim=-1)
    p, grad = _coef64(BENCH), _loss_gradient(n, seed).double()
    rain = _rain64(n, "constant", 0.02, seed, 0)
    if kind == "adjoint":
        st = list(_terrain_planes(n, seed, BENCH, "constant").double())
        st, g, c = _gradient64(st, p, case, rain, grad)
        return {"grad_h0": g, "grad_coef": c, **dict(zip(STATE, st))}
    st = [torch.zeros(n, n, dtype=torch.float64, device=DEV) for _ in range(9)]
    st[0] = _heights(n, seed, 32.0).double()
    st, g, c = _gradient64(st, p, case, rain, grad)
    return {"height": st[0] + st[1], "grad_h0": g, "grad_coef": c}
