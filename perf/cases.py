"""Cases for timing this framework through its public entry points.

Four kinds of call:
  frames   a rollout from a given state: reset to positions, set velocities,
           step `frames` times, read the state back (ADMMBackendHIP)
  detect   one collision detection on host positions and its contact list
           (CollisionDetector)
  forward  warm-start network inference on host rows (MLP.forward)
  train    warm-start network training from given weights (MLP.train)

Scenes are the package's own generated ones with the settings of
parallel_admm_amd.configs.  A program builds a scene's backend or detector once
(the factorization is part of it) and then feeds it states, so handles are kept
per scene here and a prepared state is positions and velocities for one.

A pass sets the whole state of its handle before it computes, so states that
share a handle do not see each other.  Frames (positions and velocities, the
state a step hands on) are returned in single precision, as a renderer or a
training set takes them: inside a step only displacements are held in FP32, so
positions agree to about 1e-9 and velocities to about 1e-7.
"""
from __future__ import annotations

import functools
import math

import numpy as np

import parallel_admm_amd as pa
from parallel_admm_amd.configs import config_for, folded_flap_state
from parallel_admm_amd.warm_start import DEFAULT_MODEL, Model


def listed():
    return [
        # the smallest batch member (side 16 cloth draped over its sphere) alone: every launch is latency
        dict(name="frames-member16", kind="frames", scene="member", side=16, radius=0.1, precond=2, frames=2),
        # the 32 x 32 pinned cloth in free fall, no contact found: detection, local and global phases of a small scene
        dict(name="frames-cloth32-fall", kind="frames", scene="cloth32", frames=2),
        # the largest batch member alone, odd side, with contact
        dict(name="frames-member95", kind="frames", scene="member", side=95, radius=0.3, precond=2, frames=1),
        # a batch member with the AMG-preconditioned CG, the solver that AdmmConfig selects by default
        dict(name="frames-member64-amg", kind="frames", scene="member", side=64, radius=0.2, precond=1, frames=1),
        # the 20^3-cell tet box landing on the ground: tetrahedra, few large fronts
        dict(name="frames-tetbox", kind="frames", scene="tetbox", frames=1),
        # the 256 x 256 cloth landing on its sphere to residual 1e-4: the benchmark's own step
        dict(name="frames-cloth256", kind="frames", scene="cloth256", cols=0, frames=1),
        # the same cloth with a small flap folded over it: some 1e4 contacts
        dict(name="frames-cloth256-fold3", kind="frames", scene="cloth256", cols=3, frames=1),
        # the same with the 24-column flap: about 1e5 contacts
        dict(name="frames-cloth256-flap24", kind="frames", scene="cloth256", cols=24, frames=1),
        # uneven members merged into one batch
        dict(name="frames-batch160", kind="frames", scene="batch", count=160, scene_seed=1, frames=1),
        # the detector alone: a small scene, and the folded cloth
        dict(name="detect-member33", kind="detect", scene="member", side=33, radius=0.2, precond=2),
        dict(name="detect-cloth256-fold3", kind="detect", scene="cloth256", cols=3),
        # training the warm-start network
        dict(name="train-65536", kind="train", rows=65536, batch=8192, epochs=4),
    ]


def draw(rng):
    kind = rng.choice(["member", "member", "cloth256", "batch", "cloth32", "tetbox", "detect", "detect", "forward", "train"])
    side = int(round(math.exp(rng.uniform(math.log(16), math.log(96)))))
    member = dict(scene="member", side=side, radius=round(rng.uniform(0.1, 0.3), 3), precond=rng.choice([2, 2, 1]))
    cloth = dict(scene="cloth256", cols=rng.randint(0, 24))
    if kind == "member":
        return dict(kind="frames", frames=rng.randint(1, 2), **member)
    if kind == "cloth256":
        return dict(kind="frames", frames=1, **cloth)
    if kind == "batch":
        return dict(kind="frames", scene="batch", count=int(round(math.exp(rng.uniform(math.log(3), math.log(160))))),
                    scene_seed=rng.randint(2, 10 ** 6), frames=1)
    if kind == "cloth32":
        return dict(kind="frames", scene="cloth32", frames=rng.randint(1, 12))
    if kind == "tetbox":
        return dict(kind="frames", scene="tetbox", frames=rng.randint(1, 2), tilt=round(rng.uniform(0.0, 0.01), 4))
    if kind == "detect":
        return dict(kind="detect", **rng.choice([member, cloth]))
    rows = int(round(math.exp(rng.uniform(math.log(100), math.log(131072)))))
    if kind == "forward":
        return dict(kind="forward", rows=rows)
    return dict(kind="train", rows=max(rows, 1000), batch=rng.choice([1024, 4096, 8192]), epochs=rng.randint(1, 4))


# ---------------------------------------------------------------------------
# scenes and handles
# ---------------------------------------------------------------------------
def _members(case):
    """(side, radius) of every cloth of the case."""
    if case["scene"] == "member":
        return [(case["side"], case["radius"])]
    rng = np.random.default_rng(case["scene_seed"])
    return [(int(rng.integers(16, 97)), float(rng.uniform(0.1, 0.3))) for _ in range(case["count"])]


def _scene_key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "kind", "frames", "cols", "tilt")))


@functools.lru_cache(maxsize=4)
def _scene(key):
    case = dict(key)
    if case["scene"] == "cloth32":
        return pa.Scene.generate(1)
    if case["scene"] == "tetbox":
        return pa.Scene.generate(2, seed=7)
    if case["scene"] == "cloth256":
        return pa.Scene.generate(3)
    parts = [pa.Scene.generate(4, side=s, radius=r) for s, r in _members(case)]
    return parts[0] if case["scene"] == "member" else pa.Scene.merge(parts)


def _config(case):
    cfg = config_for("batch" if case["scene"] in ("member", "batch") else case["scene"])
    cfg.precond = case.get("precond", cfg.precond)
    if case["scene"] == "cloth256":
        cfg.residual_tol = 1e-4  # as the benchmark runs it; the others run their fixed iteration count
    if case["scene"] == "batch":
        cfg.max_contacts = 1 << 20
    return cfg


@functools.lru_cache(maxsize=16)
def _backend(key):
    case = dict(key)
    b = pa.ADMMBackendHIP.from_scene(_scene(key), _config(case))
    b.set_sync_to_host(False)
    return b


@functools.lru_cache(maxsize=8)
def _detector(key):
    cfg = _config(dict(key))
    return pa.CollisionDetector.for_scene(_scene(key), cfg.max_contacts, cfg.thickness)


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
def _ripple(rng, x, amp, cycles=2.0):
    """A smooth random vector field over x: a few plane waves of `cycles` per extent."""
    ext = max(float(np.ptp(x, axis=0).max()), 1e-9)
    out = np.zeros_like(x)
    for _ in range(4):
        k = rng.normal(size=3) * 2 * np.pi * cycles / (2 * ext)
        out += rng.normal(size=3) * np.sin(x @ k + rng.uniform(0, 2 * np.pi))[:, None]
    return amp * out / 2


def _drape(rng, x, radius, gap):
    """A flat cloth over the sphere of `radius` at the origin, wrapped around
    its top to 0.3 rad and straight beyond; velocities: hanging part falling."""
    c = 0.5 * (x.min(axis=0) + x.max(axis=0))
    d = x - c
    rho = np.hypot(d[:, 0], d[:, 2])
    r = radius + gap
    th = np.minimum(rho / r, 0.3)
    rest = rho - r * th
    rad = r * np.sin(th) + rest * np.cos(th)
    y = r * np.cos(th) - rest * np.sin(th)
    s = np.where(rho > 0, rad / np.maximum(rho, 1e-300), 1.0)
    out = np.stack([d[:, 0] * s, y, d[:, 2] * s], axis=1)
    v = _ripple(rng, out, 0.05)
    v[:, 1] -= rng.uniform(0.1, 0.3)
    return out, v * np.minimum(rest / radius, 1.0)[:, None]


def _state(case, scene, seed):
    rng = np.random.default_rng([seed, 17])
    x = scene.mesh()["x"]
    v = np.zeros_like(x)
    n = scene.info["n_dyn"]
    d = _config(case).thickness
    if case["scene"] in ("member", "batch"):
        off = 0
        for side, radius in _members(case):
            k = side * side
            x[off:off + k], v[off:off + k] = _drape(rng, x[off:off + k], radius, rng.uniform(0.25, 0.45) * d)
            off += k
    elif case["scene"] == "cloth32":
        v[:n] = _ripple(rng, x[:n], 0.2)
    elif case["scene"] == "tetbox":
        # a face down, tilted a little, its lowest corner inside the contact distance
        p = x[:n] - x[:n].mean(axis=0)
        # rotation taking the box's own axes to the world's: its first row of vertices runs along one edge
        e0 = x[1] - x[0]
        e1 = x[21] - x[0]
        e0, e1 = e0 / np.linalg.norm(e0), e1 / np.linalg.norm(e1)
        q = p @ np.stack([e0, e1, np.cross(e0, e1)], axis=1)
        t = case.get("tilt", 0.003)
        a = rng.uniform(0, 2 * np.pi)
        ax, az = t * math.cos(a), t * math.sin(a)
        rx = np.array([[1, 0, 0], [0, math.cos(ax), -math.sin(ax)], [0, math.sin(ax), math.cos(ax)]])
        rz = np.array([[math.cos(az), -math.sin(az), 0], [math.sin(az), math.cos(az), 0], [0, 0, 1]])
        q = q @ (rx @ rz).T
        q[:, 1] += rng.uniform(0.3, 0.6) * d - q[:, 1].min()
        x[:n] = q
        v[:n] = _ripple(rng, q, 0.02) + np.array([0.0, -rng.uniform(0.3, 0.6), 0.0])
    else:
        if case["cols"]:
            x = folded_flap_state(scene, case["cols"], rng.uniform(0.4, 0.6), rng.uniform(0.4, 0.6))
        v[:n] = _ripple(rng, x[:n], 0.01)
        if not case["cols"]:
            v[:n, 1] -= rng.uniform(0.2, 0.4)  # a few frames into the fall, as it meets the sphere
    return x, v


def prepare(case, seed):
    if case["kind"] in ("forward", "train"):
        rng = np.random.default_rng([seed, 29])
        model = Model.load(DEFAULT_MODEL)
        rows = rng.normal(size=(case["rows"], 12)).astype(np.float32)  # 10 normalised features, 2 scaled targets
        rows[:, 6:8] = np.where(rows[:, 6:8] > 0, 1.0, -1.0)           # the two flags
        rows[:, 10] = np.tanh(rows[:, 1] - 0.5 * rows[:, 3]) + 0.3 * rows[:, 10]
        net = pa.MLP(seed=1)
        if case["kind"] == "forward":
            net.set_params(model.params)
            return dict(kind="forward", net=net, x=np.ascontiguousarray(rows[:, :10]))
        return dict(kind="train", net=net, start=net.params(), rows=rows, batch=case["batch"], epochs=case["epochs"], seed=int(seed) % 2 ** 31)
    key = _scene_key(case)
    x, v = _state(case, _scene(key), seed)
    if case["kind"] == "detect":
        # slots: a program's own contact buffer, above what these states reach (about 4,300 contacts per folded column)
        slots = 8192 + 4500 * case.get("cols", 0)
        return dict(kind="detect", detector=_detector(key), x=x, slots=slots)
    return dict(kind="frames", backend=_backend(key), x=x, v=v, frames=case["frames"])


def run(state):
    kind = state["kind"]
    if kind == "frames":
        b = state["backend"]
        b.reset(state["x"])
        b.set_state(v=state["v"])
        for _ in range(state["frames"]):
            b.step()
        x, v = b.get_state()
        return dict(x=x.astype(np.float32), v=v.astype(np.float32))
    if kind == "detect":
        state["detector"].detect(state["x"])
        ints, reals = state["detector"].contacts()
        out = dict(count=len(ints), ints=np.zeros((state["slots"], 7), np.int32), reals=np.zeros((state["slots"], 9)))
        out["ints"][:len(ints)], out["reals"][:len(ints)] = ints, reals
        return out
    if kind == "forward":
        return state["net"].forward(state["x"])
    net = state["net"]
    net.set_params(state["start"])
    losses = net.train(state["rows"], state["epochs"], state["batch"], 1e-3, state["seed"])
    return dict(params=net.params(), losses=losses.astype(np.float32))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _cloth_sizes(side):
    """(unknowns, constraint rows, factor entries) of a side x side cloth."""
    n = side * side
    return n, 4 * (side - 1) ** 2 + n, 14 * n * max(1, round(math.log2(n)))


def work(case):
    if case["kind"] in ("forward", "train"):
        passes = case.get("epochs", 1) * (3 if case["kind"] == "train" else 1)
        return dict(bytes=48 * case["rows"] * passes, flops=2 * case["rows"] * passes * (10 * 128 + 2 * 128 * 128 + 128 * 2))
    if case["scene"] == "tetbox":
        sizes = [(9261, 120000, 2200 * 9261)]
    elif case["scene"] == "cloth256":
        sizes = [_cloth_sizes(256)]
    elif case["scene"] == "cloth32":
        sizes = [_cloth_sizes(32)]
    else:
        sizes = [_cloth_sizes(s) for s, _ in _members(case)]
    n, m, f = (sum(q) for q in zip(*sizes))
    if case["kind"] == "detect":
        return dict(bytes=24 * n + 30 * 3 * n, flops=200 * 3 * n)
    its = {"cloth32": 20, "cloth256": 50 if case.get("cols", 0) == 0 else 12}.get(case["scene"], 30)
    # per ADMM iteration: rows read and written (z, Ue, rest data), vertices (x, x0, b, p, Uc), the matrix, the factor once each way
    per = 84 * m + 140 * n + 176 * n + 8 * f
    return dict(bytes=case["frames"] * its * per, flops=case["frames"] * its * (12 * f + 120 * m))


# ---------------------------------------------------------------------------
# 64-bit values of the outputs
# ---------------------------------------------------------------------------
def _exact_forward(case, seed):
    s = prepare(case, seed)
    w = Model.load(DEFAULT_MODEL).params.astype(np.float64)
    h, o = s["x"].astype(np.float64), 0
    for k, (rows, cols) in enumerate(((128, 10), (128, 128), (128, 128), (2, 128))):
        a = h @ w[o:o + rows * cols].reshape(rows, cols).T
        o += rows * cols
        a += w[o:o + rows]
        o += rows
        h = a / (1.0 + np.exp(-a)) if k < 3 else a
    return h


def _exact_fall(case, seed):
    """The ADMM step of a scene with no contact in 64 bits, with a dense matrix."""
    scene, cfg = _scene(_scene_key(case)), _config(case)
    x, v = _state(case, scene, seed)
    c, mass, n = scene.constraints(), scene.mass(), scene.info["n_dyn"]
    m, h = scene.info["m_rows"], cfg.dt
    D, w = np.zeros((m, n)), np.zeros(m)
    for e in range(c["n_tri"]):
        t, B = c["tri_inds"][e], c["tri_binv"][e]
        for r in range(2):
            row = c["tri_row0"] + 2 * e + r
            D[row, t] = (-(B[0, r] + B[1, r]), B[0, r], B[1, r])
            w[row] = c["tri_w"][e]
    for e in range(c["n_bend"]):
        for k in range(c["bend_ptr"][e], c["bend_ptr"][e + 1]):
            D[c["bend_row0"] + e, c["bend_inds"][k]] += c["bend_coef"][k]
        w[c["bend_row0"] + e] = c["bend_w"][e]
    pins = slice(c["pin_row0"], c["pin_row0"] + c["n_pin"])
    D[np.arange(pins.start, pins.stop), c["pin_inds"]] = 1.0
    w[pins] = c["pin_w"]
    wl = w.copy()
    wl[pins] = 0.0
    M = mass[:n]
    damp = h * cfg.damp_kl * (D.T * wl) @ D + np.diag(h * cfg.damp_km * M)
    wc = np.where(scene.surface_flags()[:n] > 0, M * cfg.w_scale, 0.0)  # h^2 w_c
    G = h * h * (D.T * w ** 2)
    inv = np.linalg.inv(np.diag(M + wc) + G @ D + damp)
    fixed = scene.mesh()["pins"]
    x0, vel = x[:n].copy(), v[:n].copy()
    ue, uc = np.zeros((m, 3)), np.zeros((n, 3))
    for _ in range(case["frames"]):
        vel[:, 1] -= cfg.g * h
        vel[fixed] = 0.0
        xt = x0 + h * vel
        xk, const = xt, M[:, None] * xt + damp @ x0
        for _ in range(cfg.admm_max_iter):
            y = D @ xk + ue
            z = 0.5 * y
            F = y[c["tri_row0"]:c["tri_row0"] + 2 * c["n_tri"]].reshape(-1, 2, 3)
            U, _, Vt = np.linalg.svd(F, full_matrices=False)
            z[c["tri_row0"]:c["tri_row0"] + 2 * c["n_tri"]] = (0.5 * (F + U @ Vt)).reshape(-1, 3)
            z[pins] = c["pin_pos"]
            hp = xk - x0 + uc
            xn = inv @ (const + G @ (z - ue) + wc[:, None] * (hp + x0 - uc))
            ue += D @ xn - z
            uc += xn - x0 - hp
            xk = xn
        vel, x0 = (xk - x0) / h, xk
    x[:n], v[:n] = x0, vel
    return dict(x=x, v=v)


def exact(case, seed):
    if case["kind"] == "forward":
        return _exact_forward(case, seed)
    if case["kind"] == "frames" and case["scene"] == "cloth32":
        return _exact_fall(case, seed)
    # contact lists are decided pair by pair, and a step with contacts by its lists: no closed 64-bit value here;
    # a training run's weights follow from its own rounding
    return None
