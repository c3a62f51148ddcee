"""GPU parity: the HIP path through the C ABI against the FP64 oracle.

Bars: contact sets bit-identical (indices, order) with float fields equal to
the oracle's FP64 values rounded to FP32; elastic prox, contact projection and
the global solve within FP32 tolerances stated per test; one time step from a
common state within 1e-5 of the FP64 oracle, measured as
||x_gpu - x_oracle|| / ||x_oracle - x_start|| over the dynamic vertices
(helpers.step_err: against the step's own motion).
"""
import numpy as np
import pytest

from helpers import drape_on_obstacle, folded_cloth, rel_err, step_err

pytestmark = pytest.mark.gpu


def _oracle(mesh, cfg, **kw):
    from oracle.pyoracle import Oracle

    return Oracle(mesh, cfg, **kw)


def _detector(pa, scene, cfg):
    return pa.CollisionDetector.for_scene(scene, capacity=cfg.max_contacts, thickness=cfg.thickness)


def _check_contacts_equal(gi, gr, oi, orr):
    assert gi.shape == oi.shape, f"contact count {gi.shape[0]} != oracle {oi.shape[0]}"
    np.testing.assert_array_equal(gi, oi)
    # float fields: FP64 computed identically, rounded to FP32 on the device
    np.testing.assert_array_equal(gr[:, :8], orr[:, :8].astype(np.float32).astype(np.float64))
    np.testing.assert_array_equal(gr[:, 8], orr[:, 8])


@pytest.mark.parametrize("kind,name", [(1, "cloth32"), (2, "tetbox")])
def test_detector_matches_oracle_on_obstacle(pa, kind, name):
    from parallel_admm_amd.configs import config_for

    cfg = config_for(name)
    sc = pa.Scene.generate(kind)
    x = drape_on_obstacle(sc, cfg.thickness).astype(np.float32).astype(np.float64)
    det = _detector(pa, sc, cfg)
    n = det.detect(x)
    gi, gr = det.contacts()
    o = _oracle(sc.mesh(), cfg)
    no = o.detect(x, brute_force=True)
    oi, orr = o.contacts()
    print(f"{name}: {n} contacts (oracle {no})")
    assert n > 0
    _check_contacts_equal(gi, gr, oi, orr)


@pytest.mark.parametrize("jitter", [0.0, 0.15])
def test_detector_matches_oracle_folded_cloth(pa, jitter):
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    x, sc = folded_cloth(side=24, spacing=0.01, gap=0.5 * cfg.thickness, jitter=jitter * cfg.thickness, seed=3)
    x = x.astype(np.float32).astype(np.float64)
    det = _detector(pa, sc, cfg)
    n = det.detect(x)
    gi, gr = det.contacts()
    o = _oracle(sc.mesh(), cfg)
    o.detect(x, brute_force=True)
    oi, orr = o.contacts()
    print(f"folded cloth jitter={jitter}: {n} contacts, PT {np.sum(gi[:, 0] == 0)}, EE {np.sum(gi[:, 0] == 1)}")
    assert n > 100
    _check_contacts_equal(gi, gr, oi, orr)


@pytest.mark.parametrize("faces", [3, 8, 9, 40, 200])
def test_detector_orders_long_segments(pa, faces):
    """One vertex over the hub of a fan of static triangles: it is in contact
    with every face, so its segment of the list has `faces` entries (below, at
    and past the eight that are ranked at a time), numbered in an order that is
    not the order in which the traversal meets them."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    a = 2 * np.pi * np.arange(faces) / faces
    fan = np.concatenate([[[0.0, 0.0, 0.0]], np.stack([0.1 * np.cos(a), 0 * a, 0.1 * np.sin(a)], axis=1)])
    x = np.concatenate([[[0, 0.5 * cfg.thickness, 0], [0.05, 0.05, 0], [0, 0.05, 0.05]], fan])
    k = np.random.default_rng(2).permutation(faces)
    tris = np.concatenate([[[0, 1, 2]], np.stack([np.full(faces, 3), 4 + (k + 1) % faces, 4 + k], axis=1)])
    density = np.concatenate([np.full(3, 1.0), np.full(faces + 1, 1e12)])
    sc = pa.Scene.from_mesh(x, 3, density, tris=tris, tri_k=np.full(len(tris), 1e3))
    det = _detector(pa, sc, cfg)
    det.detect(x)
    gi, gr = det.contacts()
    o = _oracle(sc.mesh(), cfg)
    o.detect(x, brute_force=True)
    oi, orr = o.contacts()
    assert np.sum((gi[:, 0] == 0) & (gi[:, 1] == 0)) >= faces
    _check_contacts_equal(gi, gr, oi, orr)


@pytest.mark.parametrize("side", [2, 3, 9, 60, 110, 140, 180])
def test_query_passes_agree_over_sizes(pa, side):
    """The two-pass queries against the single pass, bit for bit, on folded
    cloths from one cell up to 97,000 edges: below and above a refit block, and
    every number of queries per wave of the collect pass but the largest."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    x, sc = folded_cloth(side=side, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.1 * cfg.thickness, seed=side)
    out = []
    for single in (False, True):
        det = pa.CollisionDetector.for_scene(sc, capacity=1 << 20, thickness=cfg.thickness)
        det.set_single_pass(single)
        det.detect(x)
        out.append(det.contacts())
    assert side < 3 or len(out[0][0]) > 0
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


def test_single_pass_and_two_pass_queries_agree(pa):
    """The two query passes (collect leaf hits, then test them) and the single
    pass (traversal and FP64 test together) give the same list, bit for bit:
    on a folded cloth, and on the folded flap over the 256 x 256 cloth
    (~1e5 contacts; queries with many close leaves fill their slabs and the
    overflow list)."""
    from parallel_admm_amd.configs import config_for, folded_flap_state

    cfg = config_for("cloth32")
    x, sc = folded_cloth(side=24, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.15 * cfg.thickness, seed=3)
    sc3 = pa.Scene.generate(3)
    cases = [(sc, cfg, x.astype(np.float32).astype(np.float64)), (sc3, config_for("cloth256"), folded_flap_state(sc3))]
    for scene, c, pos in cases:
        det = _detector(pa, scene, c)
        n2 = det.detect(pos)
        gi2, gr2 = det.contacts()
        det.set_single_pass(True)
        n1 = det.detect(pos)
        gi1, gr1 = det.contacts()
        print(f"{n2} contacts (two passes), {n1} (single pass)")
        assert n1 == n2 and n2 > 100
        np.testing.assert_array_equal(gi1, gi2)
        np.testing.assert_array_equal(gr1, gr2)


def test_detector_interface(pa):
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(1)
    x = drape_on_obstacle(sc, cfg.thickness)
    det = pa.CollisionDetector.for_scene(sc, capacity=4096, thickness=cfg.thickness)
    n = det.detect(x)
    assert det.contact_count() == n and det.max_slots() == 4096 and det.peak_contact_count() >= n
    pts, nrm = det.points(), det.normals()
    assert pts.shape == (4096, 3) and nrm.shape == (4096, 3)
    assert np.all(pts[n:] == 0) and np.all(nrm[n:] == 0)
    np.testing.assert_allclose(np.linalg.norm(nrm[:n], axis=1), 1.0, atol=1e-6)
    det.clear()
    assert det.contact_count() == 0


def test_detector_overflow_reports_error(pa):
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    x, sc = folded_cloth(side=16, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.0)
    det = pa.CollisionDetector.for_scene(sc, capacity=8, thickness=cfg.thickness)
    with pytest.raises(pa.PAError) as e:
        det.detect(x)
    assert e.value.code == pa.PA_ERR_OVERFLOW


def test_elastic_prox_matches_oracle(pa):
    """z = prox(D x + Ue): tri (Stiefel polar), tet (closest rotation), bend, pin.
    Tolerance 2e-5 relative per block (FP32 vs FP64)."""
    from parallel_admm_amd.configs import config_for

    rng = np.random.default_rng(7)
    for kind, name in ((1, "cloth32"), (2, "tetbox")):
        cfg = config_for(name)
        sc = pa.Scene.generate(kind)
        m = sc.mesh()
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        x = m["x"] + 0.002 * rng.standard_normal(m["x"].shape)
        x = x.astype(np.float32).astype(np.float64)
        ue = (0.05 * rng.standard_normal((sc.info["m_rows"], 3))).astype(np.float32).astype(np.float64)
        zg = b.project_elastic(x, ue)
        zo = _oracle(m, cfg).project_elastic(x, ue)
        err = np.abs(zg - zo).max() / np.abs(zo).max()
        print(f"{name}: max |z_gpu - z_oracle| / max|z| = {err:.2e}")
        assert err < 2e-5


def test_contact_projection_matches_oracle(pa):
    """Jacobi-weighted friction-cone sweeps on the folded-cloth contact set.
    Tolerance 1e-4 relative (FP32 accumulation over gs_max_iter sweeps)."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    x, sc = folded_cloth(side=16, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.1 * cfg.thickness, seed=1)
    x = x.astype(np.float32).astype(np.float64)
    m = sc.mesh()
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    b.set_state(x=x)
    # detection through the backend's own detector
    rng = np.random.default_rng(2)
    p = (0.5 * rng.standard_normal(x.shape)).astype(np.float32).astype(np.float64)
    p[m["n_dyn"]:] = 0
    det = pa.CollisionDetector.for_scene(sc, capacity=cfg.max_contacts, thickness=cfg.thickness)
    nc = det.detect(x)
    b.attach_detector(det)
    pg, rg = b.project_contacts(p)
    o = _oracle(m, cfg)
    o.detect(x)
    po, ro = o.project_contacts(p)
    assert nc > 50
    e1 = np.abs(pg - po).max() / np.abs(po).max()
    e2 = np.abs(rg - ro).max() / max(np.abs(ro).max(), 1e-12)
    print(f"{nc} contacts: p err {e1:.2e}, r_c err {e2:.2e}")
    assert e1 < 1e-4 and e2 < 1e-4


@pytest.mark.parametrize("precond", [0, 1], ids=["jacobi", "amg"])
def test_global_solve_matches_llt(pa, precond):
    """Global solve (FP64 residual + FP32 PCG correction, two refinement passes)
    against the oracle's sparse LLT: relative error <= 1e-6, with the Jacobi
    and the smoothed-aggregation AMG preconditioners."""
    from parallel_admm_amd.configs import config_for

    rng = np.random.default_rng(5)
    for kind, name in ((1, "cloth32"), (2, "tetbox"), (3, "cloth256")):
        cfg = config_for(name)
        cfg.global_tol = 1e-5
        cfg.global_refine = 2
        cfg.global_max_iter = 2000
        cfg.precond = precond
        sc = pa.Scene.generate(kind)
        m = sc.mesh()
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        o = _oracle(m, cfg)
        n = sc.info["n_dyn"]
        xs = m["x"][:n] + 0.01 * rng.standard_normal((n, 3))
        A = o.matrix(1)
        rhs = A @ xs
        xo = o.solve(rhs)
        xg, it = b.global_solve(rhs, m["x"][:n])
        err = rel_err(xg, xo)
        print(f"{name} precond={precond}: PCG {it} iterations, rel err vs LLT {err:.2e}")
        assert err < 1e-6
        if precond == 1:
            assert it <= 60


@pytest.mark.parametrize("side", [2, 13, 128, 129])
def test_amg_solve_at_workgroup_edges(pa, side):
    """The AMG-preconditioned solve with one level, one part-filled workgroup,
    and the last size on the small workgroups (16384 rows of 8 lanes) and the
    first past it: the bar of test_global_solve_matches_llt."""
    from parallel_admm_amd.configs import config_for

    rng = np.random.default_rng(side)
    cfg = config_for("cloth32")
    cfg.global_tol = 1e-5
    cfg.global_refine = 2
    cfg.global_max_iter = 2000
    cfg.precond = 1
    sc = pa.Scene.generate(4, side=side, radius=0.1, drop=0.3)
    m = sc.mesh()
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    o = _oracle(m, cfg)
    n = sc.info["n_dyn"]
    xs = m["x"][:n] + 0.01 * rng.standard_normal((n, 3))
    rhs = o.matrix(1) @ xs
    xg, it = b.global_solve(rhs, m["x"][:n])
    err = rel_err(xg, o.solve(rhs))
    print(f"side {side}: PCG {it} iterations, rel err vs LLT {err:.2e}")
    assert err < 1e-6 and it <= 60


@pytest.mark.parametrize("passes", [1, 2])
def test_direct_solve_matches_llt(pa, passes):
    """The direct global solve (precond 2: supernodal Cholesky factored on the
    host at init, FP32 level-scheduled triangular solves on the FP64
    residual) against the oracle's sparse LLT, on the three workload scenes
    and a merged batch of four cloths (a forest of independent factor trees).
    The error is measured against the size of the correction the solve makes
    (x_o - x_start): within 2e-4 after one pass and 1e-6 after two."""
    from parallel_admm_amd.configs import config_for

    rng = np.random.default_rng(6)
    cases = [(pa.Scene.generate(k), name) for k, name in ((1, "cloth32"), (2, "tetbox"), (3, "cloth256"))]
    cases.append((pa.Scene.merge([pa.Scene.generate(4, side=s, radius=0.1, drop=0.3) for s in (16, 40, 24, 33)]), "batch"))
    for sc, name in cases:
        cfg = config_for(name)
        cfg.precond = 2
        cfg.global_refine = passes
        m = sc.mesh()
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        o = _oracle(m, cfg)
        n = sc.info["n_dyn"]
        xs = m["x"][:n] + 0.01 * rng.standard_normal((n, 3))
        A = o.matrix(1)
        rhs = A @ xs
        xo = o.solve(rhs)
        x0 = m["x"][:n]
        xg, it = b.global_solve(rhs, x0)
        err = np.linalg.norm(xg - xo) / np.linalg.norm(xo - x0)
        print(f"{name} direct, {passes} pass(es): reported {it}, error / correction {err:.2e}")
        assert it == passes
        assert err < (2e-4 if passes == 1 else 1e-6)


@pytest.mark.parametrize("sides", [(2,), (3,), (13,), (16, 2, 41), (64,), (65,), (80, 5, 64), (120,)], ids=str)
def test_direct_solve_at_factor_edges(pa, sides):
    """Cloths below, at and above a leaf's and a dense top's size (a 64 x 64
    cloth is all top, a 65 x 65 one has a level below it), alone and in
    forests, with row and column counts that are no multiples of the solve's
    tiles.  One pass against the oracle's LLT: the FP32 panels and products
    round at 6e-8 times a modest growth over the levels, so 1e-5 of the
    correction."""
    from parallel_admm_amd.configs import config_for

    rng = np.random.default_rng(8)
    cfg = config_for("batch")
    parts = [pa.Scene.generate(4, side=s, radius=0.1, drop=0.3) for s in sides]
    sc = parts[0] if len(parts) == 1 else pa.Scene.merge(parts)
    m = sc.mesh()
    n = sc.info["n_dyn"]
    o = _oracle(m, cfg)
    rhs = o.matrix(1) @ (m["x"][:n] + 0.01 * rng.standard_normal((n, 3)))
    xo = o.solve(rhs)
    x0 = m["x"][:n]
    xg, _ = pa.ADMMBackendHIP.from_scene(sc, cfg).global_solve(rhs, x0)
    err = np.linalg.norm(xg - xo) / np.linalg.norm(xo - x0)
    print(f"sides {sides}: error / correction {err:.2e}")
    assert err < 1e-5


def test_global_solve_multi_pass_matches_llt(pa):
    """A 300 x 300 cloth (90,000 rows) is more rows than one pass of the fused
    PCG grid covers, so the kernels run their multi-pass variant (each pass
    loads the next pass's row ranges ahead): against the oracle's sparse LLT
    within 1e-6 relative."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("batch")
    cfg.precond = 1  # the fused AMG-PCG kernels' multi-pass variant
    cfg.global_tol = 1e-5
    cfg.global_refine = 2
    cfg.global_max_iter = 2000
    sc = pa.Scene.generate(4, side=300, radius=0.2, drop=0.3)
    m = sc.mesh()
    n = sc.info["n_dyn"]
    assert n == 90000
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    o = _oracle(m, cfg)
    rng = np.random.default_rng(11)
    xs = m["x"][:n] + 0.01 * rng.standard_normal((n, 3))
    rhs = o.matrix(1) @ xs
    xo = o.solve(rhs)
    xg, it = b.global_solve(rhs, m["x"][:n])
    err = rel_err(xg, xo)
    print(f"side 300: PCG {it} iterations, rel err vs LLT {err:.2e}")
    assert err < 1e-6 and it <= 60


STEP_CASES = [
    # (label, config, scene kind, generator args, frames, start state, residual_tol, global solve (None: the config's))
    ("cloth32-free", "cloth32", 1, {}, 4, "rest", 0.0, None),
    ("cloth32-drape", "cloth32", 4, dict(side=32, radius=0.2, drop=0.002), 6, "rest", 0.0, None),
    ("tetbox-ground", "tetbox", 2, {}, 4, "drape", 0.0, None),
    ("cloth32-free-tol", "cloth32", 1, {}, 4, "rest", 1e-4, None),
    ("cloth32-drape-tol", "cloth32", 4, dict(side=32, radius=0.2, drop=0.002), 6, "rest", 1e-4, None),
    ("tetbox-ground-tol", "tetbox", 2, {}, 4, "drape", 1e-4, None),
    # the same with AMG-PCG instead of the workloads' direct solve
    ("cloth32-drape-amg", "cloth32", 4, dict(side=32, radius=0.2, drop=0.002), 6, "rest", 0.0, 1),
    ("tetbox-ground-amg", "tetbox", 2, {}, 4, "drape", 0.0, 1),
    ("cloth32-drape-tol-amg", "cloth32", 4, dict(side=32, radius=0.2, drop=0.002), 6, "rest", 1e-4, 1),
]


@pytest.mark.parametrize("label,name,kind,gen,frames,start,rtol,precond", STEP_CASES, ids=[c[0] for c in STEP_CASES])
def test_step_matches_fp64_oracle(pa, label, name, kind, gen, frames, start, rtol, precond):
    """One time step from a common state (x, v, Ue, Uc), per frame, within 1e-5
    of the oracle's step measured against the step's motion (step_err), with
    the workload's solver settings.  With residual_tol = 1e-4 the step stops
    on the ADMM residual: the residuals at every check agree with the
    oracle's residual_log (1e-3 relative, 1e-6 absolute) and the iteration counts
    agree within one (a residual within that band of the threshold may stop
    one side an iteration earlier)."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for(name)
    cfg.residual_tol = rtol
    if precond is not None:
        cfg.precond = precond
    sc = pa.Scene.generate(kind, **gen)
    m = sc.mesh()
    n = sc.info["n_dyn"]
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    if start == "drape":
        b.set_state(x=drape_on_obstacle(sc, cfg.thickness, frac=2.0))
    o = _oracle(m, cfg)
    worst = worst_res = 0.0
    contacts = 0
    for f in range(frames):
        x, v = b.get_state()
        ue, uc = b.get_duals()
        o.set_state(x, v)
        o.set_duals(ue, uc)
        n_log = len(o.residual_log())  # the oracle's log runs on over its steps
        st = b.step()
        so = o.step()
        xg, vg = b.get_state()
        xo, vo = o.state()
        e = step_err(xg, xo, x, n)
        worst = max(worst, e)
        contacts += st["n_contacts"]
        msg = ""
        if rtol > 0:
            rg, ro = b.residual_log(), o.residual_log()[n_log:]
            k = min(len(rg), len(ro))
            assert k > 0 and abs(len(rg) - len(ro)) <= 1 and abs(st["iterations"] - so["iterations"]) <= 1
            # relative 1e-3, above an absolute floor of 1e-6 (FP32 vectors
            # cannot resolve a residual far below the 1e-4 threshold)
            dr = float(np.max(np.abs(rg[:k] - ro[:k]) / (np.abs(ro[:k]) + 1e-3)))
            worst_res = max(worst_res, dr)
            msg = (f", ADMM iters gpu {st['iterations']} oracle {so['iterations']}, final residual gpu "
                   f"{max(rg[-1]):.3e} oracle {max(ro[-1]):.3e}, residual rel diff {dr:.2e}")
        print(f"{label} frame {f}: contacts gpu {st['n_contacts']} oracle {so['n_contacts']}, "
              f"PCG iters {st['global_iters']}, step err {e:.2e} (|x| rel {rel_err(xg, xo):.2e}){msg}")
    assert worst < 1e-5
    assert worst_res < 1e-3
    if start == "drape" or "drape" in label:
        assert contacts > 0


def test_step_with_rotating_obstacle_matches_oracle(pa):
    """A cloth draped on a sphere that spins about +y (rigid track, 2 frames
    per step as the reference's animator moves one rigid mesh): one step from a
    common state per frame within 1e-5 (step_err), same contact counts, and the
    animated static vertices equal to the oracle's (both FP64)."""
    from parallel_admm_amd.configs import config_for, rotation_track

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(4, side=24, radius=0.2, drop=0.002)
    m = sc.mesh()
    n, n_all = sc.info["n_dyn"], sc.info["n_all"]
    pos, quat = rotation_track((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 3.0, cfg.dt / 2, 64)
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    b.add_rigid_track(n, n_all - n, pos, quat, frames_per_step=2)
    o = _oracle(m, cfg)
    o.add_rigid_track(n, n_all - n, pos, quat, frames_per_step=2)
    worst, contacts = 0.0, 0
    for f in range(6):
        x, v = b.get_state()
        ue, uc = b.get_duals()
        o.set_state(x, v)
        o.set_duals(ue, uc)
        st = b.step()
        so = o.step()
        xg, vg = b.get_state()
        xo, vo = o.state()
        # the animated obstacle: both place it in FP64 from the same track
        np.testing.assert_allclose(xg[n:], xo[n:], rtol=0, atol=1e-12)
        np.testing.assert_allclose(vg[n:], vo[n:], rtol=0, atol=1e-9)
        e = step_err(xg, xo, x, n)
        worst = max(worst, e)
        contacts += st["n_contacts"]
        assert st["n_contacts"] == so["n_contacts"]
        print(f"spin frame {f}: contacts {st['n_contacts']}, step err {e:.2e}, |v_static| {np.abs(vg[n:]).max():.3f}")
    assert worst < 1e-5 and contacts > 0
    assert np.abs(vg[n:]).max() > 0.1  # the obstacle moves


@pytest.mark.parametrize("name,kind", [("tetbox", 2), ("cloth256", 3)])
def test_graph_replay_matches_eager(pa, name, kind):
    """PCG iteration pairs replayed as HIP graphs (pa_admm_config.graphs = 1)
    against the same kernels launched one by one: equal iteration counts and
    states within 1e-6 relative.  Each step replays the graphs many times with
    eager work (detection, local and contact steps, read-backs) between the
    replays."""
    from parallel_admm_amd.configs import config_for

    sc = pa.Scene.generate(kind)
    states = {}
    for graphs in (0, 1):
        cfg = config_for(name)
        cfg.precond = 1  # graphs replay PCG iteration pairs
        cfg.graphs = graphs
        cfg.admm_max_iter = 12
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        if name == "tetbox":
            b.set_state(x=drape_on_obstacle(sc, cfg.thickness, frac=2.0))
        out = []
        for _ in range(3):
            st = b.step()
            out.append((b.get_state()[0], st["global_iters"]))
        states[graphs] = out
    for (xe, ie), (xg, ig) in zip(states[0], states[1]):
        assert ie == ig and ie > 0
        # identical arithmetic; one run in about ten has shown rounding-level
        # differences (<= 1.5e-8 absolute in 5% of the coordinates), so the
        # bar is a relative 1e-6 rather than bitwise
        assert rel_err(xg, xe) < 1e-6


def test_step_deterministic(pa):
    """Two runs from the same state are bitwise identical."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(1)
    x0 = drape_on_obstacle(sc, cfg.thickness, frac=2.0)
    out = []
    for _ in range(2):
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        b.set_state(x=x0)
        for _ in range(3):
            b.step()
        out.append(b.get_state()[0])
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("tol", [0.0, 1e-4], ids=["capped", "tol-1e-4"])
def test_contact_sweeps_in_one_workgroup_match_per_sweep_launches(pa, tol):
    """Contact projections of up to 2048 contacts run every Jacobi sweep in
    one workgroup; with that off every sweep is two launches.  The two paths
    do the same arithmetic in the same order, so three steps of a draped
    cloth (~150 contacts: one contact per lane) and of a folded one (~1700:
    two per lane) give the same positions, velocities and duals, bit for bit
    (with residual_tol 1e-4 also past the device stop test)."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    cfg.residual_tol = tol
    sc = pa.Scene.generate(1)
    xf, scf = folded_cloth(side=11, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.15 * cfg.thickness, seed=3)
    for scene, x0 in ((sc, drape_on_obstacle(sc, cfg.thickness)), (scf, xf)):
        out = []
        for wg in (2048, 0):
            b = pa.ADMMBackendHIP.from_scene(scene, cfg)
            b.set_contact_sweep_wg(wg)
            b.set_state(x=x0)
            nc = [b.step()["n_contacts_max"] for _ in range(3)]
            out.append((*b.get_state(), *b.get_duals()))
        print(f"{scene.info['n_dyn']} dynamic vertices, tol {tol}: contacts per step {nc}")
        assert 0 < max(nc) <= 2048
        for a, c in zip(*out):
            np.testing.assert_array_equal(a, c)


@pytest.mark.parametrize("pairs", [1, 1024, 1025, 1500, 2048])
def test_contact_sweeps_in_one_workgroup_with_distinct_vertices(pa, pairs):
    """Isolated triangle pairs, one vertex of the upper triangle over the lower
    one: one contact of four distinct vertices per pair, so the entry and run
    counts are the largest the contact count allows, on both sides of the
    one-contact-per-lane limit and past the runs whose p fits in LDS.  The
    one-workgroup sweeps give the same bits as the per-sweep launches."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    d = cfg.thickness
    lower = np.array([[0, 0, 0], [0.01, 0, 0], [0, 0, 0.01]])
    upper = np.array([[0.0033, 0.5 * d, 0.0033], [0.0063, 0.01, 0.0033], [0.0033, 0.01, 0.0063]])
    cell = np.concatenate([lower, upper])
    k = np.arange(pairs)
    shift = 0.05 * np.stack([k % 40, np.zeros(pairs), k // 40], axis=1)
    x = (cell[None] + shift[:, None]).reshape(-1, 3)
    tris = np.arange(6 * pairs).reshape(-1, 3)
    sc = pa.Scene.from_mesh(x, len(x), np.full(len(x), 1.0), tris=tris, tri_k=np.full(len(tris), 1e3))
    v = np.random.default_rng(5).normal(size=x.shape) * 1e-3  # moves a vertex by 0.02 mm a step: every pair stays within d
    out = []
    for wg in (2048, 0):
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        b.set_contact_sweep_wg(wg)
        b.set_state(v=v)
        st = b.step()
        assert st["n_contacts_max"] == pairs
        out.append((*b.get_state(), *b.get_duals()))
    for a, c in zip(*out):
        np.testing.assert_array_equal(a, c)


def test_step_overflow_rolls_back(pa):
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    cfg.max_contacts = 4
    x, sc = folded_cloth(side=16, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.0)
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    b.set_state(x=x)
    before = b.get_state()[0]
    with pytest.raises(pa.PAError) as e:
        b.step()
    assert e.value.code == pa.PA_ERR_OVERFLOW
    np.testing.assert_array_equal(b.get_state()[0], before)


def test_cloth256_folded_flap_step_matches_fp64_oracle(pa):
    """cloth256 at the config's ~1e5 contacts: the workload's scene with a
    24-column flap folded back over the cloth (101,804 contacts at rest), one
    step on both from that state.  The step's first detection sees the full
    set (the contact response then lifts the flap to the contact distance, so
    later detections find few pairs); counts of the step's last detection
    within 0.5% or 2 (later detections run on iterates that differ at
    rounding level) and the step within 2e-5 (step_err), the bar of the other
    folded cloth256 state."""
    from oracle.pyoracle import Oracle
    from parallel_admm_amd.configs import config_for, folded_flap_state, workload_tracks

    cfg = config_for("cloth256")
    sc = pa.Scene.generate(3)
    x0 = folded_flap_state(sc)
    tracks = workload_tracks("cloth256", sc, 8)
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    o = Oracle(sc.mesh(), cfg)
    for first, count, pos, quat in tracks:
        b.add_rigid_track(first, count, pos, quat)
        o.add_rigid_track(first, count, pos, quat)
    b.set_state(x0)
    o.set_state(x0)
    n0 = o.detect(x0)
    st = b.step()
    so = o.step()
    e = step_err(b.get_state()[0], o.state()[0], x0, sc.info["n_dyn"])
    print(f"cloth256 folded flap: {n0} contacts at the start, the step's most {st['n_contacts_max']}; last detection gpu "
          f"{st['n_contacts']} oracle {so['n_contacts']}, ADMM iterations {st['iterations']}, PCG {st['global_iters']}, "
          f"step err {e:.2e}")
    assert n0 > 100000 and st["n_contacts_max"] > 95000
    assert abs(st["n_contacts"] - so["n_contacts"]) <= max(2, 0.005 * so["n_contacts"])
    assert e < 2e-5


def test_cloth256_folded_step_matches_fp64_oracle(pa):
    """cloth256 at the workload's contact density: 120 steps of the whole run
    (sphere and rotating cylinder) into a folded state with about ten thousand
    contacts, then one step from that common state on both, the oracle's
    cylinder track resumed at the same frame: within 1e-4 (step_err; the
    state's measured floor is stated below), contact counts of the step's
    last detection within 0.5% (see test_cloth256_step_matches_fp64_oracle
    for why they may differ by a few)."""
    from oracle.pyoracle import Oracle
    from parallel_admm_amd.configs import config_for, workload_tracks

    cfg = config_for("cloth256")
    sc = pa.Scene.generate(3)
    warm = 120
    tracks = workload_tracks("cloth256", sc, warm + 8)
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    b.set_sync_to_host(False)
    for first, count, pos, quat in tracks:
        b.add_rigid_track(first, count, pos, quat)
    for _ in range(warm):
        b.step()
    o = Oracle(sc.mesh(), cfg)
    for first, count, pos, quat in tracks:
        o.add_rigid_track(first, count, pos[warm:], quat[warm:])
    x, v = b.get_state()
    ue, uc = b.get_duals()
    o.set_state(x, v)
    o.set_duals(ue, uc)
    st = b.step()
    so = o.step()
    e = step_err(b.get_state()[0], o.state()[0], x, sc.info["n_dyn"])
    print(f"cloth256 frame {warm}: contacts gpu {st['n_contacts']} oracle {so['n_contacts']}, ADMM iterations {st['iterations']}, "
          f"PCG {st['global_iters']}, step err {e:.2e} (|x| rel {rel_err(b.get_state()[0], o.state()[0]):.2e})")
    assert st["n_contacts"] > 5000 and abs(st["n_contacts"] - so["n_contacts"]) <= 0.005 * so["n_contacts"]
    # Measured floor of this state: 4.1e-5 of the step's motion with the
    # direct solve (1.0-1.7e-5 on the AMG-PCG trajectory's state).  The cloth
    # lies folded on the obstacles and the step moves it little (0.055 in
    # norm over 65,536 vertices), so 4.1e-5 is about 5e-9 m per coordinate:
    # the FP32 rounding of the contact, dual and prox quantities, not the
    # solve.  The step is well conditioned: a 1e-9 m perturbation of the
    # oracle's own start state moves its result by 5e-6 of the motion, and
    # 1e-12 m by 5e-9.  The bar is 2.4 times the floor.
    assert e < 1e-4


@pytest.mark.parametrize("tracked", [False, True], ids=["plain", "rotating-obstacle"])
def test_nonfinite_state_rolls_back(pa, tracked):
    """NaN injected into x (or Inf into v) from the host: the next step
    reports PA_ERR_NUMERICAL and the state is the one after the last good
    step, bit for bit (with a rigid track: its frame counter too); stepping
    then continues as if nothing happened."""
    from parallel_admm_amd.configs import config_for, rotation_track

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(4, side=24, radius=0.2, drop=0.002)
    n, n_all = sc.info["n_dyn"], sc.info["n_all"]
    pos, quat = rotation_track((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 3.0, cfg.dt, 64)
    ref = pa.ADMMBackendHIP.from_scene(sc, cfg)
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    if tracked:
        for bb in (ref, b):
            bb.add_rigid_track(n, n_all - n, pos, quat)
    for _ in range(3):
        ref.step()
        b.step()
    frames = b.track_frames().copy()
    good_x, good_v = b.get_state()
    for field in ("x", "v"):
        x, v = b.get_state()
        if field == "x":
            x[5, 1] = np.nan
        else:
            v[7, 0] = np.inf
        b.set_state(x, v)
        with pytest.raises(pa.PAError) as e:
            b.step()
        assert e.value.code == pa.PA_ERR_NUMERICAL
        xr, vr = b.get_state()
        np.testing.assert_array_equal(xr, good_x)
        np.testing.assert_array_equal(vr, good_v)
        np.testing.assert_array_equal(b.track_frames(), frames)
    for _ in range(2):
        ref.step()
        b.step()
    np.testing.assert_array_equal(b.get_state()[0], ref.get_state()[0])
    np.testing.assert_array_equal(b.get_state()[1], ref.get_state()[1])


def test_overflow_rollback_restores_tracks_and_duals(pa):
    """A contact overflow in the middle of a run on a tracked scene: the step
    is refused, positions, velocities, duals and the track's frame are those
    of the step's start, and the run then continues exactly as one that never
    overflowed (the capacity is raised through a fresh backend built from the
    same state)."""
    from parallel_admm_amd.configs import config_for, rotation_track

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(4, side=24, radius=0.2, drop=0.002)
    n, n_all = sc.info["n_dyn"], sc.info["n_all"]
    pos, quat = rotation_track((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 3.0, cfg.dt, 64)
    small = config_for("cloth32")
    small.max_contacts = 8
    b = pa.ADMMBackendHIP.from_scene(sc, small)
    b.add_rigid_track(n, n_all - n, pos, quat)
    before = b.get_state()
    ue0, uc0 = b.get_duals()
    f0 = b.track_frames().copy()
    with pytest.raises(pa.PAError) as e:
        for _ in range(10):  # the cloth settles onto the sphere: more than 8 contacts
            before = b.get_state()
            ue0, uc0 = b.get_duals()
            f0 = b.track_frames().copy()
            b.step()
    assert e.value.code == pa.PA_ERR_OVERFLOW
    x1, v1 = b.get_state()
    ue1, uc1 = b.get_duals()
    np.testing.assert_array_equal(x1, before[0])
    np.testing.assert_array_equal(v1, before[1])
    np.testing.assert_array_equal(ue1, ue0)
    np.testing.assert_array_equal(uc1, uc0)
    np.testing.assert_array_equal(b.track_frames(), f0)


def test_step_without_detector_leaves_state(pa):
    """The reference's call order with contact enabled but no detector
    attached: step() is refused with PA_ERR_INVALID and the positions and
    velocities are the ones init was given, bit for bit; after attaching a
    detector the step runs."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(1)
    m = sc.mesh()
    b = pa.ADMMBackendHIP()
    b.apply_config(cfg)
    b.set_constraints(sc)
    b.set_constraint_dim(sc.info["m_rows"])
    b.finalize_constraints()
    b.init(m["x"], sc.mass(), sc.info["n_dyn"], sc.surface_flags(), m["pins"])
    with pytest.raises(pa.PAError) as e:
        b.step()
    assert e.value.code == pa.PA_ERR_INVALID
    x, v = b.get_state()
    np.testing.assert_array_equal(x, m["x"])
    np.testing.assert_array_equal(v, 0.0)
    b.attach_detector(pa.CollisionDetector.for_scene(sc, capacity=cfg.max_contacts, thickness=cfg.thickness))
    st = b.step()
    assert st["iterations"] == cfg.admm_max_iter and np.all(np.isfinite(b.get_state()[0]))


@pytest.mark.parametrize("tracked", [False, True], ids=["plain", "rotating-obstacle"])
def test_reset_restarts_the_run(pa, tracked):
    """Reference reset (admm_impl_gpu.cu:151-155 via ADMMImplCPUBase::reset,
    admm_impl_cpu.cpp:71-88): after some steps, reset(x_init) gives the given
    positions, zero velocities and duals and the track back at frame 0, and
    the run that follows is bit-identical to a fresh backend's."""
    from parallel_admm_amd.configs import config_for, rotation_track

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(4, side=24, radius=0.2, drop=0.002)
    m = sc.mesh()
    n, n_all = sc.info["n_dyn"], sc.info["n_all"]
    pos, quat = rotation_track((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 3.0, cfg.dt, 64)

    def fresh():
        bb = pa.ADMMBackendHIP.from_scene(sc, cfg)
        if tracked:
            bb.add_rigid_track(n, n_all - n, pos, quat)
        return bb

    b = fresh()
    for _ in range(4):
        b.step()
    b.reset(m["x"])
    x, v = b.get_state()
    ue, uc = b.get_duals()
    np.testing.assert_array_equal(x, m["x"])
    np.testing.assert_array_equal(v, 0.0)
    np.testing.assert_array_equal(ue, 0.0)
    np.testing.assert_array_equal(uc, 0.0)
    if tracked:
        np.testing.assert_array_equal(b.track_frames(), [1])
    ref = fresh()
    for _ in range(3):
        sa, sb = b.step(), ref.step()
        assert sa["n_contacts"] == sb["n_contacts"] and sa["iterations"] == sb["iterations"]
    np.testing.assert_array_equal(b.get_state()[0], ref.get_state()[0])
    np.testing.assert_array_equal(b.get_state()[1], ref.get_state()[1])


@pytest.mark.parametrize("tracked", [False, True], ids=["plain", "rotating-obstacle"])
def test_checkpoint_resume_is_bit_exact(pa, tmp_path, tracked):
    """Six steps straight equal three steps, a checkpoint, a fresh backend
    loading it, and three more steps (also with a rigid track, whose frame
    counter and last placed positions are restored)."""
    from parallel_admm_amd import checkpoint
    from parallel_admm_amd.configs import config_for, rotation_track

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(4, side=24, radius=0.2, drop=0.002)
    n, n_all = sc.info["n_dyn"], sc.info["n_all"]
    pos, quat = rotation_track((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 3.0, cfg.dt, 64)

    def fresh():
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        if tracked:
            b.add_rigid_track(n, n_all - n, pos, quat)
        return b

    straight = fresh()
    for _ in range(6):
        straight.step()
    first = fresh()
    for _ in range(3):
        first.step()
    path = str(tmp_path / "ck.npz")
    checkpoint.save(first, path, 3, cfg)
    resumed = fresh()
    assert checkpoint.load(resumed, path, cfg) == 3
    for _ in range(3):
        resumed.step()
    xs, vs = straight.get_state()
    xr, vr = resumed.get_state()
    np.testing.assert_array_equal(xr, xs)
    np.testing.assert_array_equal(vr, vs)
    other = config_for("cloth32")
    other.mu = 0.31
    with pytest.raises(ValueError):
        checkpoint.load(fresh(), path, other)


def test_degenerate_systems(pa):
    """k = 0 (no stretch or bending stiffness) with every vertex pinned: the
    system stays SPD through the mass term and the step holds every vertex at
    its pin.  A zero-density cloth (zero mass) is refused before any solve."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    cfg.enable_contact = False
    side = 6
    g = np.arange(side)
    x = np.stack([np.repeat(g, side) * 0.01, np.full(side * side, 0.5), np.tile(g, side) * 0.01], axis=1)
    tris = []
    for i in range(side - 1):
        for j in range(side - 1):
            a, b, c, d = i * side + j, (i + 1) * side + j, (i + 1) * side + j + 1, i * side + j + 1
            tris += [[a, b, c], [a, c, d]]
    tris = np.array(tris, np.int32)
    n = side * side
    sc = pa.Scene.from_mesh(x, n, np.ones(n), tris=tris, tri_k=np.zeros(len(tris)), bend_k=np.zeros(n), pins=np.arange(n))
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    for _ in range(3):
        b.step()
    xg, vg = b.get_state()
    assert np.all(np.isfinite(xg)) and np.abs(xg - x).max() < 1e-6
    with pytest.raises(pa.PAError) as e:
        sc0 = pa.Scene.from_mesh(x, n, np.zeros(n), tris=tris, tri_k=np.ones(len(tris)), bend_k=np.zeros(n))
        pa.ADMMBackendHIP.from_scene(sc0, cfg)
    assert e.value.code in (pa.PA_ERR_INVALID, pa.PA_ERR_GEOMETRY)


def test_cloth256_step_matches_fp64_oracle(pa):
    """The headline workload: 256 x 256 cloth over a sphere and a cylinder,
    four steps on the GPU into folded self-contact, then one step from that
    common state on both: within 1e-5 (step_err).  The step's later detections
    run on intermediate iterates, FP32 on the GPU and FP64 in the oracle,
    which differ by ~1e-7 relative; with thousands of contacts spread over a
    0.5 mm band a few pairs lie within that distance of the threshold and can
    flip, so the contact counts of the step's last detection agree to 0.5%
    (detection itself is bit-exact on identical positions:
    test_detector_matches_oracle_*)."""
    from oracle.pyoracle import Oracle
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth256")
    sc = pa.Scene.generate(3)
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    for _ in range(4):
        b.step()
    o = Oracle(sc.mesh(), cfg)
    for f in range(2):
        x, v = b.get_state()
        ue, uc = b.get_duals()
        o.set_state(x, v)
        o.set_duals(ue, uc)
        st = b.step()
        so = o.step()
        e = step_err(b.get_state()[0], o.state()[0], x, sc.info["n_dyn"])
        print(f"cloth256 frame {f}: contacts gpu {st['n_contacts']} oracle {so['n_contacts']}, "
              f"ADMM iterations {st['iterations']}, PCG {st['global_iters']}, step err {e:.2e} "
              f"(|x| rel {rel_err(b.get_state()[0], o.state()[0]):.2e})")
        assert st["n_contacts"] > 0 and abs(st["n_contacts"] - so["n_contacts"]) <= 0.005 * so["n_contacts"]
        assert e < 1e-5


def test_heuristic_contact_weight_step_matches_oracle(pa):
    """contact.use_heu_wc on (as the reference's 10-layers-skew.toml and
    test_GN.toml scenes set it): the draped cloth32, one step from a common
    state per frame within 1e-5 of the oracle (step_err)."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    cfg.use_heu_wc, cfg.wc_sigma, cfg.wc_beta = True, 0.01, 25.0
    sc = pa.Scene.generate(4, side=32, radius=0.2, drop=0.002)
    n = sc.info["n_dyn"]
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    o = _oracle(sc.mesh(), cfg)
    worst, contacts = 0.0, 0
    for f in range(5):
        x, v = b.get_state()
        ue, uc = b.get_duals()
        o.set_state(x, v)
        o.set_duals(ue, uc)
        st = b.step()
        so = o.step()
        e = step_err(b.get_state()[0], o.state()[0], x, n)
        worst = max(worst, e)
        contacts += st["n_contacts"]
        assert st["n_contacts"] == so["n_contacts"]
        print(f"heuristic w_c frame {f}: contacts {st['n_contacts']}, step err {e:.2e}")
    assert worst < 1e-5 and contacts > 0


def test_short_surface_edge_is_refused(pa):
    """The reference's set-up check (dcd_validation.h:8-33): a dynamic surface
    edge shorter than the contact distance makes attaching the detector fail
    with PA_ERR_GEOMETRY; a thickness below the shortest edge is accepted."""
    from parallel_admm_amd.configs import config_for

    sc = pa.Scene.generate(1)  # 1 cm cloth spacing
    for thickness, ok in ((0.02, False), (0.005, True)):
        cfg = config_for("cloth32")
        cfg.thickness = thickness
        if ok:
            pa.ADMMBackendHIP.from_scene(sc, cfg)
        else:
            with pytest.raises(pa.PAError) as e:
                pa.ADMMBackendHIP.from_scene(sc, cfg)
            assert e.value.code == pa.PA_ERR_GEOMETRY


def test_destroyed_detector_is_detached(pa):
    """Destroying a detector that a backend uses detaches it at the C ABI: the
    backend's next step reports PA_ERR_INVALID (no detector) with its state
    unchanged, a new detector can be attached, and destroying the backend
    afterwards is clean."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(1)
    m = sc.mesh()
    b = pa.ADMMBackendHIP()
    b.apply_config(cfg)
    b.set_constraints(sc)
    b.set_constraint_dim(sc.info["m_rows"])
    b.finalize_constraints()
    b.init(m["x"], sc.mass(), sc.info["n_dyn"], sc.surface_flags(), m["pins"])
    det = pa.CollisionDetector.for_scene(sc, capacity=cfg.max_contacts, thickness=cfg.thickness)
    b.attach_detector(det)
    b.step()
    x1 = b.get_state()[0]
    pa.lib().pa_detector_destroy(det._h)
    det._h = None
    b._detector = None
    with pytest.raises(pa.PAError) as e:
        b.step()
    assert e.value.code == pa.PA_ERR_INVALID
    np.testing.assert_array_equal(b.get_state()[0], x1)
    det2 = pa.CollisionDetector.for_scene(sc, capacity=cfg.max_contacts, thickness=cfg.thickness)
    b.attach_detector(det2)
    b.step()
    del b


def test_step_with_point_track_matches_oracle(pa):
    """The sphere under a draped cloth follows a point sequence (rising and
    swelling, 1 frame per step): one step from a common state per frame within
    1e-5 of the oracle (step_err), same contact counts, and the obstacle's
    positions and velocities equal to the oracle's (both FP64)."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(4, side=24, radius=0.2, drop=0.002)
    m = sc.mesh()
    n, n_all = sc.info["n_dyn"], sc.info["n_all"]
    rest = m["x"][n:]
    seq = np.stack([rest * (1.0 + 0.002 * k) + [0.0, 0.0005 * k, 0.0] for k in range(12)])
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    b.add_point_track(n, n_all - n, seq)
    o = _oracle(m, cfg)
    o.add_point_track(n, n_all - n, seq)
    worst, contacts = 0.0, 0
    for f in range(6):
        x, v = b.get_state()
        ue, uc = b.get_duals()
        o.set_state(x, v)
        o.set_duals(ue, uc)
        st = b.step()
        so = o.step()
        xg, vg = b.get_state()
        xo, vo = o.state()
        np.testing.assert_array_equal(xg[n:], xo[n:])
        np.testing.assert_allclose(vg[n:], vo[n:], rtol=1e-12, atol=1e-12)
        e = step_err(xg, xo, x, n)
        worst = max(worst, e)
        contacts += st["n_contacts"]
        assert st["n_contacts"] == so["n_contacts"]
        print(f"point track frame {f}: contacts {st['n_contacts']}, step err {e:.2e}, |v_static| {np.abs(vg[n:]).max():.4f}")
    assert worst < 1e-5 and contacts > 0
    np.testing.assert_array_equal(b.track_frames(), [7])


def _stacked_sheets(pa, layers, side, spacing, gap):
    """Square sheets exactly one above the other, `gap` apart, as one mesh."""
    k = np.arange(side * side)
    sheet = spacing * np.stack([k // side, np.zeros(side * side), k % side], axis=1)
    x = np.concatenate([sheet + [0, gap * q, 0] for q in range(layers)])
    c = (side * np.arange(side - 1)[:, None] + np.arange(side - 1)).ravel()
    cell = np.concatenate([np.stack([c, c + 1, c + side], axis=1), np.stack([c + 1, c + side + 1, c + side], axis=1)])
    tris = np.concatenate([cell + q * side * side for q in range(layers)])
    return x, pa.Scene.from_mesh(x, len(x), np.full(len(x), 1.0), tris=tris, tri_k=np.full(len(tris), 1e3))


def test_overflowing_detection_falls_back_inside_a_step(pa):
    """Eight sheets within the contact distance of each other: more close leaves
    than the queries' slabs (16 each) and the overflow list (one entry per query)
    hold, so a detection reruns as the single pass by itself.  Its list is the
    oracle's, and steps with it are the forced single pass's, bit for bit."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    cfg.max_contacts = 1 << 18
    cfg.admm_max_iter = 6  # two detections
    d = cfg.thickness
    x, sc = _stacked_sheets(pa, 8, 8, 0.01, 0.1 * d)
    t = sc.topology()["surf_tris"].reshape(-1, 3)
    lo, hi = x[t].min(axis=1), x[t].max(axis=1)
    near = np.all((x[:, None] >= lo - d) & (x[:, None] <= hi + d), axis=2)
    near[t, np.arange(len(t))[:, None]] = False
    assert near.sum() > 17 * len(x)  # vertex queries alone overflow the list
    o = _oracle(sc.mesh(), cfg)
    o.detect(x, brute_force=True)
    out = []
    for single in (False, True):
        det = _detector(pa, sc, cfg)
        det.set_single_pass(single)
        det.detect(x)
        _check_contacts_equal(*det.contacts(), *o.contacts())
        b = pa.ADMMBackendHIP.from_scene(sc, cfg)
        b.attach_detector(det)
        nc = [b.step()["n_contacts_max"] for _ in range(2)]
        out.append((*b.get_state(), *b.get_duals()))
    print(f"{near.sum()} close pairs of {len(x)} vertices, contacts per step {nc}")
    assert min(nc) > 2048
    for a, c in zip(*out):
        np.testing.assert_array_equal(a, c)


def test_overflowing_detection_of_many_waves(pa):
    """Eight sheets of 3,600 vertices: some waves of the collect pass fill the
    overflow list, the others stop where they meet it full.  The list is the
    forced single pass's, and the detector's next detection, of the sheets moved
    apart, is a fresh one's."""
    d = 1e-3
    x, sc = _stacked_sheets(pa, 8, 60, 0.01, 0.1 * d)
    apart = x * [1, 20, 1]
    apart[:3600, 1] = apart[3600, 1] + 0.5 * d  # two sheets stay close
    dets = [pa.CollisionDetector.for_scene(sc, 1 << 21, d) for _ in range(2)]
    dets[1].set_single_pass(True)
    for pos in (x, apart, x):
        n = [det.detect(pos) for det in dets]
        lists = [det.contacts() for det in dets]
        print(f"{n} contacts")
        assert n[0] == n[1] > 0
        np.testing.assert_array_equal(lists[0][0], lists[1][0])
        np.testing.assert_array_equal(lists[0][1], lists[1][1])


def test_single_pass_step_matches_two_pass_step(pa):
    """A step whose detections run the single pass (which also counts and places
    every vertex's contacts for the step) against one with the two passes, bit
    for bit: a draped cloth (one contact per lane of the sweeps), a small folded
    one (two per lane) and a larger one (a launch per sweep)."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    sc = pa.Scene.generate(1)
    cases = [(sc, drape_on_obstacle(sc, cfg.thickness))]
    for side in (11, 24):
        xf, scf = folded_cloth(side=side, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.15 * cfg.thickness, seed=3)
        cases.append((scf, xf))
    peaks = []
    for scene, x0 in cases:
        out = []
        for single in (False, True):
            det = _detector(pa, scene, cfg)
            det.set_single_pass(single)
            b = pa.ADMMBackendHIP.from_scene(scene, cfg)
            b.attach_detector(det)
            b.set_state(x=x0)
            nc = [b.step()["n_contacts_max"] for _ in range(2)]
            out.append((*b.get_state(), *b.get_duals()))
        peaks.append(max(nc))
        for a, c in zip(*out):
            np.testing.assert_array_equal(a, c)
    print(f"contacts {peaks}")
    assert 0 < peaks[0] <= 1024 < peaks[1] <= 2048 < peaks[2]


@pytest.mark.parametrize("edges", [16383, 16384, 16385])
def test_detector_at_the_small_build_limit(pa, edges):
    """The last sizes whose leaves one workgroup sorts and the first beyond: the
    list of a folded cloth cut to `edges` edges is that of the same edges with
    others far away, 20,000 in all, which are sorted by the launches."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    x, sc = folded_cloth(side=76, spacing=0.01, gap=0.5 * cfg.thickness, jitter=0.15 * cfg.thickness, seed=7)
    t = sc.topology()
    e = t["surf_edges"].reshape(-1, 2)[:edges]
    assert len(e) == edges
    n = len(x)
    lists = []
    for far in (0, 20000 - edges):
        k = np.arange(2 * far)
        xx = np.concatenate([x, np.stack([9 + 0.1 * k, 9 + 0 * k, 9 + 0 * k], axis=1)])
        ee = np.concatenate([e, n + k.reshape(-1, 2)])
        det = pa.CollisionDetector(len(xx), n, t["surf_verts"], t["surf_tris"], ee, 1 << 18, cfg.thickness)
        det.detect(xx)
        lists.append(det.contacts())
    print(f"{edges} edges: {len(lists[0][0])} contacts")
    assert len(lists[0][0]) > 2000
    np.testing.assert_array_equal(lists[0][0], lists[1][0])
    np.testing.assert_array_equal(lists[0][1], lists[1][1])


@pytest.mark.parametrize("side,refine,interval,precond", [(32, 2, 1, 2), (66, 2, 1, 2), (32, 1, 2, 2), (32, 1, 3, 2), (32, 1, 2, 1)])
def test_refinement_and_check_interval_match_oracle(pa, side, refine, interval, precond):
    """Two refinement passes per global solve (the second reads the stored
    right-hand side), and a residual check every second or third iteration
    (which reads the local step kept one iteration back), to the bars of
    test_step_matches_fp64_oracle."""
    from parallel_admm_amd.configs import config_for

    cfg = config_for("cloth32")
    cfg.residual_tol, cfg.global_refine, cfg.residual_interval, cfg.precond = 1e-4, refine, interval, precond
    sc = pa.Scene.generate(4, side=side, radius=0.2, drop=0.002)
    n = sc.info["n_dyn"]
    b = pa.ADMMBackendHIP.from_scene(sc, cfg)
    o = _oracle(sc.mesh(), cfg)
    contacts = 0
    for f in range(6):
        x, v = b.get_state()
        o.set_state(x, v)
        o.set_duals(*b.get_duals())
        n_log = len(o.residual_log())
        st, so = b.step(), o.step()
        contacts += st["n_contacts"]
        e = step_err(b.get_state()[0], o.state()[0], x, n)
        rg, ro = b.residual_log(), o.residual_log()[n_log:]
        k = min(len(rg), len(ro))
        dr = float(np.max(np.abs(rg[:k] - ro[:k]) / (np.abs(ro[:k]) + 1e-3)))
        print(f"frame {f}: contacts {st['n_contacts']}, iterations {st['iterations']} oracle {so['iterations']}, checks {len(rg)}, "
              f"step err {e:.2e}, residual rel diff {dr:.2e}")
        assert k > 0 and abs(len(rg) - len(ro)) <= 1 and abs(st["iterations"] - so["iterations"]) <= interval
        assert e < 1e-5 and dr < 1e-3
    assert contacts > 0
