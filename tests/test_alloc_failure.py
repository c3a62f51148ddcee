"""Device allocations that fail: the call reports an error and the handle stays
usable, so the same call repeated leaves the allocations of a handle that never
failed (a size that is recorded before its allocation would be taken as
allocated from then on, and kernels would run on null buffers).  The library's
own host code runs on tests/fake_hip.cpp, a HIP runtime on host memory, in a
process of its own per test.  CPU only."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def fake_hip(tmp_path_factory):
    out = tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(out), os.path.join(ROOT, "tests", "fake_hip.cpp")], check=True)
    return str(out)


def _fails_everywhere(pa, fake, make, call):
    """`call` on fresh handles with each of its allocations failing in turn."""
    h = make()
    before, first = fake.fake_live(), fake.fake_allocs()
    call(h)
    want, count = fake.fake_live() - before, fake.fake_allocs() - first
    assert count > 0
    for k in range(1, count + 1):
        h = make()
        before = fake.fake_live()
        fake.fake_fail_at(k)
        try:
            call(h)
            raise AssertionError(f"allocation {k} of {count} failed unnoticed")
        except pa.PAError as e:
            assert e.code == pa.PA_ERR_HIP
        fake.fake_fail_at(0)
        call(h)
        assert fake.fake_live() - before == want, f"allocation {k} of {count}"


def _detector(pa, side):
    sc = pa.Scene.generate(4, side=side, radius=0.1)
    return pa.CollisionDetector.for_scene(sc, 1000, 1e-3), sc.mesh()["x"]


def network(pa, fake):
    x = np.zeros((100, pa.MLP_FEATURES), np.float32)
    t = np.zeros((100, pa.MLP_OUTPUTS), np.float32)
    rows = np.zeros((1000, 12), np.float32)
    for call in (lambda m: m.forward(x), lambda m: m.gradients(x, t), lambda m: m.adam_step(x, t, 1e-3),
                 lambda m: m.train(rows, 1, batch=96)):
        _fails_everywhere(pa, fake, pa.MLP, call)


def inference(pa, fake):
    """Inference holds its input and output rows (48 bytes each), none of the
    training buffers."""
    m, before = pa.MLP(), fake.fake_live()
    m.forward(np.zeros((4096, pa.MLP_FEATURES), np.float32))
    assert fake.fake_live() - before <= 4096 * 48 and fake.fake_launches(b"k_ones_rows") == 0
    m.forward(np.zeros((4097, pa.MLP_FEATURES), np.float32))
    assert fake.fake_live() - before <= 4097 * 48 + 4096 * 4  # the output grows by half


def noalloc_scratch(pa, fake):
    """The allocation-free forward's device array holds its input and output rows
    (48 bytes each) and nothing else."""
    assert fake.fake_var_bytes(b"scratch") == pa.MLP_NOALLOC_MAX_ROWS * 48


def detection(pa, fake):
    for side in (9, 90):  # leaves sorted in one workgroup, and by the radix sort with its scratch
        x = _detector(pa, side)[1]
        _fails_everywhere(pa, fake, lambda: _detector(pa, side)[0], lambda d: d.detect(x))


def single_pass(pa, fake):
    """The single pass, which a step falls back to in the middle of its work,
    allocates nothing of its own."""
    for side in (9, 90):
        d, x = _detector(pa, side)
        d.detect(x)
        before = fake.fake_allocs()
        d.set_single_pass(True)
        d.detect(x)
        assert fake.fake_launches(b"k_single") > 0 and fake.fake_allocs() == before


def segments(pa, fake):
    """A segmented detector keeps its segments when setting others fails."""
    d, x = _detector(pa, 9)
    d.set_segments(np.zeros(len(x), np.int32))
    d.detect(x)
    before, first = fake.fake_live(), fake.fake_allocs()
    d.set_segments(np.zeros(len(x), np.int32))
    for k in range(1, fake.fake_allocs() - first + 1):
        fake.fake_fail_at(k)
        try:
            d.set_segments(np.ones(len(x), np.int32))
            raise AssertionError("no error")
        except pa.PAError as e:
            assert e.code == pa.PA_ERR_HIP
        fake.fake_fail_at(0)
        assert fake.fake_live() == before
        d.detect(x)


def contact_log(pa, fake):
    """No step logs into a buffer that was not allocated."""
    from parallel_admm_amd.configs import config_for

    sc = pa.Scene.generate(4, side=9, radius=0.1)
    b = pa.ADMMBackendHIP.from_scene(sc, config_for("batch"))
    fake.fake_last_pinned()[0] = 5  # the contacts that a detection finds
    b.set_contact_log(1000)
    b.step()
    b.step()
    logged = fake.fake_launches(b"k_ws_log")
    assert logged > 0
    b.set_contact_log(0)
    fake.fake_fail_at(1)
    try:
        b.set_contact_log(2000)
        raise AssertionError("no error")
    except pa.PAError as e:
        assert e.code == pa.PA_ERR_HIP
    b.step()
    b.step()
    assert fake.fake_launches(b"k_ws_log") == logged


def creation(pa, fake):
    """A handle whose creation fails leaves nothing behind: no memory, stream,
    event or pinned slot."""
    from parallel_admm_amd.configs import config_for

    sc = pa.Scene.generate(4, side=9, radius=0.1)
    for make in (pa.MLP, lambda: _detector(pa, 9)[0], lambda: pa.ADMMBackendHIP.from_scene(sc, config_for("batch"))):
        before = fake.fake_live(), fake.fake_handles()
        first = fake.fake_allocs()
        make()
        count = fake.fake_allocs() - first
        assert (fake.fake_live(), fake.fake_handles()) == before and count > 0
        for k in range(1, count + 1):
            fake.fake_fail_at(k)
            try:
                make()
                raise AssertionError("no error")
            except pa.PAError as e:
                assert e.code == pa.PA_ERR_HIP
            fake.fake_fail_at(0)
            assert (fake.fake_live(), fake.fake_handles()) == before, f"allocation {k} of {count}"


def early_detector(pa, fake):
    """A detector attached before apply_config and init, when the backend's sizes
    are not known yet, is refused by init if it does not fit them: its contacts
    index per-vertex counts and fill per-contact buffers of the backend."""
    from parallel_admm_amd.configs import config_for

    sc, big = pa.Scene.generate(4, side=9, radius=0.1), pa.Scene.generate(4, side=10, radius=0.1)
    m = sc.mesh()
    for scene, capacity, fits in ((sc, 1000, True), (big, 1000, False), (sc, 2000, False)):
        cfg = config_for("batch")
        cfg.max_contacts = 1000
        b = pa.ADMMBackendHIP()
        b.attach_detector(pa.CollisionDetector.for_scene(scene, capacity, 1e-3))
        b.apply_config(cfg)
        b.set_constraints(sc)
        b.set_constraint_dim(sc.info["m_rows"])
        b.finalize_constraints()
        try:
            b.init(m["x"], sc.mass(), sc.info["n_dyn"], sc.surface_flags(), m["pins"])
            assert fits
            b.step()
        except pa.PAError as e:
            assert not fits and e.code == pa.PA_ERR_INVALID


@pytest.mark.parametrize("case", ["network", "detection", "single_pass", "segments", "contact_log", "creation"])
def test_failed_allocation(fake_hip, case):
    _run(fake_hip, case)


@pytest.mark.parametrize("case", ["inference", "noalloc_scratch"])
def test_inference_memory(fake_hip, case):
    _run(fake_hip, case)


def test_detector_attached_before_init(fake_hip):
    _run(fake_hip, "early_detector")


def _run(fake_hip, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake_hip, case], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    _fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    for _name in ("fake_live", "fake_var_bytes"):
        getattr(_fake, _name).restype = C.c_size_t
    for _name in ("fake_allocs", "fake_launches", "fake_handles"):
        getattr(_fake, _name).restype = C.c_long
    _fake.fake_last_pinned.restype = C.POINTER(C.c_uint32)
    sys.path.insert(0, ROOT)
    import parallel_admm_amd as _pa

    _pa.lib()
    globals()[sys.argv[2]](_pa, _fake)
