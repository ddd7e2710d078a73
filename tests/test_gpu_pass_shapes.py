"""The engine's passes at the edges of their lengths and row shapes, and the
trial's control launches.

Tolerances: fields 5e-6 of the largest against the FP64 oracle (FP32 transforms,
a few 1e-7 x log2 P); launch shapes and the way trials are driven change no bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CELL = (4e-9, 3e-9, 5e-9)


def cfg_of(size, m0, **kw):
    c = dict(size=size, cellsize=CELL, msat=8e5, aexch=1.3e-11, alpha=0.1, solver="rk4", dt=2e-14, m0=m0)
    c.update(kw)
    return c


def random_m(size, seed):
    m = np.random.default_rng(seed).standard_normal((3,) + size)
    return (m / np.linalg.norm(m, axis=0)).astype(np.float32)


# padded Y 4, 6, 8, 12, 64, 96, 128, 1024, 1536, 2048, 4096: one lane group per wave up to one block per line
@pytest.mark.parametrize("ny", [2, 3, 4, 5, 31, 47, 64, 400, 700, 1000, 1600])
def test_film_column_lengths_vs_oracle(mm, orc, ny):
    size = (1, ny, 5)
    m0 = random_m(size, ny)
    s = mm.workloads.make_sim(cfg_of(size, m0))
    o = orc.sim(m0, **mm.workloads.oracle_kwargs(cfg_of(size, m0)))
    h = s.heff(m0)
    ref = o.heff(m0).reshape(h.shape)
    s.free()
    assert np.abs(h - ref).max() < 5e-6 * np.abs(ref).max()


# 1025..1536 cells are padded to 3072, the longest 3 * 2^a: columns, rows, and the Y passes of a 3-D grid
@pytest.mark.parametrize("size", [(1, 1100, 5), (1, 3, 1536), (2, 1025, 3), (2, 2, 1201)])
def test_axes_padded_to_3072(mm, orc, size):
    m0 = random_m(size, 4)
    cfg = cfg_of(size, m0, solver="rkdp", maxerror=1e-4, dt=1e-14, max_dt=1e-14)
    s = mm.workloads.make_sim(cfg)
    o = orc.sim(m0, **mm.workloads.oracle_kwargs(cfg))
    h = s.heff(m0)
    ref = o.heff(m0).reshape(h.shape)
    assert np.abs(h - ref).max() < 5e-6 * np.abs(ref).max()
    t = mm.workloads.make_sim(cfg)
    b = mm.Batch([t])
    b.start(steps=2)
    while b.trials(2):
        pass
    b.free()
    s.steps(2)
    assert s.state()["steps"] == t.state()["steps"] == 2
    assert np.array_equal(s.m, t.m)
    dts, acc = s.trial_log()
    assert all(acc) and len(dts) == 2
    o.step_replay(dts[:1], acc[:1])
    o.step_replay(dts[1:], acc[1:])
    dm = np.abs(s.m.reshape(-1) - np.asarray(o.m).reshape(-1)).max()
    for x in (s, t):
        x.free()
    assert dm < 1e-5


# every tableau's stages with their forward passes in the epilogues: even and odd rows, the shortest, partly
# filled tiles, and the dt control after the first stage (which keeps the passes apart)
@pytest.mark.parametrize("solver", ["rk2", "rk12", "rk3", "rk23", "rk4", "rkck", "rkdp"])
@pytest.mark.parametrize("size,kw", [((1, 21, 30), {}), ((3, 9, 51), {}), ((2, 12, 3), {}), ((2, 5, 2), {}),
                                     ((4, 10, 16), {"max_dt": 1.5e-14})])
def test_fused_stages_vs_oracle(mm, orc, solver, size, kw):
    m0 = random_m(size, 9)
    cfg = cfg_of(size, m0, solver=solver, dt=1e-14, maxerror=1e-4, field=("static", (1e-2, 2e-2, -3e-2)), **kw)
    s = mm.workloads.make_sim(cfg)
    s.steps(6)
    dts, acc = s.trial_log()
    o = orc.sim(m0, **mm.workloads.oracle_kwargs(cfg))
    i = 0
    while i < len(dts):
        j = i
        while not acc[j]:
            j += 1
        o.step_replay(dts[i:j + 1], acc[i:j + 1])
        i = j + 1
    assert s.state()["steps"] == 6
    dm = np.abs(s.m.reshape(-1) - np.asarray(o.m).reshape(-1)).max()
    s.free()
    assert dm < 1e-5


# row lengths of every part of the Z kernels, odd and even, with partly filled row tiles
@pytest.mark.parametrize("size", [(2, 9, 40), (3, 21, 51), (1, 17, 130), (1, 35, 301), (2, 5, 640), (1, 3, 1601)])
def test_row_variants_give_the_same_steps(mm, lib, tmp_path, size):
    m0 = random_m(size, 3)
    out = []
    try:
        for zr, er in [(0, 0), (1, 1), (2, 2), (3, 1), (4, 3)]:
            table = tmp_path / "t.txt"
            table.write_text("%d %d %d %d %d 8 4 8 0 0\n" % (size + (zr, er)))
            lib.mm_tune_clear()
            assert lib.mm_tune_load(str(table).encode()) == 1
            s = mm.workloads.make_sim(cfg_of(size, m0, solver="rkdp", maxerror=1e-4, dt=1e-14, max_dt=1e-14))
            s.steps(3)
            out.append(s.m)
            s.free()
    finally:
        lib.mm_tune_clear()
        lib.mm_tune_load(mm.gpukern.TUNE_TABLE.encode())
    for m in out[1:]:
        assert np.array_equal(m, out[0])


@pytest.mark.parametrize("solver", ["rkdp", "rk23", "rkck", "rk4"])
@pytest.mark.parametrize("size", [(2, 12, 30), (9, 40, 4)])
def test_runs_steps_and_batches_take_the_same_trials(mm, solver, size):
    """A first-same-as-last stage carried over, step by step, in one go and
    through a batch between two runs of the simulation alone; the batch's blocks
    (and so its per-block maxima) are others than the simulation's own, and of the
    short rows there are more blocks than blocks of 256 cells."""
    kw = dict(solver=solver, maxerror=1e-5, dt=1e-14)
    res = []
    for how in ("go", "single", "batch"):
        s = mm.workloads.make_sim(cfg_of(size, random_m(size, 1), **kw))
        if how == "go":
            s.steps(13)
        elif how == "single":
            for _ in range(13):
                s.steps(1)
        else:
            s.steps(4)
            b = mm.Batch([s])
            b.start(steps=5)
            while b.trials(4):
                pass
            b.free()
            s.steps(4)
        assert s.state()["steps"] == 13
        dts, acc = s.trial_log()
        res.append((s.m, dts, acc))
        s.free()
    for r in res[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(r, res[0]))


def test_run_to_a_stop_time_in_pieces(mm):
    """run_until in pieces that end on step boundaries takes the steps of one run."""
    size = (1, 16, 24)
    a, b = (mm.workloads.make_sim(cfg_of(size, random_m(size, 2), solver="rkdp", maxerror=1e-5, dt=0.0)) for _ in "ab")
    n = a.run(2e-12)
    stop = a.state()["time"]
    b.run(0.0)
    k = 0
    for f in (0.1, 0.5, 0.9, 1.0):
        k += b.run_until(f * stop)
    assert k == n and np.array_equal(a.m, b.m) and np.array_equal(a.trial_log()[0], b.trial_log()[0])
    a.free()
    b.free()


# padded X of every X.K.X kernel: an item per block (24 to 128, 256 to 512) and walked with a prefetch (192)
@pytest.mark.parametrize("size", [(9, 34, 4), (13, 9, 4), (40, 3, 6), (50, 4, 5), (66, 5, 6), (96, 34, 2), (100, 3, 4),
                                  (130, 6, 5), (192, 9, 3), (200, 4, 4)])
def test_x_axis_lengths_vs_oracle(mm, orc, size):
    m0 = random_m(size, 6)
    cfg = cfg_of(size, m0, solver="rkdp", maxerror=1e-4, dt=1e-14, max_dt=1e-14)
    s, t = mm.workloads.make_sim(cfg), mm.workloads.make_sim(cfg)
    o = orc.sim(m0, **mm.workloads.oracle_kwargs(cfg))
    h = s.heff(m0)
    ref = o.heff(m0).reshape(h.shape)
    assert np.abs(h - ref).max() < 5e-6 * np.abs(ref).max()
    s.steps(2)
    b = mm.Batch([t])
    b.start(steps=2)
    b.trials(2)
    b.free()
    assert np.array_equal(s.m, t.m)
    for x in (s, t):
        x.free()


def test_a_relaxation_enqueues_no_further_than_its_end(mm):
    """A relaxed state ends its next relaxation within a few steps, also where many
    more are allowed: nearly all of 1024 trials enqueued at once would do nothing
    (each a dozen launches, some 25 us: 25 ms). The allowance of 5 ms is a fifth of that."""
    import time

    size = (1, 24, 40)
    m0 = np.zeros((3,) + size, np.float32)
    m0[2] = 1
    s = mm.workloads.make_sim(cfg_of(size, m0, alpha=1.0, dt=1e-13))
    s.relax(4000)
    took = {}
    for most in (0, 20000):
        took[most] = []
        for _ in range(4):
            s.sync()
            t = time.perf_counter()
            s.relax(most)
            took[most].append(time.perf_counter() - t)
    s.free()
    assert min(took[20000]) < min(took[0]) + 5e-3


# columns and rows of the drop-in plan: register lengths, LDS lengths, Bluestein lengths, their largest
@pytest.mark.parametrize("size,P", [((1, 11, 13), (1, 22, 26)), ((1, 2039, 3), (1, 2039, 6)), ((2, 1500, 3), (4, 3072, 6)),
                                    ((1, 4096, 4), (1, 4096, 8)), ((3, 7, 1536), (6, 14, 3072)), ((2, 9, 4078), (3, 9, 4078)),
                                    ((2, 3, 4050), (2, 6, 8100)), ((1, 3, 4096), (1, 6, 8192)), ((1, 5, 17), (1, 9, 17)), ((5, 8, 45), (10, 16, 45)),
                                    ((70, 6, 2), (140, 12, 4)), ((1, 33, 6), (1, 66, 12))])
def test_dropin_transform_lengths(lib, size, P):
    from test_zz_no_alloc import download, forward_both, i3, upload

    ref, got, npref = forward_both(lib, size, P, 5)
    assert np.array_equal(ref.view(np.uint32), got.view(np.uint32))  # the two calls run the same kernels
    assert np.abs(ref.view(np.complex64).reshape(npref.shape) - npref).max() < 2e-6 * np.abs(npref).max()
    plan = lib.new_gpuFFT3dPlan_padded(i3(*size), i3(*P))
    d, back = upload(lib, ref), lib.new_gpu_array(int(np.prod(size)))
    lib.gpuFFT3dPlan_inverse(plan, d, back)
    x = download(lib, back, int(np.prod(size))).reshape(size) / np.prod(P)
    want = np.random.default_rng(5).standard_normal(size).astype(np.float32)
    assert np.abs(x - want).max() < 2e-6 * np.abs(want).max() * np.log2(np.prod(P))
    for p in (d, back):
        lib.free_gpu_array(p)
    lib.delete_gpuFFT3dPlan(plan)


# the real data at the start of the spectrum's memory and further in: register rows, LDS rows, Bluestein rows, odd length
@pytest.mark.parametrize("size,P", [((4, 16, 32), (8, 32, 64)), ((2, 9, 15), (4, 18, 30)), ((2, 11, 13), (4, 22, 26)),
                                    ((3, 6, 45), (6, 12, 45)), ((1, 1, 2), (1, 1, 4))])
@pytest.mark.parametrize("call", ["gpuFFT3dPlan_forward", "gpuFFT3dPlan_forward_noalloc"])
def test_dropin_transform_of_shared_memory(lib, size, P, call):
    """Input and output that overlap give the bits that separate arrays give, both ways."""
    from test_zz_no_alloc import download, i3, upload

    n, n_out = int(np.prod(size)), P[0] * P[1] * 2 * (P[2] // 2 + 1)
    x = np.random.default_rng(8).standard_normal(size).astype(np.float32)
    plan = lib.new_gpuFFT3dPlan_padded(i3(*size), i3(*P))
    a, b, c = upload(lib, x), lib.new_gpu_array(n_out), lib.new_gpu_array(n)
    getattr(lib, call)(plan, a, b)
    spec = download(lib, b, n_out)
    lib.gpuFFT3dPlan_inverse(plan, b, c)
    back = download(lib, c, n)
    for at in (0, (n_out - n) // 4 * 2):
        d = lib.new_gpu_array(n_out)
        lib.memcpy_to_gpu(x.ctypes.data, d + 4 * at, n)
        getattr(lib, call)(plan, d + 4 * at, d)
        assert np.array_equal(download(lib, d, n_out).view(np.uint32), spec.view(np.uint32)), at
        lib.gpuFFT3dPlan_inverse(plan, d, d + 4 * at)
        assert np.array_equal(download(lib, d + 4 * at, n).view(np.uint32), back.view(np.uint32)), at
        lib.free_gpu_array(d)
    for p in (a, b, c):
        lib.free_gpu_array(p)
    lib.delete_gpuFFT3dPlan(plan)
