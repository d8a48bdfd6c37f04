"""Launch shapes that depend on the grid: each rule at the sizes where its
choice changes, against the CPU oracle (FP64, <= 1e-12 relative L2)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import chanflow as cf
import oracle_lib as ol

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def step_parity(shape, steps, seed=5, **kw):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="tanh", dt=5e-4, nu=1.0 / 2800.0, **kw)
    f = cf.initial_fields(cfg, seed=seed)
    names = "uvwc" if cfg.scalar else "uvw"
    orc = ol.OracleRun(ol.oracle_cfg(cfg, cf.grid_dz(cfg)))
    for n in names:
        orc.put(n, f[n])
    orc.project_ic(1.0)
    init = {n: orc.get(n) for n in names}
    orc.steps(steps)
    with cf.Run(cfg) as run:
        for n in names:
            run.upload(n, init[n])
        run.step(steps)
        run.sync()
        errs = {n: rel(run.download(n), orc.get(n)) for n in names}
    assert max(errs.values()) <= 1e-12, errs


# z-chunks of the fused RHS: one level each (also nz = 2, all walls), two
# levels with a shorter last chunk, four, five, and the 16-level cap
@pytest.mark.parametrize("shape", [(8, 6, 2), (16, 12, 17), (64, 64, 49), (200, 90, 35), (96, 96, 41), (256, 256, 97)])
def test_rhs_chunk_lengths(shape):
    step_parity(shape, 2)


# every field of the general right-hand side in one launch, and the
# constraint from weighted sums of the right-hand side beside the z solve:
# blocks with idle lanes and rows, one level a block, the nz = 257 system
# that Thomas solves, the order-4 tiles and the per-field order-4 kernels
@pytest.mark.parametrize("shape,kw", [((6, 6, 3), dict(scalar=1)), ((64, 9, 4), dict(scalar=1, betg_z=0.1)),
                                      ((16, 6, 257), dict()), ((16, 6, 257), dict(scalar=1)),
                                      ((32, 8, 9), dict(order=4, scalar=1)), ((30, 9, 7), dict(order=4, scalar=1))])
def test_constraint_beside_the_solve(shape, kw):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="tanh", dt=1e-3, nu=1.0 / 500.0, uframe=0.3,
                    want_cvolavg=0.1, cvolavgmode=kw.get("scalar", 0), **kw)
    f = cf.initial_fields(cfg, seed=9)
    names = "uvwc" if cfg.scalar else "uvw"
    orc = ol.OracleRun(ol.oracle_cfg(cfg, cf.grid_dz(cfg)))
    for n in names:
        orc.put(n, f[n])
    orc.project_ic(1.0)
    init = {n: orc.get(n) for n in names}
    want = orc.steps(4)
    with cf.Run(cfg) as run:
        for n in names:
            run.upload(n, init[n])
        run.step(4)
        got = run.log()
        for n in names:
            assert rel(run.download(n), orc.get(n)) <= 1e-12, n
    # forcings divide a cancellation by the unit response: absolute (test_gpu_parity.check_log)
    for col in range(13):
        assert np.allclose(got[:, col], want[:, col], rtol=1e-10, atol=1e-10), cf.LOG_COLUMNS[col]


# FFT lengths with a run-time plan (each radix alone and together, one line
# pair a workgroup, several workgroups of a short last one) and compiled ones
@pytest.mark.parametrize("shape", [(90, 75, 3), (45, 27, 41), (2, 3, 2), (18, 54, 200), (1215, 4, 2), (2048, 2, 3), (125, 2, 5),
                                   (64, 50, 9), (96, 15, 7), (128, 36, 5)])
def test_fft3d_lengths(shape):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="uniform")
    a = np.random.default_rng(3).standard_normal(cfg.shape)
    ref = np.fft.fft(np.fft.rfft(a, axis=0) / cfg.nx, axis=1) / cfg.ny
    with cf.Run(cfg) as run:
        spec = run.fft3d_fwd(a)
        back = run.fft3d_bwd(spec)
    assert np.abs(spec - ref).max() <= 1e-14 * np.abs(ref).max() * np.log2(cfg.nx * cfg.ny)
    assert np.abs(back - a).max() <= 1e-13 * np.abs(a).max()


# the divergence + x FFT at its pair counts: through the projection, which
# leaves the velocity free of divergence
@pytest.mark.parametrize("prec,tol", [(cf.CF_FP64, 1e-11), (cf.CF_FP32, 2e-3)])
@pytest.mark.parametrize("shape", [(64, 6, 3), (128, 9, 4), (96, 8, 5), (90, 15, 4), (24, 40, 33), (512, 6, 4), (600, 6, 4)])
def test_divergence_pair_counts(shape, prec, tol):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="uniform", precision=prec)
    f = cf.initial_fields(cfg, seed=2)
    with cf.Run(cfg) as run:
        for n in "uvw":
            run.upload(n, f[n])
        before = run.max_divergence()
        run.project(1.0)
        assert run.max_divergence() <= tol * before


# ... and of grids with lines enough for full workgroups of them (from 512):
# the fewest such lines and just below, an odd line and a short last
# workgroup, compiled lengths and run-time plans
@pytest.mark.parametrize("prec,tol", [(cf.CF_FP64, 1e-11), (cf.CF_FP32, 2e-3)])
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("shape", [(320, 32, 64), (384, 48, 43), (480, 45, 47), (512, 36, 64), (512, 30, 64), (300, 48, 64),
                                   (300, 48, 63), (400, 75, 31), (200, 75, 69)])
def test_divergence_pair_counts_many_lines(shape, order, prec, tol):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="uniform", order=order, precision=prec)
    f = cf.initial_fields(cfg, seed=2)
    with cf.Run(cfg) as run:
        for n in "uvw":
            run.upload(n, f[n])
        before = run.max_divergence()
        run.project(1.0)
        assert run.max_divergence() <= tol * before
        if prec == cf.CF_FP64:
            a = np.random.default_rng(3).standard_normal(cfg.shape)
            ref = np.fft.fft(np.fft.rfft(a, axis=0) / cfg.nx, axis=1) / cfg.ny
            got = run.fft3d_fwd(a)
            assert np.abs(got - ref).max() <= 1e-14 * np.abs(ref).max() * np.log2(cfg.nx * cfg.ny)


# rows per wave and columns per march of the spectra, levels and partials of
# the plane sums
@pytest.mark.parametrize("shape", [(2, 6, 3), (12, 6, 5), (16, 64, 4), (18, 135, 3), (45, 27, 7), (90, 80, 5)])
def test_statistics_launch_shapes(shape):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="uniform")
    nx, ny = cfg.nx, cfg.ny
    rng = np.random.default_rng(5)
    with cf.Run(cfg) as run:
        f = {}
        for n in "uv":
            f[n] = 0.3 + rng.standard_normal(cfg.shape)
            run.upload(n, f[n])
        for a, b in ("uu", "uv"):
            s = [np.fft.fft(np.fft.rfft(f[n], axis=0) / nx, axis=1) / ny for n in (a, b)]
            q = s[0] * s[1].conj()
            q[0, 0] = 0
            sx, sy = run.xy_stats("spec", a, b)
            inner = q[1:(nx + 1) // 2].sum(0)
            mirror = np.conj(inner[-np.arange(ny // 2 + 1) % ny])
            want = q.sum(0)[:ny // 2 + 1] + mirror
            # sums of at most nx ny products: a few units of rounding of the largest
            scale = 1e-13 * np.abs(q).sum(axis=(0, 1)).max()
            assert np.abs(sx - q.sum(1)).max() <= scale and np.abs(sy - want).max() <= scale
            d = [f[n] - f[n].mean(axis=(0, 1)) for n in (a, b)]
            assert np.abs(run.xy_stats("corr", a, b) - (d[0] * d[1]).mean(axis=(0, 1))).max() <= 1e-13
            assert np.abs(run.xy_stats("avg", b) - f[b].mean(axis=(0, 1))).max() <= 1e-13
        assert np.abs(run.xy_stats("moment", "u", en=3.0) - ((f["u"] - f["u"].mean(axis=(0, 1))) ** 3).mean(axis=(0, 1))).max() <= 1e-11


# the fully implicit driver's solves of all fields in one launch: an odd
# number of cells, w's faces in a shorter chunk than the cells, one thread a
# mode (rounding grows as nz^2), and order 4's solves field by field
@pytest.mark.parametrize("shape,kw,tol", [((9, 9, 9), dict(), 1e-12), ((15, 9, 7), dict(scalar=1), 1e-12),
                                          ((16, 6, 33), dict(scalar=1), 1e-12), ((6, 6, 520), dict(), 4e-12),
                                          ((16, 8, 7), dict(order=4, scalar=1), 1e-12)])
def test_implicit_solves_together(shape, kw, tol):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="tanh", dt=1e-3, nu=1.0 / 500.0,
                    driver=cf.CF_DRIVER_CHANNEL, **kw)
    f = cf.initial_fields(cfg, seed=4)
    names = "uvwc" if cfg.scalar else "uvw"
    orc = ol.OracleRun(ol.oracle_cfg(cfg, cf.grid_dz(cfg)))
    for n in names:
        orc.put(n, f[n])
    orc.project_ic(1.0)
    init = {n: orc.get(n) for n in names}
    orc.steps(4)
    with cf.Run(cfg) as run:
        for n in names:
            run.upload(n, init[n])
        run.step(4)
        for n in names:
            assert rel(run.download(n), orc.get(n)) <= tol, n


# plain downloads, and from 32 MB on in chunks by several threads, the last
# chunk whole or short; two threads downloading at once
@pytest.mark.parametrize("shape", [(64, 64, 32), (90, 75, 50), (256, 128, 65), (256, 128, 128), (256, 150, 125)])
def test_download_chunks(shape):
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="uniform")
    rng = np.random.default_rng(6)
    with cf.Run(cfg) as one, cf.Run(cfg) as two, ThreadPoolExecutor(2) as pool:
        a = {n: rng.standard_normal(cfg.shape) for n in "uv"}
        for run in (one, two):
            for n in a:
                run.upload(n, a[n])
        got = list(pool.map(lambda q: [q[0].download(q[1]) for _ in range(3)], [(one, "u"), (two, "v")]))
    for n, downloads in zip("uv", got):
        for g in downloads:
            assert np.array_equal(g, a[n])


# the Poisson solve's chunk lengths, with a short group of modes and a short
# last chunk; the projection leaves what rounding times the condition leaves
@pytest.mark.parametrize("prec,tol,per_nz2", [(cf.CF_FP64, 1e-11, 1e-15), (cf.CF_FP32, 2e-3, 1e-6)])
@pytest.mark.parametrize("nz", [3, 17, 47, 100, 176, 193, 230, 257, 300, 400, 512, 513])
def test_poisson_chunk_lengths(nz, prec, tol, per_nz2):
    cfg = cf.Config(nx=12, ny=6, nz=nz, stretch="uniform", precision=prec)
    f = cf.initial_fields(cfg, seed=2)
    with cf.Run(cfg) as run:
        for n in "uvw":
            run.upload(n, f[n])
        before = run.max_divergence()
        run.project(1.0)
        assert run.max_divergence() <= (tol + per_nz2 * nz * nz) * before


# the projection's workgroups: rows of whole waves with a short last group of
# rows, and consecutive cells, in runs that project in place and in those
# whose state is materialised (one component, then all)
@pytest.mark.parametrize("shape,kw", [((64, 6, 5), dict()), ((128, 9, 6), dict(scalar=1)), ((64, 9, 7), dict(order=4, scalar=1)),
                                      ((60, 9, 7), dict(order=4)), ((90, 10, 5), dict()), ((192, 20, 4), dict()), ((160, 9, 5), dict()),
                                      ((120, 6, 6), dict(order=4))])
def test_projection_workgroups(shape, kw):
    step_parity(shape, 2, **kw)
    cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], stretch="tanh", dt=5e-4, **kw)
    f = cf.initial_fields(cfg, seed=3)
    with cf.Run(cfg) as run:
        for n in f if cfg.scalar else "uvw":
            run.upload(n, f[n])
        run.step(2)
        one = {n: run.xy_stats("avg", n) for n in "uvw"}      # materialises one component
        for n in "uvw":
            assert np.abs(one[n] - run.download(n).mean(axis=(0, 1))).max() <= 1e-13


# the same chunk lengths in FP32 against the FP64 solve of the same input, on
# a grid whose modes past the FP64 ones take 18 workgroups, the last a short
# one.  FP32 rounds the fields (three times), the transforms (log2 of 768
# points) and the solves, whose modes past |k| = 4 have a condition of at most
# 4 (nz / lz)^2 / 25
@pytest.mark.parametrize("nz", [17, 33, 47, 64, 79, 95, 111, 127, 143, 159, 175, 191, 193, 223, 239, 255, 257, 321, 385, 449, 512])
def test_poisson_fp32_against_fp64(nz):
    got = {}
    for prec in (cf.CF_FP64, cf.CF_FP32):
        cfg = cf.Config(nx=32, ny=24, nz=nz, lz=2.0, stretch="uniform", precision=prec)
        f = cf.initial_fields(cfg, seed=2)
        with cf.Run(cfg) as run:
            for n in "uvw":
                run.upload(n, f[n])
            run.project(1.0)
            got[prec] = {n: run.download(n) for n in "uvw"}
    tol = 2.0 ** -24 * (3 + np.log2(768) + 4 * (nz / 2.0) ** 2 / 25)
    for n in "uvw":
        assert rel(got[cf.CF_FP32][n], got[cf.CF_FP64][n]) <= tol, n


# the divergence's pair counts in FP32 against FP64, to the same roundings and
# that of p, which its differences raise by at most max(nx, ny) / pi
@pytest.mark.parametrize("shape", [(64, 6, 3), (128, 9, 4), (128, 10, 4), (96, 8, 5), (90, 15, 4), (24, 40, 33), (256, 6, 5), (512, 6, 4),
                                   (600, 6, 4)])
def test_projection_fp32_against_fp64(shape):
    got = {}
    for prec in (cf.CF_FP64, cf.CF_FP32):
        cfg = cf.Config(nx=shape[0], ny=shape[1], nz=shape[2], lz=2.0, stretch="uniform", precision=prec)
        f = cf.initial_fields(cfg, seed=2)
        with cf.Run(cfg) as run:
            for n in "uvw":
                run.upload(n, f[n])
            run.project(1.0)
            got[prec] = {n: run.download(n) for n in "uvw"}
    tol = 2.0 ** -24 * (3 + np.log2(shape[0] * shape[1]) + 4 * (shape[2] / 2.0) ** 2 / 25 + max(shape[:2]) / np.pi)
    for n in "uvw":
        assert rel(got[cf.CF_FP32][n], got[cf.CF_FP64][n]) <= tol, n


# batches over lengths with a divergence + x FFT of their own (192 only in
# FP64) and lengths on the run-time plan, an odd number of lines in the last
# pair group: each run against the oracle
@pytest.mark.parametrize("shapes,prec,tol", [([(192, 9, 5), (90, 15, 7), (64, 9, 6)], cf.CF_FP64, 1e-12),
                                             ([(48, 6, 33), (96, 9, 5), (128, 9, 5), (192, 6, 17), (32, 15, 9)], cf.CF_FP64, 1e-12),
                                             ([(192, 9, 5), (96, 9, 7), (128, 15, 9), (90, 6, 6)], cf.CF_FP32, 5e-5)])
def test_batched_lengths(shapes, prec, tol):
    cfgs = [cf.Config(nx=s[0], ny=s[1], nz=s[2], stretch="tanh", dt=5e-4, nu=1.0 / (2000.0 + 500.0 * q), precision=prec)
            for q, s in enumerate(shapes)]
    cases = []
    for q, c in enumerate(cfgs):
        f = cf.initial_fields(c, seed=60 + q)
        orc = ol.OracleRun(ol.oracle_cfg(c, cf.grid_dz(c)))
        for n in "uvw":
            orc.put(n, f[n])
        orc.project_ic(1.0)
        cases.append((orc, {n: orc.get(n) for n in "uvw"}))
    with cf.Batch(cfgs) as b:
        for q, (orc, init) in enumerate(cases):
            for n in "uvw":
                b.upload(q, n, init[n])
        b.step(8)
        for q, (orc, _) in enumerate(cases):
            orc.steps(8)
            for n in "uvw":
                assert rel(b.download(q, n), orc.get(n)) <= tol, (shapes[q], n)
