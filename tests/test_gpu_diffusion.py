"""GPU parity of BackwardEulerDiffusionSolver (viscosity), through the C ABI,
against the FP64 oracle on the same inputs.

Bars:
  * face markers of the diffusion solve -- bit-exact (FP64 SDF samples on both
    sides);
  * Jacobi sweep counts -- equal (same stopping rule, FP64 residual);
  * velocities after the solve -- the GPU's FP64 sweeps follow the oracle's
    operation order, so the FP32 result is the rounded FP64 value: within
    1e-6 relative of the field's magnitude (one FP32 rounding is 6e-8);
  * a full substep with viscosity -- markers bit-exact, velocities within the
    substep bar of the inviscid parity test (2e-4 relative).
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from fluide_engine_amd import capi  # noqa: E402
from oracle import oracle as orc  # noqa: E402

COMPS = ((capi.GRID_U, orc.U), (capi.GRID_V, orc.V), (capi.GRID_W, orc.W))
DMARK = (capi.GRID_DMU, capi.GRID_DMV, capi.GRID_DMW)


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def _pair(ctx, n, size, nu, seed):
    desc = capi.scene_desc(n, method=capi.FLIP, size=size, gravity=(0.0, 0.0, 0.0), viscosity=nu, max_particles=64)
    g = capi.Scene(ctx, desc)
    o = orc.Scene(n, size=size, method=orc.FLIP, blend=desc.blend, max_cfl=3.0, gravity=(0.0, 0.0, 0.0))
    o.set_viscosity(nu)
    rng = np.random.default_rng(seed)
    sdf = rng.uniform(-1.0, 0.7, (n[2], n[1], n[0]))
    g.set(capi.GRID_SDF, sdf)
    o.set(orc.SDF, sdf)
    for gf, of in COMPS:
        f = rng.normal(size=g.shape(gf)).astype(np.float32)
        g.set(gf, f)
        o.set(of, f.astype(np.float64))
    return g, o


def _free_bytes():
    """Device memory left, as the library's HIP runtime has it."""
    free, total = C.c_size_t(), C.c_size_t()
    assert capi.load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _compare(g, o, gst, ost, rtol=1e-6):
    for c, (gf, of) in enumerate(COMPS):
        assert np.array_equal(g.get(DMARK[c]), o.diffusion_markers(c)), f"markers {c}"
        assert gst[c].iterations == ost[c].iterations, (c, gst[c].iterations, ost[c].iterations)
        want = o.get(of)
        got = g.get(gf).astype(np.float64)
        scale = max(1.0, float(np.abs(want).max()))
        err = float(np.abs(got - want).max())
        assert err <= rtol * scale, f"component {c}: {err:.3e}"


@pytest.mark.parametrize("n,size,nu", [((20, 16, 12), (1.0, 0.9, 0.7), 0.01), ((17, 9, 23), (1.0, 1.0, 1.0), 0.002),
                                       ((8, 8, 8), (1.0, 1.0, 1.0), 0.3)])
def test_diffusion_stage_parity(ctx, n, size, nu):
    print(f"[gpu] diffusion stage n={n} nu={nu}", flush=True)
    g, o = _pair(ctx, n, size, nu, seed=sum(n))
    dt = 1.0 / 240
    g.run_stage(capi.STAGE_DIFFUSION, dt)
    ost = o.diffusion(dt)
    gst = g.last_diffusion_stats()
    _compare(g, o, gst, ost)
    assert all(s.converged for s in gst)
    g.close()


def test_diffusion_of_large_grids(ctx):
    """Above 2^22 faces the components are solved one after another, in 34
    bytes of buffers for each face of the largest component and a byte of
    markers for each of all: the same markers, counts and values."""
    n = (164, 162, 161)
    print(f"[gpu] diffusion stage n={n}", flush=True)
    g, o = _pair(ctx, n, (1.0, 0.9, 1.1), 0.02, seed=1)
    g.set_diffusion_solver(capi.solver(capi.SOLVER_JACOBI, 8, 3, 1e-30))
    o.set_diffusion_solver(orc.solver(orc.JACOBI, 8, 3, 1e-30))
    free = _free_bytes()
    g.run_stage(capi.STAGE_DIFFUSION, 1.0 / 240)
    held = free - _free_bytes()
    faces = 165 * 162 * 161
    print(f"[gpu]   {held / faces:.1f} bytes a face of one component", flush=True)
    assert held < 48 * faces  # 34 + 3, and what allocations round up to
    ost = o.diffusion(1.0 / 240)
    gst = g.last_diffusion_stats()
    assert all(s.iterations == 8 and not s.converged and s.abs_residual > 0 for s in gst)
    _compare(g, o, gst, ost)
    g.close()


def test_diffusion_iteration_cap(ctx):
    """A viscosity high enough that Jacobi stops at the 1000-sweep cap
    (CudaJacobiIterationSolver(1000, 5, 1e-14)) on both sides."""
    print("[gpu] diffusion at the iteration cap", flush=True)
    n = (12, 10, 8)
    g, o = _pair(ctx, n, (1.0, 1.0, 1.0), 2.0, seed=4)
    dt = 1.0 / 60
    g.run_stage(capi.STAGE_DIFFUSION, dt)
    ost = o.diffusion(dt)
    gst = g.last_diffusion_stats()
    assert all(s.iterations == 1000 and not s.converged for s in gst)
    _compare(g, o, gst, ost)
    g.close()


def test_diffusion_solver_setting(ctx):
    print("[gpu] diffusion solver setting", flush=True)
    n = (10, 10, 10)
    g, o = _pair(ctx, n, (1.0, 1.0, 1.0), 0.05, seed=9)
    g.set_diffusion_solver(capi.solver(capi.SOLVER_JACOBI, 37, 4, 1e-30))
    o.set_diffusion_solver(orc.solver(orc.JACOBI, 37, 4, 1e-30))
    dt = 1.0 / 240
    g.run_stage(capi.STAGE_DIFFUSION, dt)
    ost = o.diffusion(dt)
    gst = g.last_diffusion_stats()
    assert all(s.iterations == 37 for s in gst)
    _compare(g, o, gst, ost)
    with pytest.raises(capi.FluideError):
        g.set_diffusion_solver(capi.solver(capi.SOLVER_CG, 100, 5, 1e-10))
    g.close()


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_diffusion_with_a_face_that_is_not_finite(ctx, value):
    """A velocity outside the fluid that is not finite: no FLUID row reads it,
    but its own row's residual is not a number, so that component runs to the
    cap and does not converge, as in the oracle (where it also spreads, by
    products with 0); the others do."""
    print(f"[gpu] diffusion with a face of {value}", flush=True)
    g, o = _pair(ctx, (12, 10, 8), (1.0, 0.8, 1.1), 0.01, seed=3)
    probe, other = _pair(ctx, (12, 10, 8), (1.0, 0.8, 1.1), 0.01, seed=3)
    other.diffusion(1.0 / 240)
    air = np.argwhere(other.diffusion_markers(0) == orc.AIR)
    u = g.get(capi.GRID_U)
    u[tuple(air[len(air) // 2])] = value
    g.set(capi.GRID_U, u)
    o.set(orc.U, u.astype(np.float64))
    g.set_diffusion_solver(capi.solver(capi.SOLVER_JACOBI, 60, 5, 1e-6))
    o.set_diffusion_solver(orc.solver(orc.JACOBI, 60, 5, 1e-6))
    g.run_stage(capi.STAGE_DIFFUSION, 1.0 / 240)
    ost = o.diffusion(1.0 / 240)
    gst = g.last_diffusion_stats()
    assert [s.converged for s in gst] == [0, 1, 1] and np.isnan(gst[0].abs_residual)
    assert np.isfinite(g.get(capi.GRID_U)).sum() == u.size - 1
    for c, (gf, of) in enumerate(COMPS):
        assert gst[c].iterations == ost[c].iterations
        if c > 0:
            assert np.abs(g.get(gf) - o.get(of)).max() <= 1e-6 * np.abs(o.get(of)).max()
    g.close()
    probe.close()


def test_substep_with_viscosity_parity(ctx):
    print("[gpu] substep with viscosity", flush=True)
    n = 24
    desc = capi.scene_desc((n, n, n), method=capi.FLIP, blend=0.03, max_particles=8 * n ** 3 + 64, viscosity=0.02)
    x = capi.seed_particles(desc, [capi.box((-1, -1, -1), (0.4, 0.6, 2.0))], seed=2)
    rng = np.random.default_rng(12)
    x = np.clip(x + rng.uniform(-0.004, 0.004, x.shape).astype(np.float32), 0.0, 1.0).astype(np.float32)
    v = (rng.normal(size=x.shape) * 0.3).astype(np.float32)
    g = capi.Scene(ctx, desc)
    g.upload_particles(x, v)
    o = orc.Scene((n, n, n), method=orc.FLIP, blend=0.03, max_cfl=3.0, gravity=tuple(desc.gravity))
    o.set_viscosity(0.02)
    o.set_particles(x.astype(np.float64), v.astype(np.float64))
    dt = 1.0 / 240
    g.substep(dt, capi.solver(capi.SOLVER_JACOBI, 200, 5, 1e-14))
    o.substep(dt, orc.solver(orc.JACOBI, 200, 5, 1e-14))
    assert np.array_equal(g.get(capi.GRID_FLAGS), o.get(orc.FLAGS))
    for c in range(3):
        assert np.array_equal(g.get(DMARK[c]), o.diffusion_markers(c))
    gx, gv, _ = g.download_particles()
    ox, ov, _ = o.particles()
    scale = max(1.0, float(np.abs(ov).max()))
    assert float(np.abs(gv - ov).max()) <= 2e-4 * scale
    assert float(np.abs(gx - ox).max()) <= 2e-6 * max(1.0, float(np.abs(ox).max()))
    gst = g.last_diffusion_stats()
    assert all(s.iterations > 5 for s in gst)
    g.close()


@pytest.mark.parametrize("n,nu,cap,interval", [((12, 10, 8), 0.3, 1000, 5), ((12, 10, 8), 0.3, 1001, 4),
                                               ((33, 9, 17), 0.05, 997, 7), ((2, 2, 2), 0.1, 501, 1),
                                               ((5, 31, 3), 0.2, 6, 5), ((16, 16, 33), 0.1, 300, 0)])
def test_diffusion_repeated_states(ctx, n, nu, cap, interval):
    """An unreachable tolerance: the sweeps end in repeated states long before
    the cap, and the counts, the values (to FP32) and the last residual are
    those of the whole number of sweeps: the residual's bits are those of a
    run that checks at that one sweep only, compares no states and so makes
    them all (odd and even intervals and caps, none at all)."""
    print(f"[gpu] diffusion repeated states n={n} cap={cap} interval={interval}", flush=True)
    g, o = _pair(ctx, n, (1.0, 0.8, 1.1), nu, seed=sum(n))
    g.set_diffusion_solver(capi.solver(capi.SOLVER_JACOBI, cap, interval, 1e-30))
    o.set_diffusion_solver(orc.solver(orc.JACOBI, cap, interval if interval else cap + 1, 1e-30))
    dt = 1.0 / 120
    g.run_stage(capi.STAGE_DIFFUSION, dt)
    ost = o.diffusion(dt)
    gst = g.last_diffusion_stats()
    assert all(s.iterations == cap and not s.converged for s in gst)
    _compare(g, o, gst, ost)
    for s in gst:
        if interval and cap > interval:
            assert 0.0 <= s.abs_residual < 1e-12 if cap > 100 else s.abs_residual > 1e-12
        else:
            assert s.abs_residual == -1.0
    g.close()
    if interval and cap > interval:
        g, _ = _pair(ctx, n, (1.0, 0.8, 1.1), nu, seed=sum(n))
        g.set_diffusion_solver(capi.solver(capi.SOLVER_JACOBI, cap, (cap - 1) // interval * interval, 1e-30))
        g.run_stage(capi.STAGE_DIFFUSION, dt)
        assert [s.abs_residual for s in g.last_diffusion_stats()] == [s.abs_residual for s in gst]
        g.close()


def test_diffusion_ends_at_a_repeated_state(ctx):
    """100 000 sweeps, which alone take 250 ms of the device, end within the few
    hundred that bring the states to repeat themselves (the quickest of three
    runs)."""
    import time

    print("[gpu] diffusion ends at a repeated state", flush=True)
    g, _ = _pair(ctx, (12, 10, 8), (1.0, 0.8, 1.1), 0.05, seed=30)
    g.set_diffusion_solver(capi.solver(capi.SOLVER_JACOBI, 100000, 5, 1e-30))
    took = []
    for _ in range(3):
        t0 = time.perf_counter()
        g.run_stage(capi.STAGE_DIFFUSION, 1.0 / 120)
        took.append(time.perf_counter() - t0)
        assert all(s.iterations == 100000 and not s.converged for s in g.last_diffusion_stats())
    print(f"[gpu]   {min(took) * 1e3:.1f} ms", flush=True)
    assert min(took) < 0.1
    g.close()
