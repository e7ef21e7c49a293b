"""The tiled 2D step (k_tile2d, k_chain2d, k_relax2d, k_pre2d) against the oracle and against the phase calls.

Meshes around its tiles (4 columns wide, the last one overlapping where nx is no multiple of 4; 1 to 6 rows),
velocity grids around its 64-velocity wavefronts and 256-velocity workgroups, sizes above the rule that picks it
(cells x velocities: 100 k for FP32 KCU / UGKS, 1.5 M for FP64, 2 M and 3 M for KFVS).

Tolerances: FP64 storage 1e-10 relative (max norm) on f, w and the face fluxes after 5 steps, as in
test_gpu_parity.py's phase tests; FP32 storage 1e-5 on f and w against the phase calls (their FP32 rounding over a few
steps) and 1e-4 relative L2 against the oracle.
"""
import copy

import numpy as np
import pytest

from conftest import kb, oracle

pytestmark = pytest.mark.gpu


def rel_max(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def rel_l2(a, b):
    a, b = np.asarray(a).ravel(), np.asarray(b).ravel()
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def case(space, flux, nx, ny, nu, nv):
    mk = kb.configs.cavity_2d2f2v if space == "2d2f2v" else kb.configs.cavity_2d1f2v
    ks = kb.SolverSet(mk(nx=nx, ny=ny, nu=nu, nv=nv, knudsen=0.1, flux=flux, vMeshType="rectangle"))
    ctr, face = kb.init_fvm(ks)
    ctr.f *= 1.0 + 0.02 * np.random.default_rng(nx).random(ctr.f.shape)
    return ks, ctr, face, kb.timestep(ks, ctr)


CASES = [  # space, precision, flux, nx, ny, nu, nv
    ("2d2f2v", "fp32", "ugks", 4, 300, 9, 10),  # one tile column
    ("2d2f2v", "fp32", "ugks", 5, 90, 16, 16),  # two, overlapping by three cells
    ("2d2f2v", "fp32", "ugks", 140, 3, 17, 15),  # 255 velocities, fewer rows than a tile may have
    ("2d2f2v", "fp32", "kcu", 23, 30, 13, 20),  # 260
    ("2d2f2v", "fp32", "ugks", 31, 64, 8, 8),  # one wavefront
    ("2d2f2v", "fp32", "kfvs", 46, 47, 31, 33),  # 1023
    ("2d1f2v", "fp32", "kfvs", 41, 49, 32, 32),
    ("2d2f2v", "fp64", "ugks", 7, 240, 30, 31),
    ("2d2f2v", "fp64", "kcu", 78, 77, 13, 20),
    ("2d2f2v", "fp64", "ugks", 160, 151, 9, 7),  # 63 velocities, four rows per tile
    ("2d2f2v", "fp64", "kfvs", 110, 108, 17, 15),
    ("2d1f2v", "fp64", "kfvs", 54, 55, 32, 32),
]


@pytest.mark.parametrize("space,precision,flux,nx,ny,nu,nv", CASES)
def test_tiled_step_matches_the_oracle_and_the_phases(gpu_ctx, space, precision, flux, nx, ny, nu, nv):
    """Two calls (3 + 2 steps: walls and records made by the first step's kernel and by the relaxation) with the
    face fluxes left by the last step and its residual, against the oracle; one step against the phase calls."""
    ks, ctr, face, dt = case(space, flux, nx, ny, nu, nv)
    cg, fg, cp = copy.deepcopy(ctr), copy.deepcopy(face), copy.deepcopy(ctr)
    dev = kb.DeviceSolve(ks, cg, fg, precision, gpu_ctx)
    phases = kb.DeviceSolve(ks, cp, copy.deepcopy(face), precision, gpu_ctx)
    dev.step(dt, 1)
    phases.reconstruct()
    phases.evolve(dt)
    phases.update(dt)
    dev.download(cg)
    phases.download(cp)
    phases.close()
    tol = 1e-10 if precision == "fp64" else 1e-5
    assert rel_max(cg.f, cp.f) <= tol and rel_max(cg.w, cp.w) <= tol
    dev.step(dt, 2)
    res = np.zeros(4)
    dev.step(dt, 2, res)
    dev.download(cg, fg)
    assert dev.health() == 0
    dev.close()
    o = oracle.OracleSolve(ks, ctr, face)
    for _ in range(5):
        o.reconstruct()
        o.evolve(dt)
        ro = o.update(dt)
    if precision == "fp64":
        for a, b in ((cg.f, ctr.f), (cg.w, ctr.w), (cg.prim, ctr.prim), (fg.ff, face.ff), (fg.yff, face.yff)):
            assert rel_max(a, b) <= 1e-10
        assert rel_max(fg.fw, face.fw) <= 1e-10 and rel_max(fg.yfw, face.yfw) <= 1e-10
        assert np.allclose(res, ro[:4], rtol=1e-8)
    else:
        for a, b in ((cg.f, ctr.f), (cg.w, ctr.w), (fg.ff, face.ff), (fg.yff, face.yff)):
            assert rel_l2(a, b) <= 1e-4


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_tiled_step_does_not_depend_on_the_batch(gpu_ctx, precision):
    """Alone a solve's tiles have one row (FP32) or three (FP64), beside large ones more; its relaxation shares a
    launch with the next step's walls alone and not in the batch: the same bits either way."""
    small = case("2d2f2v", "ugks", 9, 15 if precision == "fp32" else 230, 28, 28)
    big = case("2d2f2v", "ugks", 130, 131, 16, 16)
    got = []
    for batch in (False, True):
        made = [small] + [big, big] * batch
        devs = [kb.DeviceSolve(ks, copy.deepcopy(c), copy.deepcopy(f), precision, gpu_ctx) for ks, c, f, dt in made]
        kb.batch_step(devs, [m[3] for m in made], 4, ctx=gpu_ctx)
        c, f = copy.deepcopy(small[1]), copy.deepcopy(small[2])
        devs[0].download(c, f)
        got.append((c, f))
        for d in devs:
            d.close()
    for a, b in ((got[0][0].f, got[1][0].f), (got[0][0].w, got[1][0].w), (got[0][1].ff, got[1][1].ff), (got[0][1].yfw, got[1][1].yfw)):
        np.testing.assert_array_equal(a, b)


def test_tiled_step_under_graph_replay(gpu_ctx):
    """Captured steps (every one makes its own walls and records and leaves its face fluxes) give the bits of
    eager ones, over several replays."""
    ks, ctr, face, dt = case("2d2f2v", "ugks", 30, 31, 16, 16)
    got = []
    for graphs in (False, True):
        gpu_ctx.set_graphs(graphs)
        try:
            dev = kb.DeviceSolve(ks, copy.deepcopy(ctr), copy.deepcopy(face), "fp32", gpu_ctx)
            c = copy.deepcopy(ctr)
            for _ in range(3):
                dev.step(dt, 5)
                dev.download(c)
            got.append(c)
            dev.close()
        finally:
            gpu_ctx.set_graphs(False)
    np.testing.assert_array_equal(got[0].f, got[1].f)
    np.testing.assert_array_equal(got[0].w, got[1].w)


@pytest.mark.parametrize("space,flux", [("2d2f2v", "ugks"), ("2d2f2v", "kcu"), ("2d2f2v", "kfvs"), ("2d1f2v", "kfvs")])
def test_tiled_fp32_moments_are_no_less_accurate_than_the_face_parallel_ones(gpu_ctx, space, flux):
    """One FP32 step's error in w against the oracle's step from the same stored state: the tiled kernels beside
    k_flux2d / k_cell2d, to which a normal one rounding off another sends the solve.  The tiled moments add no more
    terms in FP32 than those (8 per lane) and weight them in FP64 as they do, so the rms error over the 3660 cells
    may exceed theirs by its scatter only: 1.1 for every conserved variable."""
    mk = kb.configs.cavity_2d2f2v if space == "2d2f2v" else kb.configs.cavity_2d1f2v
    ks = kb.SolverSet(mk(nx=61, ny=60, nu=25, nv=24, knudsen=0.05, flux=flux, vMeshType="rectangle"))
    ctr, face = kb.init_fvm(ks)
    dt = kb.timestep(ks, ctr)
    dev = kb.DeviceSolve(ks, ctr, face, "fp64", gpu_ctx)
    dev.step(dt, 100)
    dev.download(ctr)
    dev.close()
    ctr.f *= 1.0 + 0.02 * np.random.default_rng(3).random(ctr.f.shape)
    err, n1 = [], ks.ps.n[0, 0, 1, 0]
    for tiled in (True, False):
        ks.ps.n[0, 0, 1, 0] = n1 if tiled else np.nextafter(n1, 0.0)
        dev = kb.DeviceSolve(ks, ctr, copy.deepcopy(face), "fp32", gpu_ctx)
        got, ref = copy.deepcopy(ctr), copy.deepcopy(ctr)
        dev.download(ref)
        dev.step(dt, 1)
        dev.download(got)
        dev.close()
        o = oracle.OracleSolve(ks, ref, copy.deepcopy(face))
        o.reconstruct()
        o.evolve(dt)
        o.update(dt)
        err.append(np.sqrt(np.mean((got.w - ref.w).reshape(-1, 4) ** 2, axis=0)))
    ks.ps.n[0, 0, 1, 0] = n1
    assert np.all(err[0] <= 1.1 * err[1]), (err[0] / err[1])


@pytest.mark.parametrize("space,precision,flux,nx,ny,nu,nv", [
    ("2d2f2v", "fp32", "ugks", 4, 660, 9, 10),  # one tile column, 90 velocities
    ("2d2f2v", "fp32", "ugks", 61, 64, 8, 8),  # one wavefront, the last column overlapping by three cells
    ("2d2f2v", "fp32", "kcu", 6, 100, 16, 16),  # two columns, overlapping by two cells
    ("2d2f2v", "fp64", "kcu", 9, 240, 28, 30),
])
def test_tiled_step_on_narrow_meshes_and_few_velocities(gpu_ctx, space, precision, flux, nx, ny, nu, nv):
    """Sizes next to the edges of the rule that picks the tiles, where their lanes or columns are few."""
    test_tiled_step_matches_the_oracle_and_the_phases(gpu_ctx, space, precision, flux, nx, ny, nu, nv)
