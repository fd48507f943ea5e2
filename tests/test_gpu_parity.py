"""GPU parity: the HIP library (through the C ABI) against the CPU oracle on the same
seeded inputs, stage by stage and over whole steps.

Bar: cell indices, sort order, content flags and every integer field bit-exact;
velocities, pressures and fractions within 1e-5 relative L2 (FP32) -- the kernels
keep the reference's operation order and no FMA contraction, so most fields are
expected to be bit-identical; the tests report how many values differ.
"""
import json
import subprocess
import sys

import numpy as np
import pytest

import aquarius_amd as aq
from aquarius_amd import configs
from aquarius_amd.fluid import FlipHandle
from oracle import binding as ob

pytestmark = pytest.mark.gpu

REL_TOL = 1e-5
INT_FIELDS = ("content", "has_velocity", "particle_count")


def log(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    nb = np.linalg.norm(b)
    d = np.linalg.norm(a - b)
    return d / nb if nb > 0 else d


def check_field(name, gpu, orc, what=""):
    g = gpu.get_field(name)
    o = orc.get_field(name)
    assert g.shape == o.shape, (name, g.shape, o.shape)
    if name in INT_FIELDS:
        bad = int((g != o).sum())
        assert bad == 0, f"{what}{name}: {bad} integer mismatches"
        return 0.0
    r = rel_l2(g, o)
    ndiff = int((g.astype(np.float64) != o).sum())
    log(f"  {what}{name}: rel_l2={r:.3e} differing={ndiff}/{g.size}")
    assert np.isfinite(g).all() == np.isfinite(o).all()
    assert r <= REL_TOL, (name, r)
    return r


def check_particles(gpu, orc, what=""):
    gp, gv, gf = gpu.get_particles()
    op, ov, of = orc.get_particles()
    for name, g, o in (("pos", gp, op), ("vel", gv, ov), ("frac", gf, of)):
        r = rel_l2(g, o)
        ndiff = int((g.astype(np.float64) != o).sum())
        log(f"  {what}particles.{name}: rel_l2={r:.3e} differing={ndiff}/{g.size}")
        assert r <= REL_TOL, (name, r)


def check_cells(gpu, orc, what=""):
    gs, ge, gh, gperm = gpu.get_cells()
    os_, oe, oh, operm = orc.get_cells()
    assert np.array_equal(gs, os_), f"{what}cellStart differs"
    assert np.array_equal(ge, oe), f"{what}cellEnd differs"
    assert np.array_equal(gh, oh), f"{what}hash differs"
    assert np.array_equal(gperm, operm), f"{what}sort permutation differs"


STAGE_FIELDS = {
    "g2p": [],
    "advect": [],
    "transfer_to_grid": ["content", "velocity", "new_velocity", "has_velocity", "density",
                         "volume_fractions", "new_volume_fractions"],
    "gravity": ["new_velocity"],
    "boundary": ["new_velocity", "content"],
    "divergence": ["divergence", "particle_count"],
    "pressure": ["pressure"],
    "project": ["new_velocity", "has_velocity"],
    "extrapolate": ["new_velocity", "has_velocity"],
    "diffusion": ["new_volume_fractions", "pressure"],
}
STEP_ORDER = ["g2p", "advect", "transfer_to_grid", "gravity", "boundary", "divergence", "pressure",
              "project", "extrapolate", "diffusion"]


def pair(cfg):
    pos, frac = ob.seed(cfg)
    gpu = FlipHandle(cfg, pos=pos, frac4=frac)
    orc = ob.Oracle(cfg, pos=pos, frac4=frac)
    return gpu, orc


def run_stagewise(cfg, steps, label):
    gpu, orc = pair(cfg)
    log(f"[{label}] init, {gpu.particle_count} particles")
    check_cells(gpu, orc, "init ")
    check_particles(gpu, orc, "init ")
    for f in STAGE_FIELDS["transfer_to_grid"] + ["content"]:
        check_field(f, gpu, orc, "init ")
    for s in range(steps):
        for st in STEP_ORDER:
            log(f"[{label}] step {s} stage {st}")
            gpu.run_stage(st)
            orc.run_stage(st)
            if st in ("g2p", "advect", "transfer_to_grid"):
                check_particles(gpu, orc, f"s{s} {st} ")
            if st == "transfer_to_grid":
                check_cells(gpu, orc, f"s{s} ")
            for f in STAGE_FIELDS[st]:
                check_field(f, gpu, orc, f"s{s} {st} ")
    gpu.close()


def test_stagewise_ball_drop_16():
    run_stagewise(configs.ball_drop_16(), steps=3, label="ball_drop_16")


def test_stagewise_ball_drop_64():
    run_stagewise(configs.ball_drop_64(), steps=1, label="ball_drop_64")


def test_stagewise_multiphase_24():
    cfg = configs.make_config(24, dt=0.01, pressure_iters=40, diffusion_iters=10, radius=0.15,
                              sphere_phase=1, phase_count=2, seed=21)
    run_stagewise(cfg, steps=2, label="multiphase_24")


@pytest.mark.parametrize("n,phases", [(1, 1), (3, 3), (40, 2), (3000, 4)])
def test_exports_with_few_particles(n, phases):
    """Every export of a handle whose particle arrays are smaller than its fields (the
    exports' scratch) and, with 3,000 particles, larger than some: against the oracle, on
    odd extents, before and after a step."""
    cfg = configs.make_config(12, dt=0.01, pressure_iters=8, diffusion_iters=4, phase_count=phases, extent=(9, 12, 7))
    rng = np.random.default_rng(n)
    h = 10 / 12
    pos = (rng.uniform(0.3, 0.7, (n, 3)) * np.array([9, 12, 7]) * h).astype(np.float32)
    vel = rng.standard_normal((n, 3)).astype(np.float32)
    frac = np.zeros((n, 4), np.float32)
    frac[np.arange(n), rng.integers(0, phases, n)] = 1
    gpu, orc = FlipHandle(cfg, pos, vel, frac), ob.Oracle(cfg, pos=pos, vel=vel, frac4=frac)
    for step in range(2):
        for name in aq.FIELDS:
            if step or name != "particle_count":  # the oracle counts inside a step
                check_field(name, gpu, orc, f"step {step} ")
        check_particles(gpu, orc)
        gpu.step()
        orc.step()
    gpu.close()


def test_handles_take_over_each_others_memory():
    """A handle's memory goes to later handles of a similar size: a scene gives the same bits
    in memory that other scenes (other sizes, phases, solver state) have left, and with
    several threads creating and destroying handles at once."""
    from concurrent.futures import ThreadPoolExecutor
    scenes = [configs.make_config(n, dt=0.01, pressure_iters=20, diffusion_iters=6, phase_count=k, sphere_phase=k - 1,
                                  extent=(n, n + 2, n - 3)) for n, k in ((24, 1), (24, 2), (23, 4), (40, 2))]

    def run(i):
        with FlipHandle(scenes[i]) as h:
            h.steps(3)
            h.solve_pressure_mgpcg(1e-6)
            h.steps(1)
            return [h.get_field(f) for f in aq.FIELDS] + list(h.get_particles())
    first = [run(i) for i in range(4)]
    with ThreadPoolExecutor(4) as pool:
        for i, got in zip([0, 1, 2, 3] * 4, pool.map(run, [0, 1, 2, 3] * 4)):
            for a, b in zip(got, first[i]):
                assert np.array_equal(a.view(np.int32), b.view(np.int32))


def test_stagewise_edge_configs():
    # non-cubic grid, full boundary coverage, warm-started pressure, 4 phases
    cfg = configs.make_config(0, dt=0.01, pressure_iters=25, diffusion_iters=5, extent=(12, 16, 20),
                              sphere_phase=3, phase_count=4, ref_boundary_coverage=0,
                              pressure_init=aq.configs.AQ_PRESSURE_PREVIOUS, seed=5)
    run_stagewise(cfg, steps=2, label="edge_12x16x20")
    cfg = configs.make_config(3, dt=0.02, pressure_iters=5, diffusion_iters=2, pool_depth=0.4,
                              radius=0.3, center=(0.5, 0.6, 0.5), seed=9)
    run_stagewise(cfg, steps=2, label="tiny_3")


def test_full_steps_match_oracle_16():
    cfg = configs.ball_drop_16()
    gpu, orc = pair(cfg)
    log("[full steps 16] 5 steps")
    gpu.steps(5)
    orc.step(5)
    check_particles(gpu, orc, "5 steps ")
    check_cells(gpu, orc, "5 steps ")
    for f in ("pressure", "new_velocity", "velocity", "content", "divergence"):
        check_field(f, gpu, orc, "5 steps ")
    assert gpu.physical_time == pytest.approx(orc.physical_time, rel=0, abs=0)
    r_g, r_o = gpu.residual(), orc.residual()
    log(f"  residual gpu={r_g:.6e} oracle={r_o:.6e}")
    assert r_g == pytest.approx(r_o, rel=1e-9)
    st = gpu.stats()
    content = orc.get_field("content")[:16, :16, :16]
    assert st["fluid_cells"] == int((content == 1).sum())
    assert st["particles"] == orc.particle_count
    _, _, frac = orc.get_particles()
    np.testing.assert_allclose(st["phase_sum"][0], frac[:, 0].sum(), rtol=1e-12)
    gpu.close()


def free_running_parity(cfg, steps, full_every, label):
    """GPU and oracle stepped side by side from the same seeded particles with no state
    copied between them: the FP64 residual of both pressure fields after every step,
    and every particle and grid field (integer fields and the sort bit-exact) every
    `full_every` steps and at the end."""
    gpu, orc = pair(cfg)
    log(f"[{label}] {gpu.particle_count} particles, {steps} free-running steps")
    worst = 0.0
    for s in range(1, steps + 1):
        gpu.step()
        orc.step()
        r_g, r_o = gpu.residual(), orc.residual()
        assert np.isfinite(r_g) and r_g == pytest.approx(r_o, rel=1e-9), (s, r_g, r_o)
        worst = max(worst, abs(r_g - r_o) / max(abs(r_o), 1e-300))
        if s % full_every == 0 or s == steps:
            log(f"[{label}] step {s}: fp64 residual gpu={r_g:.6e} oracle={r_o:.6e}")
            check_cells(gpu, orc, f"s{s} ")
            check_particles(gpu, orc, f"s{s} ")
            for f in ("content", "velocity", "new_velocity", "pressure", "divergence", "has_velocity",
                      "particle_count", "density", "new_volume_fractions"):
                check_field(f, gpu, orc, f"s{s} ")
    log(f"[{label}] largest relative difference of the per-step FP64 residuals: {worst:.3e}")
    assert gpu.physical_time == orc.physical_time
    gpu.close()


def test_ball_drop_16_all_50_steps_match_oracle():
    """The 16^3 ball drop as stated: 60 Jacobi sweeps from zero, dt 0.01, all 50 steps."""
    free_running_parity(configs.ball_drop_16(), steps=50, full_every=10, label="ball_drop_16 x50")


def test_ball_drop_64_200_steps_match_oracle_with_fp64_residual_each_step():
    """The 64^3 ball drop as stated: 100 Jacobi sweeps from zero, dt 0.005, 200 steps,
    with the FP64 divergence residual compared after every step."""
    free_running_parity(configs.ball_drop_64(), steps=200, full_every=25, label="ball_drop_64 x200")


def test_fp64_error_statement_16():
    """FP32 GPU step against the FP64 oracle run of the same step (reported)."""
    cfg = configs.ball_drop_16()
    pos, frac = ob.seed(cfg)
    gpu = FlipHandle(cfg, pos=pos, frac4=frac)
    o64 = ob.Oracle(cfg, fp64=True, pos=pos, frac4=frac)
    gpu.step()
    o64.step()
    for f in ("pressure", "new_velocity"):
        r = rel_l2(gpu.get_field(f), o64.get_field(f))
        log(f"  fp32-gpu vs fp64-oracle {f}: rel_l2={r:.3e}")
        assert r < 1e-3
    gpu.close()


STATE_FIELDS = ("content", "velocity", "new_velocity", "pressure", "divergence", "density", "particle_count",
                "has_velocity", "volume_fractions", "new_volume_fractions")


@pytest.mark.parametrize("scene,at_step", [("ball_drop_16", 25), ("ball_drop_64", 100)])
def test_fp64_error_statement_mid_run(scene, at_step):
    """The FP32 GPU step against an FP64 run of the same step at the 16^3 and 64^3 ball
    drops: the GPU's whole state after `at_step` steps goes to the FP64 oracle and both
    run one step (reported; the bound only guards against a broken comparison)."""
    cfg = configs.SCENES[scene]()
    gpu = FlipHandle(cfg)
    gpu.steps(at_step)
    pos, vel, frac = gpu.get_particles()
    o64 = ob.Oracle(cfg, fp64=True, pos=pos, vel=vel, frac4=frac, init=False)
    for f in STATE_FIELDS:
        o64.set_field(f, gpu.get_field(f))
    gpu.step()
    o64.step()
    for f in ("pressure", "new_velocity", "velocity"):
        r = rel_l2(gpu.get_field(f), o64.get_field(f))
        log(f"  [{scene} step {at_step + 1}] fp32-gpu vs fp64-oracle {f}: rel_l2={r:.3e}")
        assert r < 1e-3
    gp, gv, _ = gpu.get_particles()
    op, ov, _ = o64.get_particles()
    _, _, gh, pg = gpu.get_cells()
    _, _, oh, po = o64.get_cells()
    ig, io = np.empty_like(pg), np.empty_like(po)
    ig[pg] = np.arange(pg.size)
    io[po] = np.arange(po.size)
    rp, rv = rel_l2(gp[ig], op[io]), rel_l2(gv[ig], ov[io])
    moved = int((gh[ig] != oh[io]).sum())
    log(f"  [{scene} step {at_step + 1}] particles: position rel_l2={rp:.3e}, velocity rel_l2={rv:.3e}, "
        f"{moved} of {pg.size} in another cell")
    assert rp < 1e-5 and rv < 1e-3
    gpu.close()


def test_solve_pressure_to_tolerance_16():
    cfg = configs.ball_drop_16()
    gpu = FlipHandle(cfg)
    gpu.step()
    it, rel, ok = gpu.solve_pressure(1e-4, 20000, check_every=50)
    log(f"  solve to 1e-4: iters={it} residual={rel:.3e} ok={ok}")
    assert ok and rel <= 1e-4
    # the cap is reported as a stall
    gpu2 = FlipHandle(cfg)
    gpu2.step()
    it2, rel2, ok2 = gpu2.solve_pressure(1e-12, 30, check_every=10)
    assert not ok2 and it2 == 30
    gpu.close()
    gpu2.close()


@pytest.mark.parametrize("n,every,tol,limit", [(16, 7, 1e-3, 4000), (33, 20, 1e-3, 4000), (33, 1, 3e-2, 4000),
                                               (40, 50, 1e-5, 333)])
def test_solves_that_run_ahead(monkeypatch, n, every, tol, limit):
    """Chunks of sweeps queued before the last residual is known, and undone where it ends
    the solve: the same sweeps, residual and bits as waiting for each one (no graphs),
    in a second solve and the step after it as well."""
    cfg = configs.make_config(n, dt=0.01, pressure_iters=20, pool_depth=0.4, seed=43)
    out = []
    for no_graph in ("1", "0"):
        monkeypatch.setenv("AQFLIP_NO_GRAPH", no_graph)
        h = FlipHandle(cfg)
        h.steps(2)
        got = []
        for t in (tol, tol / 3):
            sweeps, res, _ = h.solve_pressure(t, limit, every)
            got += [sweeps, res, h.get_field("pressure")]
        h.steps(1)
        out.append(got + [h.get_field("pressure"), h.residual()])
        h.close()
    assert out[0][0] > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_cpp_driver_runs():
    from aquarius_amd.build import DRIVER
    out = subprocess.run([str(DRIVER), "--n", "16", "--steps", "5"], capture_output=True, text=True,
                         timeout=120)
    assert out.returncode == 0, out.stderr
    rec = json.loads(out.stdout.strip().splitlines()[-1])
    log("  driver:", rec)
    assert rec["steps"] == 5 and rec["particles"] > 9000
    assert rec["physical_time"] == pytest.approx(0.05, rel=1e-5)
    assert rec["center"] == [5, 5, 5] and rec["container"] == 10


def test_python_fluid_surface():
    f = aq.Fluid()
    f.init(configs.ball_drop_16())
    for _ in range(3):
        f.simulationStep()
    assert f.physicalTime == pytest.approx(0.03, rel=1e-5)
    assert f.getCenter() == (5.0, 5.0, 5.0) and f.getContainerSize() == 10.0
    f.draw()


@pytest.mark.parametrize("pressure_iters,diffusion_iters", [(40, 10), (12, 30)])
def test_full_steps_match_oracle_multiphase_24(pressure_iters, diffusion_iters):
    """Whole steps of a two-phase scene through the captured step graph, whose
    diffusion sweeps share launches with the pressure sweeps (the longer chain
    finishing on its own: pressure in the first case, diffusion in the second)."""
    cfg = configs.make_config(24, dt=0.01, pressure_iters=pressure_iters, diffusion_iters=diffusion_iters,
                              radius=0.15, sphere_phase=1, phase_count=2, seed=21)
    gpu, orc = pair(cfg)
    log(f"[full steps multiphase 24 J{pressure_iters} D{diffusion_iters}] 4 steps")
    gpu.steps(4)
    orc.step(4)
    check_particles(gpu, orc, "4 steps ")
    check_cells(gpu, orc, "4 steps ")
    for f in ("pressure", "new_velocity", "new_volume_fractions", "volume_fractions", "density"):
        check_field(f, gpu, orc, "4 steps ")
    gpu.close()


@pytest.mark.parametrize("pressure_iters,diffusion_iters", [(40, 10), (12, 30)])
def test_full_steps_match_oracle_mixing_24(pressure_iters, diffusion_iters):
    """A two-phase ball resting in the pool: the phases mix from the first step, so
    every paired diffusion sweep changes the fractions and none is skipped."""
    cfg = configs.make_config(24, dt=0.01, pressure_iters=pressure_iters, diffusion_iters=diffusion_iters,
                              radius=0.15, center=(0.5, 0.2, 0.5), sphere_phase=1, phase_count=2,
                              diffusion_coeff=0.05, seed=23)
    gpu, orc = pair(cfg)
    log(f"[mixing 24 J{pressure_iters} D{diffusion_iters}] 4 steps")
    gpu.steps(4)
    orc.step(4)
    check_particles(gpu, orc, "4 steps ")
    check_cells(gpu, orc, "4 steps ")
    for f in ("pressure", "new_velocity", "new_volume_fractions", "volume_fractions", "density"):
        check_field(f, gpu, orc, "4 steps ")
    frac = gpu.get_field("new_volume_fractions")[:24, :24, :24]
    mixed = ((frac[..., 0] > 0) & (frac[..., 1] > 0)).sum()
    assert mixed > 0, "the scene must mix phases"
    gpu.close()


@pytest.mark.parametrize("extent,phases,pressure_iters,diffusion_iters,keep,depth,sparse", [
    ((5, 3, 4), 1, 16, 0, False, 0.5, False),     # fewer cells than a wave
    ((16, 16, 16), 4, 16, 40, False, 0.25, False),  # diffusion goes on alone
    ((20, 18, 27), 3, 41, 16, True, 0.1, False),  # pressure goes on alone, from the last step's
    ((20, 20, 20), 1, 30, 0, False, 1.0, True),   # five to eight cells per thread
    ((26, 26, 26), 2, 20, 17, True, 1.0, True),   # more, in both chains
    ((27, 27, 27), 1, 17, 0, True, 1.0, True),    # nearly the most cells
    ((27, 27, 28), 1, 17, 0, True, 0.1, False),   # one launch per sweep: too many cells
])
def test_sweeps_of_small_grids(extent, phases, pressure_iters, diffusion_iters, keep, depth, sparse):
    """All sweeps of a step in one launch (grids that fit in LDS), over the numbers of
    cells per thread, phases and chain lengths. sparse: one particle in every cell, so
    that all are FLUID."""
    cfg = configs.make_config(0, dt=0.01, extent=extent, pressure_iters=pressure_iters,
                              diffusion_iters=diffusion_iters, pool_depth=depth, radius=0.2,
                              center=(0.5, 0.5, 0.5), sphere_phase=phases - 1, phase_count=phases,
                              diffusion_coeff=0.05, seed=31,
                              pressure_init=configs.AQ_PRESSURE_PREVIOUS if keep else configs.AQ_PRESSURE_ZERO)
    pos, frac = ob.seed(cfg)
    if sparse:
        cell = (pos / np.float32(cfg.grid_physical_size / extent[0])).astype(np.int64)
        _, one = np.unique((cell[:, 0] * extent[1] + cell[:, 1]) * extent[2] + cell[:, 2], return_index=True)
        pos, frac = pos[one], frac[one]
    gpu = FlipHandle(cfg, pos=pos, frac4=frac)
    orc = ob.Oracle(cfg, pos=pos, frac4=frac)
    log(f"[small {extent} K{phases} J{pressure_iters} D{diffusion_iters}] {len(pos)} particles")
    gpu.steps(3)
    orc.step(3)
    check_particles(gpu, orc)
    for f in ("content", "pressure", "new_velocity", "new_volume_fractions", "volume_fractions", "density"):
        check_field(f, gpu, orc)
    gpu.close()


@pytest.mark.parametrize("extent,sweeps,keep,depth", [
    ((5, 3, 4), 9, True, 0.5),          # less than a tile; two tile launches and a single
    ((8, 16, 24), 4, False, 0.5),       # whole tiles, one launch
    ((33, 17, 26), 11, True, 0.25),     # ragged in every axis
    ((25, 40, 39), 8, False, 0.9),
    ((16, 16, 16), 21, True, 0.25),     # all sweeps in one launch
    ((104, 100, 101), 11, True, 0.25),  # long tiles, rows that end inside a thread's cells
    ((104, 101, 100), 14, False, 0.9),  # and that do not
])
def test_sweeps_per_launch_keep_the_bits(extent, sweeps, keep, depth):
    """Several pressure sweeps to a launch against one (the path of a field whose content
    was uploaded), from arbitrary values: zeros of both signs, subnormal and very large
    ones, and AIR cells that hold something."""
    cfg = configs.make_config(0, dt=0.01, extent=extent, pressure_iters=sweeps, pool_depth=depth, radius=0.2,
                              center=(0.5, 0.6, 0.5), seed=37,
                              pressure_init=configs.AQ_PRESSURE_PREVIOUS if keep else configs.AQ_PRESSURE_ZERO)
    rng = np.random.default_rng(5)
    out = []
    fields = None
    for uploaded in (False, True):
        h = FlipHandle(cfg)
        if fields is None:
            shape = h.get_field("pressure").shape

            def values():
                v = rng.standard_normal(shape) * 10.0 ** rng.integers(-3, 4, shape)
                v = np.where(rng.random(shape) < 0.1, rng.choice([0.0, -0.0, 1e-44, -3e-42, 1e-38, 1e30], shape), v)
                return v.astype(np.float32)

            fields = {"divergence": values(), "pressure": values(), "content": h.get_field("content")}
        if uploaded:
            h.set_field("content", fields["content"])
        for f in ("divergence", "pressure"):
            h.set_field(f, fields[f])
        for _ in range(2):  # the second solve starts in the other buffer and with clean AIR cells
            h.run_stage("pressure")
            out.append(h.get_field("pressure").view(np.uint32))
        h.close()
    assert np.isfinite(out[1].view(np.float32)).all()
    assert np.array_equal(out[0], out[2]) and np.array_equal(out[1], out[3])


@pytest.mark.parametrize("extent,phases,pressure_iters,diffusion_iters", [
    ((9, 10, 13), 3, 10, 11),   # two launches of four pairs, a diffusion sweep after them
    ((33, 17, 26), 2, 15, 12),
    ((16, 24, 20), 4, 14, 40),
    ((97, 66, 65), 4, 11, 10),  # a pair per launch: too many cells for four phases
])
def test_paired_launches_of_several_sweeps(monkeypatch, extent, phases, pressure_iters, diffusion_iters):
    """Several pressure and diffusion sweeps to a launch give the bits of the sequential
    order, and count every pair when none is skipped. The ball rests in the pool, so that
    the phases mix."""
    cfg = configs.make_config(0, dt=0.01, extent=extent, pressure_iters=pressure_iters,
                              diffusion_iters=diffusion_iters, radius=0.2, center=(0.5, 0.2, 0.5),
                              sphere_phase=phases - 1, phase_count=phases, diffusion_coeff=0.05, seed=41)
    pos, frac = ob.seed(cfg)
    out, computed = [], []
    for env in ({"AQFLIP_NO_FUSE": "1", "AQFLIP_NO_OVERLAP": "1"}, {}, {"AQFLIP_NO_FIXED_POINT_SKIP": "1"}):
        with monkeypatch.context() as m:
            for k, v in env.items():
                m.setenv(k, v)
            h = FlipHandle(cfg, pos=pos, frac4=frac)
        h.steps(3)
        out.append([h.get_field(f).view(np.uint32) for f in ("pressure", "new_volume_fractions")])
        computed.append(h.paired_diffusion_computed())
        h.close()
    for k in (1, 2):
        for a, b in zip(out[0], out[k]):
            assert np.array_equal(a, b)
    paired = 3 * min(pressure_iters, diffusion_iters)
    assert computed[2] == paired and computed[1] <= paired


@pytest.mark.parametrize("scene", ["separated", "mixing"])
def test_fixed_point_skip_equals_full_compute_64(monkeypatch, scene):
    """Paired diffusion sweeps after a sweep that changed nothing skip their work; the
    steps give the same bits as computing every sweep."""
    center = (0.5, 0.7, 0.5) if scene == "separated" else (0.5, 0.2, 0.5)
    cfg = configs.make_config(64, dt=0.005, pressure_iters=60, diffusion_iters=40, radius=0.15,
                              center=center, sphere_phase=1, phase_count=2, seed=29)
    pos, frac = ob.seed(cfg)
    out, computed = {}, {}
    for flag in ("1", "0"):
        monkeypatch.setenv("AQFLIP_NO_FIXED_POINT_SKIP", flag)
        h = FlipHandle(cfg, pos=pos, frac4=frac)
        log(f"[64 {scene} no_skip={flag}] 3 steps")
        h.steps(3)
        out[flag] = {f: h.get_field(f) for f in ("pressure", "new_velocity", "new_volume_fractions")}
        out[flag]["pos"] = h.get_particles()[0]
        computed[flag] = h.paired_diffusion_computed()
        h.close()
    for k in out["0"]:
        assert np.array_equal(out["0"][k].view(np.uint32), out["1"][k].view(np.uint32)), k
    paired = 3 * min(cfg.pressure_iters, cfg.diffusion_iters)
    assert computed["1"] == paired  # skipping off: every paired sweep computed
    if scene == "separated":  # one-hot phases apart: only each step's first sweep computes
        assert computed["0"] == 3
    else:
        assert 3 <= computed["0"] <= paired


def test_listed_sweeps_on_eight_workgroups_64(monkeypatch):
    """Listed sweeps read each workgroup's first two chunks from a table and the rest
    from the chunk list. With 8 workgroups (AQFLIP_LISTED_GRID=8) each walks about 25
    chunks, nearly all from the list; the steps give the same bits as the default grids
    (at most two chunks per workgroup here)."""
    cfg = configs.make_config(64, dt=0.005, pressure_iters=60, diffusion_iters=40, radius=0.15,
                              center=(0.5, 0.2, 0.5), sphere_phase=1, phase_count=2, seed=29)
    pos, frac = ob.seed(cfg)
    out = {}
    for grid in ("0", "8"):
        monkeypatch.setenv("AQFLIP_LISTED_GRID", grid)
        h = FlipHandle(cfg, pos=pos, frac4=frac)
        log(f"[64 listed grid {grid}] 3 steps")
        h.steps(3)
        out[grid] = {f: h.get_field(f) for f in ("pressure", "new_velocity", "new_volume_fractions")}
        out[grid]["pos"] = h.get_particles()[0]
        active = int((h.get_field("content") == 1).sum())
        h.close()
    assert active > 8 * 512 * 2  # more FLUID cells than 8 workgroups' table entries cover
    for k in out["0"]:
        assert np.array_equal(out["0"][k].view(np.uint32), out["8"][k].view(np.uint32)), k


def test_concurrent_diffusion_equals_sequential_128(monkeypatch):
    """Fused pressure + diffusion launches, diffusion on a second stream, and the
    reference's sequential order give the same bits at 128^3."""
    cfg = configs.multiphase_128()
    pos, frac = ob.seed(cfg)
    out = {}
    for mode, (no_fuse, no_overlap) in {"fused": ("0", "0"), "overlap": ("1", "0"),
                                        "sequential": ("1", "1")}.items():
        monkeypatch.setenv("AQFLIP_NO_FUSE", no_fuse)
        monkeypatch.setenv("AQFLIP_NO_OVERLAP", no_overlap)
        h = FlipHandle(cfg, pos=pos, frac4=frac)
        log(f"[128 {mode}] 3 steps")
        h.steps(3)
        out[mode] = {f: h.get_field(f) for f in ("pressure", "new_velocity", "new_volume_fractions")}
        out[mode]["pos"] = h.get_particles()[0]
        h.close()
    for mode in ("fused", "overlap"):
        for k in out[mode]:
            assert np.array_equal(out[mode][k].view(np.uint32), out["sequential"][k].view(np.uint32)), (mode, k)


def test_stage_timing_counts_and_matches_graph(monkeypatch):
    """The profiled (eager, event-timed) step runs the same paired sweeps as the
    captured step, reports one pass per sweep, and gives the same bits."""
    cfg = configs.make_config(24, dt=0.01, pressure_iters=40, diffusion_iters=10, radius=0.15,
                              sphere_phase=1, phase_count=2, seed=21)
    pos, frac = ob.seed(cfg)
    out = {}
    for mode in ("graph", "timed"):
        h = FlipHandle(cfg, pos=pos, frac4=frac)
        log(f"[timing {mode}] 2 steps")
        if mode == "timed":
            h.set_timing(True)
        h.steps(2)
        if mode == "timed":
            t = h.timing()
            assert t["pressure_diffusion"][1] == 2 * 10
            assert t["pressure"][1] == 2 * 30
            assert t["diffusion"][1] == 0
            assert t["extrapolate"][1] == 2 * 3
            assert t["g2p"][1] == 2 and t["transfer_to_grid"][1] == 2 and t["p2g"][1] == 2
            assert all(ms >= 0 for ms, _ in t.values())
        out[mode] = {f: h.get_field(f) for f in ("pressure", "new_velocity", "new_volume_fractions")}
        out[mode]["pos"] = h.get_particles()[0]
        h.close()
    for k in out["graph"]:
        assert np.array_equal(out["graph"][k].view(np.uint32), out["timed"][k].view(np.uint32)), k
    monkeypatch.setenv("AQFLIP_NO_FUSE", "1")
    h = FlipHandle(cfg, pos=pos, frac4=frac)
    h.set_timing(True)
    h.steps(1)
    t = h.timing()
    h.close()
    assert t["pressure_diffusion"][1] == 0 and t["pressure"][1] == 40 and t["diffusion"][1] == 10


def test_full_steps_match_oracle_non_cubic_64_rows():
    """Whole steps on a 20 x 24 x 64 grid (X != Y, and z rows of 65 faces, so a wave of
    the last two extrapolation passes spans at most two face rows and tests them both
    with scalar loads) against the oracle: the near-row passes, their row stamps and the
    interleaved velocity copy the next step's G2P reads."""
    cfg = configs.make_config(0, dt=0.01, pressure_iters=30, diffusion_iters=5, extent=(20, 24, 64),
                              sphere_phase=1, phase_count=2, radius=0.25, center=(0.45, 0.65, 0.55), seed=11)
    gpu, orc = pair(cfg)
    log("[full steps 20x24x64] 6 steps")
    gpu.steps(6)
    orc.step(6)
    check_particles(gpu, orc, "6 steps ")
    check_cells(gpu, orc, "6 steps ")
    for f in ("pressure", "new_velocity", "velocity", "has_velocity", "content", "volume_fractions"):
        check_field(f, gpu, orc, "6 steps ")
    gpu.close()


def test_steps_after_a_field_upload_match_an_uninterrupted_run():
    """Uploading a velocity field (here unchanged) marks the interleaved (newVelocity,
    velocity) copy stale; the next step rebuilds it in full and must continue exactly as
    a run without the upload."""
    cfg = configs.ball_drop_64()
    a, b = FlipHandle(cfg), FlipHandle(cfg)
    a.steps(8)
    b.steps(7)
    b.set_field("new_velocity", b.get_field("new_velocity"))
    b.set_field("velocity", b.get_field("velocity"))
    b.steps(1)
    for f in ("pressure", "new_velocity", "velocity", "has_velocity", "content"):
        np.testing.assert_array_equal(a.get_field(f), b.get_field(f), err_msg=f)
    for x, y in zip(a.get_particles(), b.get_particles()):
        np.testing.assert_array_equal(x, y)
    a.close()
    b.close()


def test_an_export_leaves_fractions_the_handle_does_not_carry_at_zero():
    """Two phases: an export, a step, and a field upload that raises the phases to four.
    The particles have never held fractions 2 and 3, so both are 0 (also in the sums)."""
    cfg = configs.make_config(16, dt=0.01, pressure_iters=20, diffusion_iters=5, sphere_phase=1, phase_count=2, seed=47)
    h = FlipHandle(cfg)
    h.get_particles()
    h.steps(1)
    f = h.get_field("volume_fractions")
    f[0, 0, 0, 3] = 0.5
    h.set_field("volume_fractions", f)
    frac = h.get_particles()[2]
    assert frac[:, :2].sum() > 0 and not frac[:, 2:].any()
    sums = h.stats()["phase_sum"]
    assert sums[0] > 0 and sums[2:] == [0.0, 0.0]
    h.close()


@pytest.mark.parametrize("pressure_iters,diffusion_iters", [(40, 20), (20, 40), (18, 21), (24, 24)])
def test_timed_small_steps_keep_the_bits(pressure_iters, diffusion_iters):
    """Both chains of sweeps in one launch, and with stage timing on, where the longer
    chain's rest has launches of its own. The ball rests in the pool, so the phases mix."""
    cfg = configs.make_config(14, dt=0.01, pressure_iters=pressure_iters, diffusion_iters=diffusion_iters, radius=0.2,
                              center=(0.5, 0.2, 0.5), sphere_phase=1, phase_count=2, diffusion_coeff=0.05, seed=59)
    out = []
    for timed in (False, True):
        h = FlipHandle(cfg)
        h.set_timing(timed)
        h.steps(3)
        out.append([h.get_field(f).view(np.uint32) for f in ("pressure", "new_velocity", "new_volume_fractions")])
        out[-1].append(h.paired_diffusion_computed())
        h.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_fields_larger_than_the_export_scratch():
    """130^3 cells and 64 particles: velocities (36 MB) and their flags (35 MB) leave in two
    pieces of at most 32 MiB. What was uploaded comes back."""
    n = 130
    cfg = configs.make_config(n, dt=0.01, pressure_iters=4)
    rng = np.random.default_rng(61)
    h = FlipHandle(cfg, pos=(rng.uniform(0.3, 0.7, (64, 3)) * 10).astype(np.float32))
    vel = rng.standard_normal((n + 1, n + 1, n + 1, 4)).astype(np.float32)
    vel[..., 3] = 0
    flags = rng.integers(0, 2, (n, n, n, 4)).astype(np.int32)
    flags[..., 3] = 0
    h.set_field("velocity", vel)
    h.set_field("has_velocity", flags)
    assert np.array_equal(h.get_field("velocity").view(np.uint32), vel.view(np.uint32))
    assert np.array_equal(h.get_field("has_velocity"), flags)
    h.close()


@pytest.mark.parametrize("extent,phases", [((33, 33, 33), 1), ((40, 40, 25), 3), ((40, 40, 26), 3), ((34, 33, 33), 1)])
def test_exports_on_both_sides_of_the_small_sizes(extent, phases):
    """Every export where a field or the particles are small enough to be rearranged on the
    host (up to 40,000 elements and 4,096 particles), and just above: against the oracle."""
    n = 4096 if extent[2] == 33 else 4097
    cfg = configs.make_config(0, dt=0.01, pressure_iters=8, diffusion_iters=4, phase_count=phases, extent=extent)
    rng = np.random.default_rng(n)
    pos = (rng.uniform(0.2, 0.8, (n, 3)) * np.array(extent) * (10 / extent[1])).astype(np.float32)
    vel = rng.standard_normal((n, 3)).astype(np.float32)
    frac = np.zeros((n, 4), np.float32)
    frac[np.arange(n), rng.integers(0, phases, n)] = 1
    gpu, orc = FlipHandle(cfg, pos, vel, frac), ob.Oracle(cfg, pos=pos, vel=vel, frac4=frac)
    gpu.step()
    orc.step()
    for name in aq.FIELDS:
        check_field(name, gpu, orc)
    check_particles(gpu, orc)
    gpu.close()


@pytest.mark.parametrize("coefficient", [0.05, 1e-5])
@pytest.mark.parametrize("extent,rest", [((33, 17, 26), 1), ((33, 17, 26), 4), ((33, 17, 26), 9), ((64, 24, 40), 22)])
def test_diffusion_sweeps_after_the_paired_ones(monkeypatch, extent, rest, coefficient):
    """Diffusion sweeps beyond the pressure's, every fourth of which records whether it
    changed anything so that later ones can be skipped, give the bits of the sequential
    order: phases that mix, and ones that have settled after a few sweeps."""
    cfg = configs.make_config(0, dt=0.01, extent=extent, pressure_iters=6, diffusion_iters=6 + rest, radius=0.2,
                              center=(0.5, 0.2, 0.5), sphere_phase=1, phase_count=2, diffusion_coeff=coefficient,
                              seed=67)
    pos, frac = ob.seed(cfg)
    out = []
    for flag in ("1", "0"):
        monkeypatch.setenv("AQFLIP_NO_FUSE", flag)
        monkeypatch.setenv("AQFLIP_NO_OVERLAP", flag)
        h = FlipHandle(cfg, pos=pos, frac4=frac)
        h.steps(4)
        out.append([h.get_field(f).view(np.uint32) for f in ("pressure", "new_volume_fractions")])
        h.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
