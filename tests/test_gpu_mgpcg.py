"""Multigrid-preconditioned CG (aq_flip_solve_pressure_mgpcg): against a dense FP64
solve of the legacy matrix on small random systems, as a Jacobi fixed point, and on
the 128^3 workload against plain Jacobi."""
import numpy as np
import pytest

from aquarius_amd import configs
from aquarius_amd.fluid import FlipHandle
from aquarius_amd.unet import attach_solver, solver_stats

from test_gpu_parity import log
from test_oracle_pins import AIR, FLUID, SOLID, build_dense_A

pytestmark = pytest.mark.gpu


def random_system(X, Y, Z, seed):
    rng = np.random.default_rng(seed)
    content = np.full((X + 1, Y + 1, Z + 1), SOLID, np.int32)
    inner = np.where(rng.random((X, Y, Z)) < 0.8, FLUID, AIR)
    inner[:, Y - 1, :] = AIR  # free surface: every fluid region touches air
    content[:X, :Y, :Z] = inner
    div = rng.standard_normal((X, Y, Z)).astype(np.float32)
    dens = (0.5 + rng.random((X, Y, Z))).astype(np.float32)
    cfg = configs.make_config(4, dt=0.01, pressure_iters=10, extent=(X, Y, Z))
    h = FlipHandle(cfg)
    h.set_field("content", content)
    h.set_field("divergence", div)
    h.set_field("density", dens)
    h.set_field("pressure", np.zeros((X, Y, Z), np.float32))
    A, fluid = build_dense_A(content, X, Y, Z)
    b = np.array([-float(div[c]) * float(dens[c]) for c in fluid])
    return h, A, b, fluid


@pytest.mark.parametrize("shape,seed", [((8, 6, 10), 1), ((13, 9, 7), 2), ((16, 16, 16), 3)])
def test_mgpcg_matches_dense_solve(shape, seed):
    h, A, b, fluid = random_system(*shape, seed)
    it, rel, ok = h.solve_pressure_mgpcg(1e-12, max_iters=300)
    p = h.get_field("pressure")
    got = np.array([p[c] for c in fluid], np.float64)
    want = np.linalg.solve(A, b)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    log(f"  {shape}: {it} CG iterations, FP64 residual of the FP32 result {rel:.2e}, error vs dense {err:.2e}")
    assert ok
    assert err < 2e-6  # FP32 storage of an FP64 solution
    content = h.get_field("content")[: shape[0], : shape[1], : shape[2]]
    assert np.all(p[content != FLUID] == 0)
    h.close()


def sparse_A(content, X, Y, Z):
    """The pressure matrix over the FLUID cells of the interior, assembled per direction."""
    import scipy.sparse as sp
    fl = content[:X, :Y, :Z] == FLUID
    num = np.full((X, Y, Z), -1)
    num[fl] = np.arange(fl.sum())
    diag = np.full((X, Y, Z), 6.0)
    rows, cols = [], []
    for axis, n in enumerate((X, Y, Z)):
        for end in (0, n - 1):
            diag[tuple(end if a == axis else slice(None) for a in range(3))] -= 1
        lo = tuple(slice(0, n - 1) if a == axis else slice(None) for a in range(3))
        hi = tuple(slice(1, n) if a == axis else slice(None) for a in range(3))
        both = fl[lo] & fl[hi]
        rows += [num[lo][both], num[hi][both]]
        cols += [num[hi][both], num[lo][both]]
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    return sp.csr_matrix((-np.ones(rows.size), (rows, cols)), shape=(fl.sum(),) * 2) + sp.diags(diag[fl]), fl


@pytest.mark.parametrize("shape", [(33, 40, 26), (5, 70, 3), (1, 6, 40), (81, 80, 83)])
def test_mgpcg_matches_sparse_cg(shape):
    """Extents that leave remainders of the V-cycle's tiles and of four-cell groups, levels on
    both sides of the rule that picks a level's kernels, and degenerate axes, against
    scipy's CG in FP64 on the assembled matrix; both solved far below FP32's resolution."""
    from scipy.sparse.linalg import cg
    X, Y, Z = shape
    rng = np.random.default_rng(sum(shape))
    content = np.full((X + 1, Y + 1, Z + 1), SOLID, np.int32)
    inner = np.where(rng.random(shape) < 0.8, FLUID, AIR)
    inner[:, Y - 1, :] = AIR
    content[:X, :Y, :Z] = inner
    div = rng.standard_normal(shape).astype(np.float32)
    with FlipHandle(configs.make_config(4, dt=0.01, pressure_iters=10, extent=shape)) as h:
        h.set_field("content", content)
        h.set_field("divergence", div)
        h.set_field("density", np.ones(shape, np.float32))
        A, fl = sparse_A(content, X, Y, Z)
        want, info = cg(A, -div[fl].astype(np.float64), rtol=1e-12, maxiter=20000)
        assert info == 0
        first = None
        for _ in range(3):  # the second solve on a handle captures its iterations, the third replays
            it, rel, ok = h.solve_pressure_mgpcg(1e-12, max_iters=300)
            p = h.get_field("pressure")
            assert ok
            assert np.linalg.norm(p[fl] - want) <= 2e-6 * np.linalg.norm(want)
            assert np.all(p[~fl] == 0)
            first = p if first is None else first
            assert np.array_equal(p, first)


def test_mgpcg_solution_is_a_jacobi_fixed_point_128():
    h = FlipHandle(configs.multiphase_128())
    h.steps(1)
    it, rel, ok = h.solve_pressure_mgpcg(1e-9, max_iters=200)
    p0 = h.get_field("pressure")
    log(f"  128^3: {it} CG iterations to 1e-9, FP64 residual of the FP32 field {rel:.2e}")
    assert ok and it < 200
    assert rel < 1e-5  # far below plain FP32 Jacobi's floor (~1e-4 at this size)
    h.solve_pressure(1.0, 1, 1)  # one Jacobi sweep
    p1 = h.get_field("pressure")
    assert np.linalg.norm(p1 - p0) <= 1e-5 * np.linalg.norm(p0)
    # plain Jacobi to 1e-4 agrees with it to the accuracy of that tolerance
    h.set_field("pressure", np.zeros_like(p0))
    jit, jrel, jok = h.solve_pressure(1e-4, 60000, 100)
    pj = h.get_field("pressure")
    d = np.linalg.norm(pj - p0) / np.linalg.norm(p0)
    log(f"  plain Jacobi: {jit} sweeps to {jrel:.2e}; relative difference to MG-PCG {d:.2e}")
    assert jok and d < 5e-2
    h.close()


def test_mgpcg_solver_mode_steps():
    h = FlipHandle(configs.ball_drop_64())
    attach_solver(h, "mgpcg", tol=1e-8, max_iters=200, check_every=1)
    h.steps(3)
    st = solver_stats(h)
    log(f"  mgpcg mode: {st}")
    assert st["solves"] == 3 and st["capped"] == 0
    assert st["last_residual"] < 1e-5
    h.close()


def test_solves_after_one_that_overflowed():
    """81^3 cells, four to a thread, so that the last thread owns cells past the grid's end.
    A right-hand side that overflows the FP32 preconditioner ends a solve without a result;
    the next solve on the handle equals that of a fresh handle bit for bit."""
    n = 81
    rng = np.random.default_rng(53)
    divergence = rng.standard_normal((n, n, n)).astype(np.float32)
    cfg = configs.make_config(n, dt=0.01, pressure_iters=20, pool_depth=0.5, center=(0.95, 0.95, 0.95), radius=0.15,
                              seed=53)
    out = []
    for overflow in (False, True):
        h = FlipHandle(cfg)
        zero = np.zeros((n, n, n), np.float32)
        assert h.get_field("content")[n - 1, n - 1, n - 1] == FLUID  # the last thread has work
        if overflow:
            h.set_field("divergence", np.abs(divergence) * np.float32(1e37))
            it, rel, ok = h.solve_pressure_mgpcg(1e-6, max_iters=20)
            assert not ok and it > 0
        h.set_field("divergence", divergence)
        h.set_field("pressure", zero)
        it, rel, ok = h.solve_pressure_mgpcg(1e-6, max_iters=60)
        out.append((it, rel, ok, h.get_field("pressure")))
        h.close()
    assert out[0][2]
    assert out[0][:3] == out[1][:3]
    assert np.array_equal(out[0][3].view(np.uint32), out[1][3].view(np.uint32))
