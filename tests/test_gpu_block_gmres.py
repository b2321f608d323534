"""Shared-basis block GMRES on the device (sbh_block_gmres) against the
oracle's restatement of block_gmres_inner (block_gmres.rs:666-1120) and LAPACK.

The device and the oracle run the same recurrence (block Arnoldi on one
basis, block CGS with the DGKS trigger, per-column CGS2 QR with rank-drop
deflation, Givens least squares after each block step) with different
summation orders, so they take the same number of block steps and their
solutions agree far below the 1e-8 tolerance.  Cases: the 1280-panel sphere
with 12 and 64 plane waves, restarts, the Jacobi preconditioner, an initial
guess, duplicated and zero right-hand sides (deflation), exact-residual
checkpoints, one right-hand side (scalar GMRES), device-resident blocks, and
the checked boundary's rejections.
"""

import numpy as np
import pytest

import oracle
from oracle import mie
import sonium_amd as sa
from sonium_amd.mesh import fibonacci_directions, icosphere

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sphere1280(ctx):
    m = icosphere(1.0, 3)
    k = 2.0
    tm = sa.TbemMesh(ctx, m)
    ph = sa.PhysicsParams.from_wavenumber(k)
    beta = ph.burton_miller_beta()
    system = sa.build_tbem_system_with_beta(ctx, tm, ph, beta)
    A = system.matrix
    c, nn, area = m.element_geometry()
    dirs = fibonacci_directions(64)
    B = np.stack([oracle.plane_wave_rhs(c, nn, k, beta, direction=d) for d in dirs], 1)
    yield {"mesh": m, "tm": tm, "sys": system, "A": A, "B": B, "dirs": dirs, "k": k, "area": area, "c": c}
    system.close()
    tm.close()


def _compare(A, B, sol, ref, st, label, steps_slack=1):
    X = sol.x
    Xl = np.linalg.solve(A, B)
    err_o = np.linalg.norm(X - ref, axis=0) / np.linalg.norm(ref, axis=0)
    err_l = np.linalg.norm(X - Xl, axis=0) / np.linalg.norm(Xl, axis=0)
    res = np.linalg.norm(B - A @ X, axis=0) / np.linalg.norm(B, axis=0)
    print(f"{label}: {sol.iterations} block steps (oracle {st['iterations']}), basis {sol.max_basis}, "
          f"max true residual {res.max():.2e} (reported {sol.true_residuals.max():.2e}), "
          f"vs oracle {err_o.max():.2e}, vs LAPACK {err_l.max():.2e}")
    assert abs(sol.iterations - st["iterations"]) <= steps_slack
    assert sol.converged == st["converged"]
    np.testing.assert_allclose(sol.true_residuals, res, rtol=1e-6, atol=1e-14)
    np.testing.assert_allclose(sol.true_residuals, st["true_residuals"], rtol=0.5, atol=2e-10)
    return err_o, err_l, res


@pytest.mark.parametrize("s", [12, 64])
def test_block_gmres_matches_oracle_and_lapack(sphere1280, ctx, s):
    A, B = sphere1280["A"], sphere1280["B"][:, :s]
    op = sa.DenseMatrixOperator(sphere1280["sys"])
    cfg = sa.BlockGmresConfig(max_iterations=100, restart=50, tolerance=1e-8)
    sol = sa.block_gmres(op, B, cfg)
    ref, st = oracle.block_gmres(A, B, restart=50, max_iterations=100, tol=1e-8)
    err_o, err_l, res = _compare(A, B, sol, ref, st, f"{s} plane waves")
    assert sol.converged and res.max() <= 1e-8
    assert err_o.max() <= 1e-7 and err_l.max() <= 1e-7
    # the shared basis: fewer block steps than the single-RHS solve needs
    x1, st1 = oracle.gmres(A, B[:, 0], restart=50, max_iterations=100, tol=1e-8)
    assert sol.iterations < st1["iterations"]
    # surface pressure against the Mie series per direction
    m = sphere1280
    for col in (0, s - 1):
        p = mie.surface_pressure(m["k"], 1.0, m["c"], direction=m["dirs"][col])
        assert mie.weighted_relative_l2(sol.x[:, col], p, m["area"]) < 0.02
    op.close()


def test_block_gmres_restarts_jacobi_and_guess(sphere1280):
    A, B = sphere1280["A"], sphere1280["B"][:, :12]
    op = sa.DenseMatrixOperator(sphere1280["sys"])
    # restart 3: several cycles
    cfg = sa.BlockGmresConfig(max_iterations=100, restart=3, tolerance=1e-8)
    sol = sa.block_gmres(op, B, cfg)
    ref, st = oracle.block_gmres(A, B, restart=3, max_iterations=100, tol=1e-8)
    _, err_l, res = _compare(A, B, sol, ref, st, "restart 3")
    assert sol.restart_cycles > 1 and res.max() <= 1e-8 and err_l.max() <= 1e-7
    # Jacobi
    pc = sa.JacobiPreconditioner(op)
    cfg = sa.BlockGmresConfig(max_iterations=100, restart=30, tolerance=1e-8)
    sol = sa.block_gmres_preconditioned_with_guess(op, B, pc, None, cfg)
    ref, st = oracle.block_gmres(A, B, restart=30, max_iterations=100, tol=1e-8, jacobi=True)
    _, err_l, res = _compare(A, B, sol, ref, st, "Jacobi")
    assert res.max() <= 1e-8 and err_l.max() <= 1e-7
    # initial guess: the LAPACK solution perturbed
    Xl = np.linalg.solve(A, B)
    rng = np.random.default_rng(3)
    X0 = Xl + 1e-3 * (rng.standard_normal(Xl.shape) + 1j * rng.standard_normal(Xl.shape))
    sol = sa.block_gmres_preconditioned_with_guess(op, B, None, X0, cfg)
    ref, st = oracle.block_gmres(A, B, X0=X0, restart=30, max_iterations=100, tol=1e-8)
    _, err_l, res = _compare(A, B, sol, ref, st, "initial guess")
    assert res.max() <= 1e-8
    # exact guess: converged at the first residual, no block step
    sol = sa.block_gmres_preconditioned_with_guess(op, B, None, Xl, cfg)
    assert sol.converged and sol.iterations == 0
    op.close()


def test_block_gmres_deflation_and_zero_columns(sphere1280):
    A = sphere1280["A"]
    B0 = sphere1280["B"][:, :4]
    # duplicated, scaled and zero columns (block_gmres.rs:1383-1500 cases)
    B = np.concatenate([B0, B0[:, :2], 3.0 * B0[:, 1:2], np.zeros((A.shape[0], 1))], axis=1)
    op = sa.DenseMatrixOperator(sphere1280["sys"])
    cfg = sa.BlockGmresConfig(max_iterations=50, restart=30, tolerance=1e-8)
    sol = sa.block_gmres(op, B, cfg)
    ref, st = oracle.block_gmres(A, B, restart=30, max_iterations=50, tol=1e-8)
    live = slice(0, B.shape[1] - 1)
    X = sol.x
    res = np.linalg.norm(B[:, live] - A @ X[:, live], axis=0) / np.linalg.norm(B[:, live], axis=0)
    err_o = np.linalg.norm(X[:, live] - ref[:, live], axis=0) / np.linalg.norm(ref[:, live], axis=0)
    print(f"deflation: {sol.iterations} block steps (oracle {st['iterations']}), {sol.deflated} directions "
          f"dropped, max true residual {res.max():.2e}, vs oracle {err_o.max():.2e}")
    assert abs(sol.iterations - st["iterations"]) <= 1 and sol.converged == st["converged"]
    assert err_o.max() <= 1e-7
    # the initial block QR drops both duplicates, the multiple and the zero column
    assert sol.deflated >= 4
    assert np.all(sol.x[:, -1] == 0) and sol.true_residuals[-1] == 0.0
    np.testing.assert_allclose(sol.x[:, 4:6], sol.x[:, :2], rtol=0, atol=1e-9 * np.abs(sol.x).max())
    np.testing.assert_allclose(sol.x[:, 6], 3.0 * sol.x[:, 1], rtol=0, atol=1e-8 * np.abs(sol.x).max())
    assert res.max() <= 1e-8
    op.close()


def test_block_gmres_checkpoints_single_rhs_and_device(sphere1280, ctx):
    A, B = sphere1280["A"], sphere1280["B"][:, :8]
    op = sa.DenseMatrixOperator(sphere1280["sys"])
    cfg = sa.BlockGmresConfig(max_iterations=100, restart=40, tolerance=1e-8, exact_residual_check_interval=3)
    sol = sa.block_gmres(op, B, cfg)
    ref, st = oracle.block_gmres(A, B, restart=40, max_iterations=100, tol=1e-8, exact_residual_check_interval=3)
    _compare(A, B, sol, ref, st, "exact checkpoints every 3 steps")
    assert sol.exact_residual_checks >= sol.iterations // 3
    # one right-hand side: the block recurrence is scalar GMRES
    b = B[:, :1]
    sol1 = sa.block_gmres(op, b, sa.BlockGmresConfig(max_iterations=100, restart=50, tolerance=1e-8))
    x_s, st_s = oracle.gmres(A, b[:, 0], restart=50, max_iterations=100, tol=1e-8)
    print(f"one right-hand side: {sol1.iterations} block steps, scalar GMRES {st_s['iterations']}")
    assert abs(sol1.iterations - st_s["iterations"]) <= 1
    assert np.linalg.norm(sol1.x[:, 0] - x_s) / np.linalg.norm(x_s) <= 1e-7
    # device-resident blocks give the host-path solution
    n, s = B.shape
    dB = sa.DeviceVector(ctx, n * s)
    dB.upload(B)
    dX = sa.DeviceVector(ctx, n * s)
    cfg = sa.BlockGmresConfig(max_iterations=100, restart=50, tolerance=1e-8)
    sd = sa.block_gmres_device(op, dB, s, dX, cfg)
    sh = sa.block_gmres(op, B, cfg)
    Xd = dX.download().reshape(n, s)
    assert sd.iterations == sh.iterations and np.array_equal(Xd, sh.x)
    dB.close()
    dX.close()
    op.close()


def test_block_gmres_checked_boundary(sphere1280):
    A, B = sphere1280["A"], sphere1280["B"][:, :2].copy()
    op = sa.DenseMatrixOperator(sphere1280["sys"])
    for bad in (sa.BlockGmresConfig(max_iterations=0), sa.BlockGmresConfig(restart=0),
                sa.BlockGmresConfig(tolerance=0.0), sa.BlockGmresConfig(tolerance=float("nan"))):
        with pytest.raises(sa.SbhError) as e:
            sa.block_gmres(op, B, bad)
        assert e.value.status == 1
    Bn = B.copy()
    Bn[3, 1] = np.nan
    with pytest.raises(sa.SbhError) as e:
        sa.block_gmres(op, Bn)
    assert "right-hand side" in str(e.value)
    X0 = np.zeros_like(B)
    X0[0, 0] = np.inf
    with pytest.raises(sa.SbhError) as e:
        sa.block_gmres_preconditioned_with_guess(op, B, None, X0)
    assert "initial guess" in str(e.value)
    op.close()


@pytest.mark.parametrize("n_theta,n_phi", [(5, 3), (5, 17), (9, 40), (21, 61)])
@pytest.mark.parametrize("k", [1, 8, 9, 24, 33, 41, 56, 57, 64, 70])
def test_block_product_tiles_and_slices(ctx, n_theta, n_phi, k):
    """Every column tile count (8 columns each, the last ragged, two chunks at
    70) on 24 to 2440 panels, one to 16 K slices with a short last one; FP64 sums
    in another order: 1e-14 of |A| |X|, and the allocation-free entry point's
    bits."""
    from sonium_amd.mesh import fibonacci_sphere

    m = fibonacci_sphere(1.0, n_theta, n_phi)
    n = m.num_elements
    ph = sa.PhysicsParams.from_wavenumber(1.0)
    system = sa.build_tbem_system(ctx, sa.TbemMesh(ctx, m), ph)
    op = sa.DenseMatrixOperator(system)
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k))
    Y = op.apply_block(X)
    A = system.matrix
    assert np.max(np.abs(Y - A @ X) / (np.abs(A) @ np.abs(X))) <= 1e-14
    x, y = sa.DeviceVector(ctx, n * k), sa.DeviceVector(ctx, n * k)
    x.upload(X)
    op.apply_block_noalloc(x, y, k)
    assert np.array_equal(y.download().reshape(n, k), Y)


@pytest.mark.parametrize("n_theta,n_phi", [(5, 3), (5, 17), (9, 40), (21, 61)])
@pytest.mark.parametrize("s", [1, 2, 8, 9, 17, 24, 25, 33, 49, 64])
def test_block_gmres_tiles(ctx, n_theta, n_phi, s):
    """Every tile width of the block products and of the Cholesky QR (16 and 32
    basis vectors, 16 to 128 real columns, ragged) on 24 to 2440 rows, with
    blocks as wide as the space itself, against the oracle's steps.  The reported
    residuals are those of the returned solution to 1e-6, and to 1e-13 where
    rounding of A x is all that is left of them; an error of a solution is at
    most cond(A) times its residual."""
    from sonium_amd.mesh import fibonacci_sphere

    m = fibonacci_sphere(1.0, n_theta, n_phi)
    n = m.num_elements
    system = sa.build_tbem_system(ctx, sa.TbemMesh(ctx, m), sa.PhysicsParams.from_wavenumber(1.0))
    op = sa.DenseMatrixOperator(system)
    rng = np.random.default_rng(n + s)
    B = rng.standard_normal((n, s)) + 1j * rng.standard_normal((n, s))
    A = system.matrix
    sol = sa.block_gmres(op, B, sa.BlockGmresConfig(max_iterations=20, restart=30, tolerance=1e-8))
    ref, st = oracle.block_gmres(A, B, restart=30, max_iterations=20, tol=1e-8)
    assert sol.converged and st["converged"]
    assert abs(sol.iterations - st["iterations"]) <= 1
    norm = np.linalg.norm(B, axis=0)
    residual = np.linalg.norm(B - A @ sol.x, axis=0) / norm
    np.testing.assert_allclose(sol.true_residuals, residual, rtol=1e-6, atol=1e-13)
    smallest = np.linalg.svd(A, compute_uv=False)[-1]
    exact = np.linalg.solve(A, B)
    assert np.all(np.linalg.norm(sol.x - exact, axis=0) <= 1.01 * (residual + 1e-13) * norm / smallest)


@pytest.mark.parametrize("s", [1, 8, 40])
def test_block_gmres_at_the_ends_of_the_range(ctx, s):
    """Squares that still fit (1e150), that overflow (1e160) and that vanish
    (1e-170): solved, refused as numerical, and zero to the norms, with a block
    wider than the 20-panel space among them."""
    system = sa.build_tbem_system(ctx, sa.TbemMesh(ctx, icosphere(1.0, 0)), sa.PhysicsParams.from_wavenumber(1.0))
    op = sa.DenseMatrixOperator(system)
    rng = np.random.default_rng(s)
    B = rng.standard_normal((op.num_rows(), s)) + 1j * rng.standard_normal((op.num_rows(), s))
    cfg = sa.BlockGmresConfig(max_iterations=5, restart=30, tolerance=1e-8)
    assert sa.block_gmres(op, 1e150 * B, cfg).converged
    with pytest.raises(sa.SbhError, match="NaN or infinity"):
        sa.block_gmres(op, 1e160 * B, cfg)
    assert sa.block_gmres(op, 1e-170 * B, cfg).iterations == 0


@pytest.mark.parametrize("n,s,restart", [(48, 1, 200), (60, 12, 20), (60, 24, 20), (80, 40, 20), (200, 64, 9)])
def test_block_gmres_basis_beyond_the_space(ctx, n, s, restart):
    """An operator of rank n / 2 and a tolerance out of reach: once the basis
    fills the space, what rounding leaves of a step passes the rank-drop test, and
    two whole cycles run to an unconverged end with finite results, as in the
    oracle, on more directions than n + 2 s (and, with one column, more steps than
    n + 1)."""
    rng = np.random.default_rng(n + s)
    c = lambda *shape: rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    A, B = c(n, n // 2) @ c(n // 2, n) / n, c(n, s)
    _, st = oracle.block_gmres(A, B, restart=restart, max_iterations=2, tol=1e-30)
    assert st["iterations"] == 2 * restart and not st["converged"] and np.all(np.isfinite(st["true_residuals"]))
    op = sa.CallbackOperator(ctx, n, lambda x: A @ x)
    sol = sa.block_gmres(op, B, sa.BlockGmresConfig(max_iterations=2, restart=restart, tolerance=1e-30))
    assert sol.iterations == 2 * restart and sol.restart_cycles == 2 and sol.max_basis > n + 2 * s
    assert not sol.converged and sol.status == "max_iterations"
    assert np.all(np.isfinite(sol.x)) and np.all(np.isfinite(sol.true_residuals))
    assert np.all(sol.residuals == 0.0)  # as the reference reports a spent budget
    op.close()


@pytest.mark.parametrize("sizes", [[150], [100, 101], [2, 5, 11, 24, 47, 90], [60] * 3 + [61], [30] * 16 + [9] * 9,
                                   [10] * 12 + [25] * 12 + [40] * 16, [3] * 10 + [7] * 10 + [12] * 44])
def test_block_gmres_deflates_within_a_cycle(ctx, sizes):
    """A unitary operator that takes column c sizes[c] steps, and not one less, in
    a space of its own, all hidden by a unitary basis and by mixed columns: the
    block narrows whenever one of them is done, in groups of least-squares steps
    of every width.  The last step solves all columns; with a condition of one
    their errors are the rounding of some 100 projections, 1e-12 with room."""
    rng = np.random.default_rng(len(sizes))
    c = lambda *shape: rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    n, s, o = sum(sizes), len(sizes), 0
    A, B = np.zeros((n, n), complex), np.zeros((n, s), complex)
    for i, d in enumerate(sizes):
        Q = np.linalg.qr(c(d, d))[0]
        A[o:o + d, o:o + d] = (Q * np.exp(2j * np.pi * np.arange(d) / d)) @ Q.conj().T
        B[o:o + d, i] = c(d)
        o += d
    P = np.linalg.qr(c(n, n))[0]
    A, B = P @ A @ P.conj().T, P @ B @ c(s, s)
    op = sa.CallbackOperator(ctx, n, lambda x: A @ x)
    sol = sa.block_gmres(op, B, sa.BlockGmresConfig(max_iterations=1, restart=200, tolerance=1e-10))
    assert sol.converged and sol.iterations == max(sizes) and sol.max_basis <= n
    assert np.linalg.norm(sol.x - A.conj().T @ B) <= 1e-12 * np.linalg.norm(B)
    op.close()
