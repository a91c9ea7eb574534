"""phys.expm in FP64: blocks of steps for small matrices, step by step on the staged tiles for large ones.
Both sides against RK4 in NumPy: FP64 sums of M products of order one, N steps of h |A| ~ 0.1: 1e-13."""
import numpy as np
import pytest


def test_large_matrices_do_not_run_on_the_products_made_for_few_rows():
    from lime_amd.phys import _steps_in_blocks
    for M, steps in ((1, 1), (144, 1), (144, 500), (320, 1), (512, 64)):
        assert _steps_in_blocks(M, steps), (M, steps)
    for M, steps in ((400, 3), (513, 64), (1024, 9), (2048, 3), (4096, 1)):
        assert not _steps_in_blocks(M, steps), (M, steps)


@pytest.mark.gpu
@pytest.mark.parametrize("M,steps", [(1, 3), (5, 0), (5, 70), (320, 2), (321, 2), (321, 20), (600, 2)])
def test_both_routes_step_rk4(M, steps):
    from lime_amd import phys
    rng = np.random.default_rng(M)
    A = (rng.standard_normal((M, M)) + 1j * rng.standard_normal((M, M))) / np.sqrt(M)
    h, X, ref = 0.05, np.eye(M, dtype=complex), [np.eye(M)]
    for _ in range(steps):
        k1 = A @ X
        k2 = A @ (X + h / 2 * k1)
        k3 = A @ (X + h / 2 * k2)
        X = X + h / 6 * (k1 + 2 * k2 + 2 * k3 + A @ (X + h * k3))
        ref.append(X)
    for form in (A, A[None]):
        U = phys.expm(form, h * np.arange(steps + 1))
        assert len(U) == steps + 1 and all(u.shape == (M, M) for u in U)
        assert max(np.abs(u - r).max() for u, r in zip(U, ref)) < 1e-13 * max(1.0, np.abs(ref[-1]).max())


@pytest.mark.gpu
def test_redfield_takes_a_tensor_with_a_leading_set():
    from lime_amd.oqs import _redfield
    rng = np.random.default_rng(1)
    R, rho = 0.1 * rng.standard_normal((9, 9)) + 0j, np.diag([0.5, 0.3, 0.2]) + 0j
    a, b = (_redfield(r, rho, Nt=3, dt=0.1) for r in (R, R[None]))
    assert np.array_equal(np.array(a.rholist), np.array(b.rholist))


def test_what_is_no_square_matrix_is_refused():
    from lime_amd import phys
    for bad in (np.zeros((2, 3)), np.zeros(4), np.zeros((2, 3, 3))):
        with pytest.raises((ValueError, RuntimeError)):
            phys.expm(bad, np.arange(3))
