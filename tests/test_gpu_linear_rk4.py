"""lime_linear_rk4 (RK4 of dx/dt = G x in blocks of steps) against RK4 step by step in NumPy.

Tolerance: the increments are rounded to eps = 2.2e-16 of their largest entry and a block of 64
steps is 6 doublings, so after N steps the states are off by at most a few N M eps of the largest
(N <= 200, M <= 65: 3e-12)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 3, 4, 16, 17, 33, 65])
@pytest.mark.parametrize("rows,steps", [(1, 1), (1, 2), (3, 63), (1, 64), (2, 65), (1, 200)])
def test_matches_step_by_step_rk4(M, rows, steps):
    from lime_amd.redfield import linear_rk4
    rng = np.random.default_rng(100 * M + steps)
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    G, x, E, h = c(M, M) / np.sqrt(M) - 0.5 * np.eye(M), c(rows, M), c(2, M), 0.05
    up = lambda a: torch.as_tensor(a, device="cuda")
    x0 = up(x)
    last, states, obs = linear_rk4(G, x0, h, steps, up(E))
    assert np.array_equal(x0.cpu().numpy(), x)              # the caller's vectors are not changed
    ref = []
    for _ in range(steps):
        k1 = x @ G.T
        k2 = (x + h / 2 * k1) @ G.T
        k3 = (x + h / 2 * k2) @ G.T
        x = x + h / 6 * (k1 + 2 * k2 + 2 * k3 + (x + h * k3) @ G.T)
        ref.append(x)
    ref = np.array(ref)
    tol = 3e-12 * max(1.0, np.max(np.abs(ref)))
    assert np.max(np.abs(states.cpu().numpy() - ref)) < tol
    assert np.max(np.abs(last.cpu().numpy() - ref[-1])) < tol
    assert np.max(np.abs(obs.cpu().numpy() - ref @ E.T)) < 10 * M * tol
    again, none, obs2 = linear_rk4(G, x0, h, steps, up(E), keep=False)
    assert none is None and torch.equal(again, last) and torch.equal(obs2, obs)


def test_refuses_what_does_not_fit():
    from lime_amd.redfield import linear_rk4
    x = torch.zeros(1, 4, dtype=torch.complex128, device="cuda")
    with pytest.raises(ValueError):
        linear_rk4(np.eye(3), x, 0.1, 1)
    with pytest.raises(ValueError):
        linear_rk4(np.eye(4), x, 0.1, 1, torch.zeros(1, 3, dtype=torch.complex128, device="cuda"))
