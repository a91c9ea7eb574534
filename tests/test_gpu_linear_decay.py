"""lime_linear_rk4 on decaying systems: every record relative to its own size, against RK4 step by step
in 80 bits.  The matrices of a block hold 106 bits, so a record r carries the rounding of the
products of states that lead to it: at most 7 + r / 64, each a sum of M <= 17 terms of the record's size
(normal generators; the fastest modes decay below the slowest ones, so no product cancels), under
10 eps of the record."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
STEPS = 200
TOL = 10 * 2.2e-16 * (7 + np.arange(STEPS) / 64.0)


def _rk4(G, x, h, steps, dtype=np.clongdouble):
    x, GT, h = x.astype(dtype), G.T.astype(dtype), np.longdouble(h) if dtype == np.clongdouble else h
    out = []
    for _ in range(steps):
        k1 = x @ GT
        k2 = (x + h / 2 * k1) @ GT
        k3 = (x + h / 2 * k2) @ GT
        x = x + h / 6 * (k1 + 2 * k2 + 2 * k3 + (x + h * k3) @ GT)
        out.append(x)
    return np.array(out)


def _generator(kind, M, z, rng):
    c = rng.standard_normal((M, M)) + 1j * rng.standard_normal((M, M))
    Q = np.linalg.qr(c)[0]
    if kind == "uniform":
        return -z * np.eye(M) + 0j
    if kind == "rotating":                                    # uniform damping of coupled oscillators
        return -z * np.eye(M) + 1j * Q @ np.diag(rng.uniform(-0.5, 0.5, M)) @ Q.conj().T
    return Q @ np.diag(-z * np.linspace(0.5, 1.0, M)) @ Q.conj().T      # "rates"


@pytest.mark.parametrize("kind", ["uniform", "rotating", "rates"])
@pytest.mark.parametrize("M", [1, 4, 17])
@pytest.mark.parametrize("z", [0.02, 0.25, 0.5, 1.0, 1.6])
def test_records_of_damped_systems_keep_their_digits(kind, M, z):
    from lime_amd.redfield import linear_rk4
    rng = np.random.default_rng(int(1000 * z) + M)
    h = 0.05
    G = _generator(kind, M, z, rng) / h
    x = rng.standard_normal((2, M)) + 1j * rng.standard_normal((2, M))
    ref = _rk4(G, x, h, STEPS)
    _, states, _ = linear_rk4(G, torch.as_tensor(x, device="cuda"), h, STEPS)
    err = np.abs(states.cpu().numpy() - ref).max(axis=(1, 2)) / np.abs(ref).max(axis=(1, 2))
    print(f"{kind} M={M} z={z}: {float(np.max(err / TOL)):.2e} of the bound, last {float(err[-1]):.1e}")
    assert np.all(err < TOL)


def test_every_decoupled_element_keeps_its_digits_and_expm_too():
    from lime_amd import phys
    from lime_amd.redfield import linear_rk4
    rng = np.random.default_rng(5)
    z, h = np.array([0.0, 1e-3, 0.1, 0.3, 0.5, 0.7, 1.0, 2.0]), 0.05
    G = np.diag(-z / h + 1j * rng.uniform(-5, 5, len(z)))
    x = rng.standard_normal((1, len(z))) + 1j
    ref = _rk4(G, x, h, STEPS)
    _, states, _ = linear_rk4(G, torch.as_tensor(x, device="cuda"), h, STEPS)
    err = np.abs(states.cpu().numpy() - ref) / np.abs(ref)
    assert np.all(err < TOL[:, None, None])
    U = np.array(phys.expm(G, h * np.arange(STEPS + 1)))
    want = _rk4(G, np.ones((1, len(z))), h, STEPS)[:, 0]
    got = np.einsum("kii->ki", U[1:])
    assert np.all(np.abs(got - want) / np.abs(want) < TOL[:, None])
