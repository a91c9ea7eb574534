"""The one-lane-per-element kernel (n <= 16) against the FP64 oracle, and its bits against the MFMA
tiles.  Large batches of n = 9 .. 16 run on the tiles, single operators here: the same operator
has to give the same bits either way.  Against the oracle the FP32 products give 2e-7 of the
largest element after a few steps of dt 0.05 (operators of order one)."""
import numpy as np
import pytest

from oracle import lindblad as ol

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _c(rng, *s):
    return rng.standard_normal(s) + 1j * rng.standard_normal(s)


def _system(n, kd, seed):
    rng = np.random.default_rng(seed)
    x, y = _c(rng, n, n), _c(rng, n, n)
    H = (x + x.conj().T) / (4 * np.sqrt(n))
    c_ops = [0.2 * _c(rng, n, n) / n for _ in range(kd)] + [0.3 * np.diag(rng.standard_normal(n))]
    rho0 = y @ y.conj().T
    return rng, H, c_ops, rho0 / np.trace(rho0)


@pytest.mark.parametrize("kd", [0, 1, 3])
@pytest.mark.parametrize("n", range(1, 17))
def test_matches_the_oracle_with_records(n, kd):
    from lime_amd.propagator import LindbladPropagator
    rng, H, c_ops, rho0 = _system(n, kd, 31 * n + kd)
    batch, steps, dt = 6, 8, 0.05
    E = [_c(rng, n, n), np.eye(n)]
    prop = LindbladPropagator(H, c_ops, group=batch)
    rho, obs, states = prop.run(rho0, dt, steps, e_ops=E, nout=2, store_states=True, renorm=True)
    x = rho0
    for k in range(steps):
        x = ol.propagate(H, x, c_ops, dt, 1)[0]
        x = x / np.trace(x).real
        if k % 2:
            r = k // 2
            got, o = states[:, r].cpu().numpy(), obs[:, r].cpu().numpy()
            assert np.max(np.abs(got - x)) < 2e-7, (k, np.max(np.abs(got - x)))
            assert np.max(np.abs(o - [np.trace(e @ x) for e in E])) < 2e-7 * n * 4
    assert torch.equal(rho, states[:, -1]) and torch.equal(rho, rho[:1].expand_as(rho))


@pytest.mark.parametrize("renorm", [False, True])
@pytest.mark.parametrize("n,kd", [(9, 0), (9, 2), (12, 0), (13, 1), (16, 0), (16, 3)])
def test_bits_of_the_tiles(n, kd, renorm):
    from lime_amd.propagator import LindbladPropagator
    rng, H, c_ops, rho0 = _system(n, kd, 17 * n + kd)
    batch = 1100                                       # on the tiles
    x = torch.as_tensor(np.stack([rho0, rho0 @ rho0, rho0.T]), device="cuda")
    y = x.repeat(-(-batch // 3), 1, 1)[:batch].contiguous()
    LindbladPropagator(H, c_ops, group=batch).step(y, 0.05, 5, renorm=renorm)
    one = LindbladPropagator(H, c_ops)
    for k in range(3):
        z = x[k:k + 1].clone()
        one.step(z, 0.05, 5, renorm=renorm)
        assert torch.equal(z[0], y[k])
