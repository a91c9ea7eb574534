"""Dense jump operators resident in LDS, and driven systems in one launch: the same bits as the
paths they replace."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _c(rng, *s):
    return rng.standard_normal(s) + 1j * rng.standard_normal(s)


def _system(n, kd, seed, diag=True):
    rng = np.random.default_rng(seed)
    x = _c(rng, n, n)
    D = 0.05 * _c(rng, n, n) if diag else None
    L, R = 0.2 * _c(rng, 1, kd, n, n) / n, 0.2 * _c(rng, 1, kd, n, n) / n
    return rng, (x + x.conj().T) / (4 * np.sqrt(n)) - 0.02j * np.eye(n), D, L if kd else None, R if kd else None


@pytest.mark.parametrize("sandwich", [False, True])
@pytest.mark.parametrize("n,kd", [(1, 1), (3, 2), (4, 7), (15, 1), (16, 5), (17, 1), (24, 3), (31, 2), (32, 5), (33, 1),
                                  (48, 2), (49, 1), (64, 1)])
def test_resident_operands_give_the_bits_of_the_staged_ones(n, kd, sandwich):
    """One operator alone keeps its jump operators in LDS; in a batch whose workgroups per CU
    leave no room for them they are staged.  Its bits do not depend on that."""
    from lime_amd.propagator import LindbladPropagator
    rng, H, D, L, R = _system(n, kd, 10 * n + kd)
    batch = 256 * 20 + 1                             # more workgroups than any CU count holds
    x = torch.as_tensor(_c(rng, 3, n, n), device="cuda")
    E = torch.as_tensor(_c(rng, 1, 2, n, n), device="cuda")
    many = LindbladPropagator.from_folded(H, D, L, R if sandwich else None, group=batch)
    one = LindbladPropagator.from_folded(H, D, L, R if sandwich else None)
    y = x.repeat(-(-batch // 3), 1, 1)[:batch].contiguous()
    many.step(y, 0.02, 3)
    for k in range(3):
        z = x[k:k + 1].clone()
        obs = torch.empty(1, 3, 2, dtype=torch.complex128, device="cuda")
        one.step(z, 0.02, 3, eops_t=E, obs=obs, nout=1, rec_capacity=3)
        assert torch.equal(z[0], y[k]) and torch.equal(z[0], y[batch - 3 + (k - (batch - 3)) % 3])
        ref = torch.einsum("eij,ij->e", E[0], z[0])
        assert float((obs[0, 2] - ref).abs().max()) < 1e-12 * max(1.0, float(ref.abs().max())) * n


@pytest.mark.parametrize("n,kd", [(3, 0), (8, 2), (16, 0), (17, 0), (24, 1), (32, 0), (33, 0), (33, 2), (49, 0), (64, 0),
                                  (64, 2), (65, 0), (72, 0), (100, 1)])
def test_driven_call_gives_the_bits_of_a_call_per_step(n, kd):
    from lime_amd.propagator import LindbladPropagator
    rng, H, D, L, _ = _system(n, kd, 7 * n + kd)
    steps, batch = 5, 3
    hs = torch.as_tensor(np.stack([H + 0.1 * k * _c(rng, n, n) / n for k in range(steps)])[:, None], device="cuda")
    hs = hs.to(torch.complex64).contiguous()
    E = torch.as_tensor(_c(rng, 1, 2, n, n), device="cuda")
    x = torch.as_tensor(_c(rng, batch, n, n), device="cuda")
    rec = lambda *s: torch.zeros(batch, steps, *s, dtype=torch.complex128, device="cuda")
    one = LindbladPropagator.from_folded(H, D, L, group=batch)
    a, obs_a, st_a = x.clone(), rec(2), rec(n, n)
    one.step(a, 0.02, steps, eops_t=E, obs=obs_a, states=st_a, nout=1, rec_capacity=steps, heff_steps=hs)
    b, obs_b, st_b = x.clone(), rec(2), rec(n, n)
    for k in range(steps):
        one.heff = hs[k]
        one.step(b, 0.02, 1, eops_t=E, obs=obs_b, states=st_b, nout=1, step_offset=k, rec_capacity=steps)
    assert torch.equal(a, b) and torch.equal(obs_a, obs_b) and torch.equal(st_a, st_b)
    with pytest.raises(ValueError):
        one.step(a, 0.02, steps + 1, heff_steps=hs)
