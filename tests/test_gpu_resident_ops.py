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


@pytest.mark.parametrize("sandwich", [False, True])
@pytest.mark.parametrize("n,kd", [(21, 1), (24, 2), (25, 3), (28, 1), (29, 2), (32, 1), (37, 2), (40, 1), (41, 1), (44, 2),
                                  (45, 1), (48, 1)])
def test_unrolled_reductions_give_the_bits_of_the_staged_ones(n, kd, sandwich):
    """Every length of the reduction that has its own kernel, without and with records, and driven."""
    from lime_amd.propagator import LindbladPropagator
    rng, H, D, L, R = _system(n, kd, 3 * n + kd)
    batch, steps = 256 * 20 + 1, 3
    x = torch.as_tensor(_c(rng, 1, n, n), device="cuda")
    E = torch.as_tensor(_c(rng, 1, 2, n, n), device="cuda")
    many = LindbladPropagator.from_folded(H, D, L, R if sandwich else None, group=batch)
    one = LindbladPropagator.from_folded(H, D, L, R if sandwich else None)
    y = x.repeat(batch, 1, 1)
    many.step(y, 0.02, steps)
    z, r, d = x.clone(), x.clone(), x.clone()
    one.step(z, 0.02, steps)
    obs = torch.empty(1, steps, 2, dtype=torch.complex128, device="cuda")
    one.step(r, 0.02, steps, eops_t=E, obs=obs, nout=1, rec_capacity=steps)
    hs = torch.as_tensor(np.stack([H] * steps)[:, None], device="cuda").to(torch.complex64).contiguous()
    one.step(d, 0.02, steps, eops_t=E, obs=torch.empty_like(obs), nout=1, rec_capacity=steps, heff_steps=hs)
    assert torch.equal(z[0], y[0]) and torch.equal(z[0], y[-1])
    assert torch.equal(r, z) and torch.equal(d, z)


@pytest.mark.parametrize("n", [18, 20, 21, 24, 25, 29, 32, 34, 36, 37, 40, 41, 44, 45, 48, 50, 52, 53, 56, 57, 60, 61, 64])
def test_unrolled_reductions_without_jump_operators(n):
    """One tile a wave, reduction built in, against two tiles a wave with the length read at run time:
    each element's products in the same order."""
    from lime_amd.propagator import LindbladPropagator
    rng, H, D, _, _ = _system(n, 0, n)
    x = torch.as_tensor(_c(rng, 3, n, n), device="cuda")
    E = torch.as_tensor(_c(rng, 1, 2, n, n), device="cuda")
    out = []
    for variant in (0, 1):
        p = LindbladPropagator.from_folded(H, D, group=3)
        p.variant = variant
        y, z = x.clone(), x.clone()
        p.step(y, 0.02, 4)
        obs = torch.empty(3, 4, 2, dtype=torch.complex128, device="cuda")
        p.step(z, 0.02, 4, eops_t=E, obs=obs, nout=1, rec_capacity=4)
        assert torch.equal(y, z)
        out.append(y)
        ref = torch.einsum("eij,bij->be", E[0], z)
        assert float((obs[:, 3] - ref).abs().max()) < 1e-12 * max(1.0, float(ref.abs().max())) * n
    assert torch.equal(*out)


@pytest.mark.parametrize("n", [66, 68, 69, 72, 73, 76, 77, 80])
def test_unrolled_reductions_with_two_tiles_a_wave(n):
    """20 observables leave no room for the second buffer of S: that call reads the reduction's length at
    run time, those with one observable and none have it built in."""
    from lime_amd.propagator import LindbladPropagator
    rng, H, D, _, _ = _system(n, 0, n)
    x = torch.as_tensor(_c(rng, 3, n, n), device="cuda")
    p = LindbladPropagator.from_folded(H, D, group=3)
    out = []
    for ne in (0, 1, 20):
        y = x.clone()
        if ne:
            E = torch.as_tensor(_c(rng, 1, ne, n, n), device="cuda")
            obs = torch.empty(3, 4, ne, dtype=torch.complex128, device="cuda")
            p.step(y, 0.02, 4, eops_t=E, obs=obs, nout=1, rec_capacity=4)
        else:
            p.step(y, 0.02, 4)
        out.append(y)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
