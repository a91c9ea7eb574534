"""Dense jump operators at n = 16 m + 1 .. 4: core tiles and edge outputs apart, the bits of the padded kernel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _c(rng, *s):
    return rng.standard_normal(s) + 1j * rng.standard_normal(s)


@pytest.mark.parametrize("n", [17, 18, 19, 20, 33, 34, 35, 36])
@pytest.mark.parametrize("kd,sandwich,diag,renorm,driven", [(1, False, True, False, False), (2, True, True, False, False),
                                                            (3, False, False, True, False), (1, True, True, True, True)])
def test_edge_layout_gives_the_bits_of_the_padded_one(n, kd, sandwich, diag, renorm, driven):
    """Zero jump operators, enough that the set does not fit the LDS, take a call to the padded kernel
    without changing a value.  Observables are FP64 sums over other lanes: they differ in the last bits."""
    from lime_amd.propagator import LindbladPropagator
    rng = np.random.default_rng(100 * n + kd)
    steps, batch, ne = 4, 3, 3
    x = _c(rng, n, n)
    H = (x + x.conj().T) / (4 * np.sqrt(n)) - 0.02j * np.eye(n)
    D = 0.05 * _c(rng, n, n) if diag else None
    L, R = 0.2 * _c(rng, 1, kd, n, n) / n, 0.2 * _c(rng, 1, kd, n, n) / n
    zeros = np.zeros((1, 60 if n < 32 else 20, n, n), dtype=np.complex128)
    more = lambda M: np.concatenate([M, zeros], axis=1)
    rho = _c(rng, batch, n, n)
    rho = rho @ rho.conj().transpose(0, 2, 1)
    rho /= np.trace(rho, axis1=1, axis2=2)[:, None, None]
    E = torch.as_tensor(_c(rng, 1, ne, n, n), device="cuda")
    hs = None
    if driven:
        hs = torch.as_tensor(np.stack([H + 0.1 * k * _c(rng, n, n) / n for k in range(steps)])[:, None], device="cuda")
        hs = hs.to(torch.complex64).contiguous()
    out = []
    for l, r in ((L, R), (more(L), more(R))):
        prop = LindbladPropagator.from_folded(H, D, l, r if sandwich else None, group=batch)
        z = torch.as_tensor(rho, device="cuda").clone()
        obs = torch.zeros(batch, steps // 2, ne, dtype=torch.complex128, device="cuda")
        states = torch.zeros(batch, steps // 2, n, n, dtype=torch.complex128, device="cuda")
        kw = dict(heff_steps=hs) if driven else {}
        prop.step(z, 0.02, steps, eops_t=E, obs=obs, states=states, nout=2, rec_capacity=steps // 2, renorm=renorm, **kw)
        out.append((z, obs, states))
    (z, obs, states), (zp, obsp, statesp) = out
    assert torch.equal(z, zp) and torch.equal(states, statesp) and torch.equal(states[:, -1], z)
    assert float((obs - obsp).abs().max()) < 1e-12 * n
    one = LindbladPropagator.from_folded(H, D, L, R if sandwich else None, group=batch)
    y = torch.as_tensor(rho, device="cuda").clone()              # without records
    one.step(y, 0.02, steps, renorm=renorm, **(dict(heff_steps=hs) if driven else {}))
    assert torch.equal(y, z)
