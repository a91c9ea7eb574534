"""Lazily conjugated tensors: the kernels read a tensor's memory, so what reaches them has to hold the
conjugated numbers."""
import pytest

torch = pytest.importorskip("torch")


def _c(*s):
    g = torch.Generator().manual_seed(7)
    return torch.complex(*(torch.randn(*s, dtype=torch.float64, generator=g) for _ in range(2)))


def _memory(t):
    """A tensor's numbers as they lie in memory."""
    assert t.is_contiguous()
    return torch.view_as_complex(torch.view_as_real(t.conj() if t.is_conj() else t)).clone()


def test_a_conjugate_view_becomes_its_numbers():
    from lime_amd.propagator import as_c128
    x = _c(2, 3)
    for view in (x.conj(), x.conj().t(), x[:, :1].conj(), x.to(torch.complex64).conj()):
        got = as_c128(view, torch.device("cpu"))
        assert got.is_contiguous() and not got.is_conj()
        assert torch.equal(_memory(got), torch.conj_physical(view.conj()).to(torch.complex128))


@pytest.mark.parametrize("n", [1, 3])
def test_operators_of_the_adjoint_generator(n):
    from lime_amd.propagator import LindbladPropagator
    p = object.__new__(LindbladPropagator)
    p.variant, p.force_tiled, p.one_sided, p.precision = 0, True, False, "fp32"
    p.heff_c128 = _c(2, n, n)
    p.heff, p.dmat = p.heff_c128.to(torch.complex64), _c(2, n, n).to(torch.complex64)
    p.lops = p.rops = _c(2, 1, n, n).to(torch.complex64)
    a = p.adjoint()
    star = torch.conj_physical
    for got, want in ((a.dmat, star(p.dmat)), (a.heff, -star(p.heff.transpose(-1, -2))),
                      (a.lops, star(p.lops.transpose(-1, -2))), (a.rops, star(p.rops.transpose(-1, -2)))):
        assert not got.is_conj() and torch.equal(_memory(got), want)


def test_buffers_that_are_conjugate_views_are_refused():
    from lime_amd.propagator import _check
    x = _c(2, 2)
    _check(x, "x", (2, 2), torch.complex128, x.device)
    with pytest.raises(ValueError):
        _check(x.conj(), "x", (2, 2), torch.complex128, x.device)


@pytest.mark.gpu
@pytest.mark.parametrize("B", [1, 2])
def test_a_gradient_handed_in_as_a_conjugate_view(B):
    from lime_amd.adjoint import ChainAbsorption
    ns, nt = 4, 6
    up = lambda t: t.to("cuda")
    eps, J = up(_c(B, ns).real.contiguous()), up(_c(B, ns - 1).real.contiguous())
    gamma, mu, G = torch.tensor(0.02, dtype=torch.float64, device="cuda"), up(_c(ns).real.contiguous()), up(_c(B, nt))
    args = [t.requires_grad_(True) for t in (eps, J, gamma)]
    C = ChainAbsorption.apply(*args, mu, 0.05, nt)
    a = torch.autograd.grad(C, args, grad_outputs=G.conj(), retain_graph=True)
    b = torch.autograd.grad(C, args, grad_outputs=torch.conj_physical(G))
    assert all(torch.equal(x, y) for x, y in zip(a, b))
