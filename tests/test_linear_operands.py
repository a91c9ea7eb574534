"""The buffers that linear_rk4 hands to the C ABI: row-major complex128 whatever the caller's type and
strides, since the kernels index them from the sizes alone."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")


def _cases():
    g = torch.Generator().manual_seed(3)
    c = lambda *s: torch.complex(*(torch.randn(*s, dtype=torch.float64, generator=g) for _ in range(2)))
    x, E = c(2, 4), c(3, 4)
    return {
        "plain": (x, E),
        "transposed": (x.t().contiguous().t(), E.t().contiguous().t()),
        "conjugated": (x.conj(), E.conj()),
        "strided": (torch.stack([x, x], dim=2)[:, :, 0], torch.stack([E, E], dim=1)[:, 0]),
        "complex64": (x.to(torch.complex64), E.to(torch.complex64)),
        "real": (x.real.contiguous(), E.real.to(torch.float32)),
        "no observables": (x, None),
    }


@pytest.mark.parametrize("name", _cases())
def test_operands_are_row_major_complex128(name):
    from lime_amd.redfield import _linear_operands
    x, E = _cases()[name]
    Gt, y, F = _linear_operands(np.eye(4), x, E)
    for got, want in ((Gt, torch.eye(4)), (y, x), (F, E)):
        if want is None:
            assert got is None
            continue
        assert got.dtype == torch.complex128 and got.is_contiguous() and not got.is_conj()
        assert torch.equal(got, want.to(torch.complex128))
    assert y.data_ptr() != x.data_ptr()


def test_what_does_not_fit_is_refused():
    from lime_amd.redfield import _linear_operands, linear_rk4
    x = torch.zeros(2, 4, dtype=torch.complex128)
    for bad in ((np.eye(3), x, None), (np.eye(4), x[0], None), (np.eye(4), np.zeros((2, 4)), None),
                (np.eye(4), x, torch.zeros(1, 3)), (np.eye(4), x, torch.zeros(4))):
        with pytest.raises(ValueError):
            _linear_operands(*bad)
    with pytest.raises(ValueError, match="GPU"):
        linear_rk4(np.eye(4), x, 0.1, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("name", _cases())
def test_results_do_not_depend_on_type_or_strides(name):
    from lime_amd.redfield import linear_rk4
    x, E = _cases()[name]
    G = -0.3 * np.eye(4) + 0.2j * np.diag([1, 2, 3], 1)
    up = lambda t: None if t is None else t.to("cuda")
    plain = lambda t: None if t is None else t.to(torch.complex128).resolve_conj().contiguous()
    a, sa, oa = linear_rk4(G, up(x), 0.05, 70, up(E))
    b, sb, ob = linear_rk4(G, plain(up(x)), 0.05, 70, plain(up(E)))
    assert torch.equal(a, b) and torch.equal(sa, sb) and (oa is None or torch.equal(oa, ob))
