"""The K-panels of the per-stage kernels at the edges of tiles and panels: the 32 x 32 and 64 x 64
tiles, the K-split parts (empty ones among them) and the deep panels of single large systems."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _prop(n, batch, kd, precision, variant, one_sided=False):
    from lime_amd.propagator import LindbladPropagator
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 * n + kd)
    c = lambda *s: torch.complex(*(torch.randn(*s, dtype=torch.float64, device="cuda", generator=g) for _ in range(2)))
    x = c(1, n, n)
    H = ((x + x.conj().transpose(-1, -2)) / (4 * n ** 0.5)).resolve_conj().contiguous()
    D = 0.05 * c(1, n, n)
    L, R = (0.3 * c(1, kd, n, n) / n, 0.3 * c(1, kd, n, n) / n) if kd else (None, None)
    p = LindbladPropagator.from_folded(H, D, L, R, group=batch, precision=precision, force_tiled=True,
                                       one_sided=one_sided)
    p.variant = variant
    return p, (c(1, n, n) / n).repeat(batch, 1, 1).contiguous()


def _run(*args, steps=2, **kw):
    p, x = _prop(*args, **kw)
    p.step(x, 0.05, steps)
    return x


@pytest.mark.parametrize("precision", ["fp32", "fp64", "3xbf16"])
@pytest.mark.parametrize("n,kd", [(1, 1), (3, 0), (15, 1), (16, 0), (17, 2), (31, 0), (32, 1), (33, 0), (47, 1), (63, 0),
                                  (64, 2), (65, 0), (96, 1), (97, 0), (100, 2), (129, 0)])
def test_tiles_agree_bit_for_bit_and_with_fp64(n, kd, precision):
    """Both tile edges sum the products of an element in the same order (but for the bordered
    layout, which only the 32-tiles have at n = 33, 97 without dense operators); the K-split
    sums parts, so it differs by rounding.  FP32 sums of n (2 + kd) products of order 1 / n each, two steps of
    dt 0.05: 1e-6 of the largest element, and of FP64 1e-13."""
    small = _run(n, 2, kd, precision, 1)
    assert torch.equal(small, _run(n, 2, kd, precision, 2)) or (kd == 0 and n % 64 == 33)
    ref = _run(n, 2, kd, "fp64", 1)
    scale = float(ref.abs().max())
    tol = (1e-13 if precision == "fp64" else 1e-6) * scale
    for v in range(5):
        assert float((_run(n, 2, kd, precision, v) - ref).abs().max()) < tol, v


@pytest.mark.parametrize("n,kd", [(128, 2), (130, 1), (160, 0), (190, 1), (192, 1), (194, 1), (206, 0), (208, 1), (223, 1),
                                  (224, 0), (258, 1), (286, 0), (288, 1), (289, 0), (290, 1), (322, 0)])
def test_split_products_at_the_sizes_where_the_panel_loads_change(n, kd):
    """3xBF16 with untested loads (no remainder panel, or many whole ones at even n) and with tested ones.
    The split keeps 16 bits of an element, 7.6e-6; two steps of dt 0.05 whose derivative is of the order of
    the state and whose n (2 + kd) errors average: under 1e-6 of the largest element."""
    small = _run(n, 2, kd, "3xbf16", 1)
    assert torch.equal(small, _run(n, 2, kd, "3xbf16", 2)) or (kd == 0 and n % 64 == 33)
    ref = _run(n, 2, kd, "fp64", 1)
    for v in (0, 1, 3, 4):
        assert float((_run(n, 2, kd, "3xbf16", v) - ref).abs().max()) < 1e-6 * float(ref.abs().max()), v


@pytest.mark.parametrize("one_sided", [False, True])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n,kd", [(256, 0), (256, 3), (305, 2), (320, 1), (500, 2), (512, 1)])
def test_deep_panels_give_the_bits_of_the_tiles(n, kd, precision, one_sided):
    """One system of n >= 256 runs on the deep panels, a batch of more than 256 tiles does not."""
    batch = 256 // (-(-n // 32)) ** 2 + 1
    one = _run(n, 1, kd, precision, 1, one_sided=one_sided)
    many = _run(n, batch, kd, precision, 1, one_sided=one_sided)
    assert torch.equal(one[0], many[0]) and torch.equal(one[0], many[-1])
    assert bool(torch.isfinite(torch.view_as_real(one)).all())
