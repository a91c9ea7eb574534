"""The deep panels of a single large system with the bordered layout (no dense operators, n = 32 m + 1):
n = 417 and 481 are the sizes that take both by default, and sizes with a narrower last panel that take
the deep panels alone.  Against the ordinary 32-tiles, which a batch of them runs on, bit for bit, and
against FP64 products in torch: FP32 sums of n products of order 1 / n, two steps of dt 0.05: 1e-6 of
the largest element; FP64 1e-13."""
import pytest
from test_gpu_tiled_panels import _prop, _run

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _deep(n, batch):
    """deep_stage of the library: one tile a CU at most, whole 64-wide panels or nearly."""
    core = n - 1 if n % 32 == 1 else n
    return n >= 256 and batch * (-(-core // 32)) ** 2 <= 256 and -(-n // 64) * 64 * 25 <= n * 27


def _reference(n, steps=2, dt=0.05):
    p, x = _prop(n, 1, 0, "fp64", 1)
    H, D, X = p.heff[0], p.dmat[0], x[0]
    Hd = H.conj().resolve_conj().t().contiguous()
    f = lambda y: -1j * (H @ y - y @ Hd) + D * y
    for _ in range(steps):
        a = f(X)
        b = f(X + dt / 2 * a)
        c = f(X + dt / 2 * b)
        X = X + dt / 6 * (a + 2 * b + 2 * c + f(X + dt * c))
    return X


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [417, 481, 310, 500, 509])
def test_deep_panels_with_a_border_or_a_narrow_last_panel(n, precision):
    many = 256 // (-(-(n - 1 if n % 32 == 1 else n) // 32)) ** 2 + 1
    assert _deep(n, 1) and not _deep(n, many)
    one, batch = _run(n, 1, 0, precision, 1), _run(n, many, 0, precision, 1)
    assert torch.equal(one[0], batch[0]) and torch.equal(one[0], batch[-1])
    ref = _reference(n)
    err = float((one[0] - ref).abs().max() / ref.abs().max())
    print(f"n={n} {precision}: {err:.2e}")
    assert err < (1e-6 if precision == "fp32" else 1e-13)
    assert torch.equal(_run(n, 1, 0, precision, 0), one)          # the default takes the same route
