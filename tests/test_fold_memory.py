"""fold_jump_operators with stacks of bounded size: the same results however the operators are cut, and no
copy of all diagonal operators at once."""
import tracemalloc

import numpy as np
import pytest
import scipy.sparse as sp

import test_fold

torch = pytest.importorskip("torch")


def _limits(monkeypatch, stack, large):
    from lime_amd import propagator
    for name, value in (("_STACK_BYTES", stack), ("_LARGE_BYTES", large)):
        monkeypatch.setattr(propagator, name, value)


LIMITS = [(1, 1), (16 * 2 * 36, 1 << 30), (1200, 1), (1 << 30, 1), (1200, 400)]


@pytest.mark.parametrize("limits", LIMITS)
def test_forms_on_the_host_however_they_are_cut(limits, monkeypatch):
    _limits(monkeypatch, *limits)
    test_fold._check(torch.device("cpu"))


@pytest.mark.parametrize("n", [1, 2, 300])
def test_what_is_diagonal(n):
    from lime_amd.propagator import _is_diagonal
    t = np.zeros((2, n, n), complex)
    assert _is_diagonal(t)
    t[:, range(n), range(n)] = 1 + np.arange(n)
    assert _is_diagonal(t)
    for i, j, v in ((n - 1, 0, 1e-300), (0, n - 1, np.nan), (n // 2, n // 2 - 1, 1j)):
        if i != j and j >= 0:
            u = t.copy()
            u[1, i, j] = v
            assert not _is_diagonal(u)
            u[1, i, i] = 0                                       # as many entries as a diagonal has
            assert not _is_diagonal(u)
    for v in (np.nan, np.inf):
        u = t.copy()
        u[0, n - 1, n - 1] = v
        assert not _is_diagonal(u)


def test_sparse_diagonal_operators_are_not_held_as_matrices():
    from lime_amd.propagator import fold_jump_operators
    n, K = 256, 48
    ops = [sp.csr_matrix(([1.0], ([k], [k])), shape=(n, n)) for k in range(K)]
    H = torch.zeros(n, n, dtype=torch.complex128)
    tracemalloc.start()
    fold_jump_operators(H, ops, torch.device("cpu"))
    peak = tracemalloc.get_traced_memory()[1]
    tracemalloc.stop()
    assert peak < 8 * 16 * n * n, peak / (16 * n * n)            # a few matrices, not 48


@pytest.mark.parametrize("large", [1, 1 << 30])
def test_the_order_of_the_operators_is_kept(large, monkeypatch):
    """Dense operators found on the host, on the GPU and in the first rows or past them."""
    from lime_amd.propagator import fold_jump_operators
    _limits(monkeypatch, 3 * 16 * 25, large)
    n = 5
    ops = [(k + 1) * np.eye(n, dtype=complex) for k in range(9)]
    for k, at in ((1, (4, 0)), (3, (0, 4)), (4, (2, 1)), (8, (4, 3))):
        ops[k][at] = 1j
    _, D, L = fold_jump_operators(np.zeros((n, n)), ops, torch.device("cpu"))
    assert np.array_equal(L[0].numpy(), np.stack([ops[k] for k in (1, 3, 4, 8)]))
    assert np.array_equal(D[0].numpy(), np.full((n, n), sum((k + 1) ** 2 for k in (0, 2, 5, 6, 7))))


@pytest.mark.gpu
@pytest.mark.parametrize("limits", LIMITS)
def test_forms_on_the_gpu_however_they_are_cut(limits, monkeypatch):
    _limits(monkeypatch, *limits)
    test_fold.test_forms_on_the_gpu()


@pytest.mark.gpu
@pytest.mark.parametrize("dense", [0, 8])
def test_memory_on_the_gpu(dense):
    from lime_amd.propagator import _STACK_BYTES, fold_jump_operators
    n, K, dev = 512, 64, torch.device("cuda", torch.cuda.current_device())
    one = 16 * n * n
    ops = [torch.diag_embed(torch.randn(n, dtype=torch.complex128, device=dev)) for _ in range(K)]
    ops += [torch.randn(n, n, dtype=torch.complex128, device=dev) for _ in range(dense)]
    H = torch.zeros(n, n, dtype=torch.complex128, device=dev)
    fold_jump_operators(H, ops[:2] + ops[K:K + 1], dev)          # the libraries' own workspaces exist
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats(dev)
    base = torch.cuda.memory_allocated(dev)
    out = fold_jump_operators(H, ops, dev)
    peak = torch.cuda.max_memory_allocated(dev) - base
    # a stack and its mask, the dense operators once, a few matrices
    assert peak < 1.2 * _STACK_BYTES + (dense + 10) * one, peak / one
    assert out[1] is not None and (out[2] is not None) == (dense > 0)


@pytest.mark.parametrize("large", [1, 16 * 9, 1 << 30])
def test_operators_of_any_size_stack_alike(large, monkeypatch):
    from lime_amd.propagator import as_c128_stack
    _limits(monkeypatch, 1 << 20, large)
    rng, cpu = np.random.default_rng(4), torch.device("cpu")
    c = [rng.standard_normal((3, 3)) + 1j * rng.standard_normal((3, 3)) for _ in range(4)]
    xs = [c[0], c[1].tolist(), sp.csr_matrix(c[2]), torch.as_tensor(c[3]).conj()]
    for dim in (0, 1):
        got = as_c128_stack(xs, cpu, dim=dim)
        assert got.is_contiguous() and np.array_equal(got.numpy(), np.stack([*c[:3], c[3].conj()], axis=dim))
    for bad in ([], [c[0], c[1][:2]]):
        with pytest.raises(RuntimeError):
            as_c128_stack(bad, cpu)


@pytest.mark.parametrize("large", [1, 1 << 30])
def test_reversed_arrays(large, monkeypatch):
    """NumPy views with negative strides, which torch does not take."""
    from lime_amd.propagator import as_c128, as_c128_stack, fold_jump_operators
    _limits(monkeypatch, 1 << 20, large)
    cpu = torch.device("cpu")
    a = np.arange(9.0).reshape(3, 3) + 1j
    d = np.diag([1.0 + 0j, 2, 3])
    assert np.array_equal(as_c128(a[::-1], cpu).numpy(), a[::-1])
    assert np.array_equal(as_c128_stack([a[::-1], a.T], cpu).numpy(), np.stack([a[::-1], a.T]))
    _, D, L = fold_jump_operators(a[:, ::-1], [d[::-1, ::-1], a[::-1]], cpu)
    assert np.array_equal(L[0, 0].numpy(), a[::-1]) and np.array_equal(D[0].numpy(), np.outer([3, 2, 1], [3, 2, 1]))
