"""fold_jump_operators with stacks of bounded size: the same results however the operators are cut, and no
copy of all diagonal operators at once."""
import tracemalloc

import numpy as np
import pytest
import scipy.sparse as sp

import test_fold

torch = pytest.importorskip("torch")


def _limits(monkeypatch, stack, copy, look):
    from lime_amd import propagator
    for name, value in (("_STACK_BYTES", stack), ("_COPY_BYTES", copy), ("_LOOK_BYTES", look)):
        monkeypatch.setattr(propagator, name, value)


LIMITS = [(1, 1, 1), (16 * 2 * 36, 1, 1 << 30), (1200, 1 << 30, 1), (1 << 30, 1, 1), (1200, 600, 400)]


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


@pytest.mark.parametrize("look", [1, 1 << 30])
def test_the_order_of_the_operators_is_kept(look, monkeypatch):
    """Dense operators found on the host, on the GPU and in the first rows or past them."""
    from lime_amd.propagator import fold_jump_operators
    _limits(monkeypatch, 3 * 16 * 25, 1, look)
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
