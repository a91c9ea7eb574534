"""fold_jump_operators over the forms it takes, against its definition operator by operator.  The
sums are FP64: 1e-14 of the largest element (K <= 5 operators of order one, n <= 6)."""
import numpy as np
import pytest
import scipy.sparse as sp

torch = pytest.importorskip("torch")


def _ops(S, n, rng):
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    real_diag = np.diag(rng.standard_normal(n))
    sets_diag = np.stack([np.diag(c(n)) for _ in range(S)])
    mixed = np.stack([np.diag(c(n)) for _ in range(S)])        # diagonal in every set but the last
    mixed[-1, 0, n - 1] = 1e-300
    return {
        "none": [],
        "diagonal": [real_diag, np.diag(c(n))],
        "lists_sparse_tensors": [real_diag.tolist(), sp.csr_matrix(np.diag(c(n))), torch.as_tensor(c(n, n)),
                                 torch.as_tensor(c(n, n)).conj(), torch.eye(n, dtype=torch.bfloat16)],
        "sets": [sets_diag, c(S, n, n), real_diag, c(n, n), c(1, n, n)],
        "tiny_off_diagonal": [mixed, np.zeros((n, n))],
        "nan": [np.diag(np.full(n, np.nan)), np.where(np.eye(n), 0, np.nan)],
    }


def _definition(H, c_ops, S, n):
    G, D, dense = np.zeros((S, n, n), complex), None, []
    for c in c_ops:
        x = c.to(torch.complex128).resolve_conj().cpu().numpy() if isinstance(c, torch.Tensor) else c
        x = np.asarray(x.toarray() if hasattr(x, "toarray") else x, dtype=complex)
        x = np.broadcast_to(x, (S, n, n))
        d = np.einsum("sii->si", x)
        if np.any((x - d[:, :, None] * np.eye(n) != 0) & ~np.eye(n, dtype=bool)):
            dense.append(x)
            G = G + np.conj(np.swapaxes(x, 1, 2)) @ x
        else:
            G = G + np.einsum("si,ij->sij", np.abs(d) ** 2, np.eye(n))
            D = (0 if D is None else D) + d[:, :, None] * d[:, None].conj()
    return H - 0.5j * G, D, dense


def _check(dev, to=lambda x: x):
    from lime_amd.propagator import fold_jump_operators
    rng = np.random.default_rng(3)
    for S, n in ((1, 1), (1, 5), (3, 4), (2, 6)):
        H = rng.standard_normal((S, n, n)) + 0j
        for name, c_ops in _ops(S, n, rng).items():
            if n == 1 and name != "diagonal":
                continue
            heff, D, L = fold_jump_operators(H if S > 1 else H[0], [to(c) for c in c_ops], dev)
            rh, rD, rL = _definition(H, c_ops, S, n)
            assert heff.is_contiguous() and heff.shape == (S, n, n)
            assert (D is None) == (rD is None) and (L is None) == (not rL), name
            if name == "nan":
                assert L.shape == (S, len(rL), n, n)
                continue
            assert np.allclose(heff.cpu().numpy(), rh, rtol=0, atol=1e-13), name
            if D is not None:
                assert D.is_contiguous() and np.allclose(D.cpu().numpy(), rD, rtol=0, atol=1e-13), name
            if L is not None:
                assert L.is_contiguous() and np.array_equal(L.cpu().numpy(), np.stack(rL, 1)), name
        for bad in ([np.eye(n + 1)], [np.zeros((S + 1, n, n))], [np.zeros(n)]):
            with pytest.raises(ValueError):
                fold_jump_operators(H, [to(b) for b in bad], dev)


def test_forms_on_the_host():
    _check(torch.device("cpu"))


@pytest.mark.gpu
def test_forms_on_the_gpu():
    dev = torch.device("cuda")
    _check(dev)
    dense = lambda c: c.toarray() if hasattr(c, "toarray") else np.asarray(c) if isinstance(c, list) else c
    _check(dev, lambda c: torch.as_tensor(dense(c), device=dev))
