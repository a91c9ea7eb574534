"""Array primitives of lime's hot path (lime/phys.py), for NumPy arrays or torch tensors.

They operate on whatever array type they are given (a GPU torch tensor stays on the GPU).
The propagation itself never goes through ``rk4`` here: the solvers call the fused kernel.

* ``rk4``        -- phys.py:636-649 (classic RK4, in-place update of ``rho``)
* ``comm``       -- phys.py:741-743;  ``anticomm`` -- :746-748;  ``dag`` -- :758
* ``obs_dm``     -- phys.py:837-844: Tr[d rho] (no conjugate on d), here in O(N^2)
* ``transform``  -- phys.py:706-718: v^dag A v
* ``isherm``, ``ket2dm``, ``basis``, ``destroy``, ``pauli`` -- phys.py:1429, 579, 879, 615, 773
* ``expm``       -- phys.py:1352-1401 ('EOM': U(t) from dU/dt = A U by RK4, on the GPU
  kernels); ``ldo`` -- phys.py:1409-1425 (A b)
"""
import numpy as np


def _is_torch(x):
    return type(x).__module__.startswith("torch")


def dag(a):
    if _is_torch(a):
        return a.conj().transpose(-1, -2)
    if hasattr(a, "getH"):
        return a.getH()
    return np.conjugate(a).T


def comm(A, B):
    assert A.shape == B.shape
    return A @ B - B @ A


def anticomm(A, B):
    assert A.shape == B.shape
    return A @ B + B @ A


commutator = comm
anticommutator = anticomm
dagger = dag


def obs_dm(rho, d):
    """Tr[d rho] = sum_ij d_ij rho_ji."""
    if _is_torch(rho):
        return (d * rho.transpose(-1, -2)).sum(dim=(-1, -2))
    if hasattr(rho, "toarray"):
        rho = rho.toarray()
    if hasattr(d, "toarray"):
        d = d.toarray()
    return np.sum(np.asarray(d) * np.asarray(rho).T)


def rk4(rho, fun, dt, *args):
    dt2 = dt / 2.0
    k1 = fun(rho, *args)
    k2 = fun(rho + k1 * dt2, *args)
    k3 = fun(rho + k2 * dt2, *args)
    k4 = fun(rho + k3 * dt, *args)
    rho += (k1 + 2 * k2 + 2 * k3 + k4) / 6.0 * dt
    return rho


def transform(A, v):
    return dag(v) @ (A @ v)


def isherm(a, tol=1e-8):
    a = a.toarray() if hasattr(a, "toarray") else np.asarray(a)
    return np.allclose(a, np.conjugate(a).T, atol=tol)


def ket2dm(psi):
    psi = np.asarray(psi).reshape(-1)
    return np.outer(psi, psi.conj())


def basis(N, j):
    b = np.zeros(N, dtype=np.complex128)
    b[j] = 1.0
    return b


def destroy(N):
    return np.diag(np.sqrt(np.arange(1, N)), 1).astype(np.complex128)


def pauli():
    s0 = np.eye(2, dtype=np.complex128)
    sx = np.array([[0, 1], [1, 0]], dtype=np.complex128)
    sy = np.array([[0, -1j], [1j, 0]], dtype=np.complex128)
    sz = np.array([[1, 0], [0, -1]], dtype=np.complex128)
    return s0, sx, sy, sz


def ldo(b, A):
    """Linear differential operator A b (phys.py:1409-1425)."""
    return A @ b


def _steps_in_blocks(M, steps):
    """Does ``expm`` in FP64 run on ``lime_linear_rk4`` (blocks of steps) for M x M matrices, or step by
    step on the one-sided per-stage kernels?

    All M rows of U are stepped, so the products are M x M x M, which the per-stage kernels stage
    through LDS and ``lime_linear_rk4``, made for few rows, does not (38 against 75 TFLOP/s at
    M = 2048).  It pays by its fewer launches and products while M is small, above that once many steps
    share the block's matrix.  us, one call in blocks / step by step: M = 128, 64 steps 170 / 2317,
    M = 320, 1 step 72 / 86; M = 384, 8 steps 731 / 615, 20 steps 1137 / 1522; M = 512, 8 steps 1317 / 785, 20
    steps 1825 / 1927, 64 steps 3927 / 6109; M = 640, 20 steps 3921 / 3383; M = 1024, 8 steps 9919 / 3814; M = 4096,
    1 step 57900 / 28700."""
    return M <= 320 or (M <= 512 and steps >= 20)


def expm(A, t, method="EOM", precision="fp64"):
    """U(t_k) = e^{A t_k} for the times t (phys.py:1352-1401), as lime's list of Nt arrays.

    'EOM': U(t_0) = I and each further entry one RK4 step of dU/dt = A U with
    dt = t[1] - t[0] (lime's ``interval``), i.e. U(t_k) = P(dt A)^k with the RK4 polynomial
    P; the Nt - 1 steps run on ``lime_linear_rk4`` in FP64 (the default) where
    ``_steps_in_blocks``, else on the one-sided per-stage kernels, recording every step.
    'SOS' raises NotImplementedError, as in lime.
    """
    if method == "SOS":
        raise NotImplementedError("Method of SOS has not been implemented. Choose from EOM")
    if method != "EOM":
        raise ValueError(f"unknown method {method!r}")
    import torch

    from .redfield import _column_chunk, _dense, linear_rk4, liouville_propagator
    t = np.asarray(t, dtype=np.float64)
    Nt = len(t)
    A = _dense(A)
    if A.ndim == 3 and A.shape[0] == 1:
        A = A[0]
    if A.ndim != 2 or A.shape[0] != A.shape[1]:
        raise ValueError(f"A must be (M, M), got {A.shape}")
    if precision == "fp64" and _steps_in_blocks(A.shape[0], Nt - 1):
        from .propagator import as_c128, device
        At = as_c128(A, device())
        M = At.shape[0]
        At = At.transpose(0, 1).contiguous()       # the rows of U step with A^T: U_k = U_(k-1) P(dt A)
        x = torch.eye(M, dtype=torch.complex128, device=At.device)
        out = [x.cpu().numpy()]
        done, chunk = 1, _column_chunk(M)
        while done < Nt:
            m = min(chunk, Nt - done)
            x, st, _ = linear_rk4(At, x, float(t[1] - t[0]), m)
            out.extend(st.cpu().numpy())
            done += m
        return out
    prop = liouville_propagator(A, precision)
    M = prop.n
    U = torch.eye(M, dtype=torch.complex128, device=prop.dev).unsqueeze(0).contiguous()
    out = [U[0].cpu().numpy()]
    if Nt > 1:
        dt = float(t[1] - t[0])
        done, chunk = 0, _column_chunk(M)
        while done < Nt - 1:
            m = min(chunk, Nt - 1 - done)
            st = torch.empty((1, m, M, M), dtype=torch.complex128, device=prop.dev)
            prop.step(U, dt, m, states=st, nout=1, step_offset=0, rec_capacity=m)
            out.extend(st[0].cpu().numpy())
            done += m
    return out
