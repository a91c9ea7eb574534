"""Batched Lindblad RK4 propagation on the GPU through liblime_hip.so.

``LindbladPropagator`` owns the device-side operator sets of a batch (H_eff, the
Hadamard dissipator D, the dense jump operators) and advances complex128 operators
``rho`` (density matrices or quantum-regression operators) with the fused kernel
``lime_lindblad_rk4``.  It is the engine behind the lime-compatible facade in
``lime_amd.oqs``; it replaces the per-step NumPy loop of lime's ``_lindblad``
(lime/oqs.py:1590-1688) and of the QRT drivers (oqs.py:726-800, 1227-1331).

Right-hand side (all jump operators folded):
    f(X) = -i (H_eff X - X H_eff^dag) + D o X + sum_dense L X L^dag,
    H_eff = H - (i/2) sum_all L^dag L,  D = sum_{diagonal L = diag(l)} l l^dag.
"""
import ctypes

import numpy as np
import torch

from . import _lib

_PREC_FLAGS = {"fp32": _lib.LIME_F_PREC_FP32, "3xbf16": _lib.LIME_F_PREC_3XBF16,
               "fp64": _lib.LIME_F_PREC_FP64}


def device():
    """The GPU the library runs on; raises when none is visible (no CPU fallback)."""
    if not torch.cuda.is_available():
        raise RuntimeError("lime_amd needs an AMD Instinct GPU (ROCm): no GPU is visible")
    return torch.device("cuda", torch.cuda.current_device())


def _as_tensor(a):
    """A NumPy array as a CPU tensor (torch takes no negative strides)."""
    return torch.as_tensor(a if min(a.strides, default=0) >= 0 else a.copy())


def as_c128(x, dev):
    """Array-like or tensor -> contiguous complex128 tensor on ``dev``."""
    if isinstance(x, torch.Tensor):
        # a conjugate view's memory holds the unconjugated numbers, and the kernels read the memory
        t = x.to(device=dev, dtype=torch.complex128).resolve_conj().resolve_neg()
    else:
        if hasattr(x, "toarray"):          # scipy.sparse
            x = x.toarray()
        t = _as_tensor(np.asarray(x, dtype=np.complex128)).to(dev)
    return t.contiguous()


def _check(t, what, shape, dtype, dev):
    """Every buffer handed to the C ABI is indexed by the kernels from the descriptor's
    sizes alone: its shape, dtype, layout and device are checked here, on the host."""
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{what} must be a torch tensor")
    if t.dtype != dtype or not t.is_contiguous() or t.device != dev or t.is_conj() or t.is_neg():
        raise ValueError(f"{what} must be a contiguous {dtype} tensor on {dev}")
    if tuple(t.shape) != tuple(shape):
        raise ValueError(f"{what} has shape {tuple(t.shape)}, expected {tuple(shape)}")


def _stack_sets(x, nsets, n, dev, what):
    t = as_c128(x, dev)
    if t.dim() == 2:
        t = t.unsqueeze(0)
    if t.shape[-2:] != (n, n):
        raise ValueError(f"{what} has shape {tuple(t.shape)}, expected (..., {n}, {n})")
    if t.shape[0] == 1 and nsets > 1:
        t = t.expand(nsets, n, n)
    if t.shape[0] != nsets:
        raise ValueError(f"{what} has {t.shape[0]} sets, expected {nsets}")
    return t.contiguous()


def _on_host(x):
    """NumPy complex128 of host data (arrays, lists, sparse matrices, CPU tensors); None for a
    tensor on a GPU."""
    if isinstance(x, torch.Tensor):
        return None if x.is_cuda else x.detach().to(torch.complex128).resolve_conj().resolve_neg().numpy()
    return np.asarray(x.toarray() if hasattr(x, "toarray") else x, dtype=np.complex128)


def as_c128_stack(xs, dev, dim=0):
    """Operators of one shape -> one complex128 tensor on ``dev`` (stacked along ``dim``), in
    one copy where they all come from the host and are small (a copy each costs more than the data)."""
    host = []
    for x in xs:
        h = _on_host(x)
        if h is None or h.nbytes >= _LARGE_BYTES or (host and h.shape != host[0].shape):
            return torch.stack([as_c128(x, dev) for x in xs], dim=dim)
        host.append(h)
    return torch.as_tensor(np.stack(host, axis=dim), device=dev) if host else torch.stack([], dim=dim)


#: operators are looked at on the GPU this many bytes at a time (at least one operator)
_STACK_BYTES = 64 << 20
#: host operators of this size go to the GPU one by one, smaller ones stacked on the host (ms stacked / one by
#: one: 16 of n = 64 0.09 / 0.27, n = 256 0.89 / 0.91, n = 512 6.8 / 2.9), and past their first rows they are
#: looked at there (32 diagonal ones of n = 1024: 49 ms on the host, 22 on the GPU; 64 of n = 512 25 / 14)
_LARGE_BYTES = 1 << 20


def _is_diagonal(t, rows=None):
    """Are all off-diagonal entries of (sets, n, n) (of the first ``rows`` rows) exactly zero and the
    diagonals finite?  (NumPy)"""
    d = t.diagonal(0, -2, -1)
    if t.size <= 1 << 14:
        return np.count_nonzero(t) == np.count_nonzero(d) and bool(np.isfinite(d).all())
    step = max(1, (1 << 14) // t.shape[-1])
    return bool(np.isfinite(d).all()) and all(
        np.count_nonzero(t[:, r:r + step]) == np.count_nonzero(d[:, r:r + step])
        for r in range(0, t.shape[-1] if rows is None else rows, step))


def _look(T):
    """The diagonals of a stack of operators (sets, K, n, n) and, per operator, whether it has an
    off-diagonal entry or a diagonal one that is not finite."""
    d = torch.diagonal(T, dim1=-2, dim2=-1).clone()
    nz = T != 0
    torch.diagonal(nz, dim1=-2, dim2=-1).copy_((d - d) != 0)
    return d, torch.any(nz.transpose(0, 1).reshape(T.shape[1], -1), dim=1)


def fold_jump_operators(H, c_ops, dev=None):
    """Split jump operators into H_eff, the Hadamard dissipator D and dense operators.

    H: (S, N, N) or (N, N); c_ops: list of (S, N, N) or (N, N) operators (shared).
    Returns complex128 device tensors heff (S,N,N), dmat (S,N,N) or None,
    lops (S,Kd,N,N) or None.  A jump operator is *diagonal* when every off-diagonal
    entry of every set is exactly zero and its diagonal is finite.

    Small host operators are looked at on the host, large ones and operators on the GPU in stacks of up to
    ``_STACK_BYTES`` there (those on the GPU with one read-back for all); of the diagonal ones only the
    diagonals are kept, so many of them cost no memory.  (A product, a test and a synchronisation per
    operator took 110 us each: 3.4 of 5.0 ms of a two-time correlation with 16 on-site operators.)
    """
    dev = dev or device()
    Ht = as_c128(H, dev)
    if Ht.dim() == 2:
        Ht = Ht.unsqueeze(0)
    if Ht.dim() != 3 or Ht.shape[-1] != Ht.shape[-2]:
        raise ValueError(f"H must be (N, N) or (S, N, N), got {tuple(Ht.shape)}")
    S, n = Ht.shape[0], Ht.shape[-1]
    ops, diag = {}, {}                         # dense (or not looked at yet), and diagonals, by number
    groups = {}                                # GPU operators by their number of sets
    large = {}                                 # large host operators by number of sets: a stack, its numbers

    def look_at_large(sets):
        T, ks = large.pop(sets)
        T = T[:, :len(ks)]
        d, off = _look(T)
        for x, (k, dense) in enumerate(zip(ks, off.tolist())):
            (ops if dense else diag)[k] = (T if dense else d)[:, x]

    c_ops = list(c_ops or [])

    def take(k, c):
        t = _on_host(c)
        t = c if t is None else t
        t = t[None] if t.ndim == 2 else t
        if t.shape[-2:] != (n, n):
            raise ValueError(f"c_ops[{k}] has shape {tuple(t.shape)}, expected (..., {n}, {n})")
        sets = t.shape[0]
        if t.ndim != 3 or sets not in (1, S):
            raise ValueError(f"c_ops[{k}] has {sets} sets, expected {S}")
        if isinstance(t, torch.Tensor):
            ops[k] = t
            groups.setdefault(sets, []).append(k)
            return
        small = t.nbytes < _LARGE_BYTES
        if not _is_diagonal(t, None if small else 1):
            ops[k] = t
        elif small:
            diag[k] = t.diagonal(0, -2, -1).copy()
        else:
            if sets not in large:
                room = min(len(c_ops) - k, max(1, _STACK_BYTES // t.nbytes))
                large[sets] = torch.empty((sets, room, n, n), dtype=torch.complex128, device=dev), []
            T, ks = large[sets]
            T[:, len(ks)] = _as_tensor(t)
            ks.append(k)
            if len(ks) == T.shape[1]:
                look_at_large(sets)

    for k, c in enumerate(c_ops):
        take(k, c)
    for sets in list(large):
        look_at_large(sets)
    looked, stacks = [], {}
    for sets, ks in groups.items():
        many = max(1, _STACK_BYTES // max(1, 16 * sets * n * n))
        for part in (ks[x:x + many] for x in range(0, len(ks), many)):
            T = torch.stack([ops[k].to(device=dev, dtype=torch.complex128) for k in part], dim=1)   # (sets, K, n, n)
            d, off = _look(T)
            looked.append((part, d, off))
            if len(part) == len(ks):
                stacks[tuple(ks)] = T
            del T                                           # before the next stack is made
    if looked:
        off = torch.cat([x for _, _, x in looked]).tolist()
        for part, d, _ in looked:
            diag.update({k: d[:, x] for x, k in enumerate(part) if not off[x]})
            del off[:len(part)]
    diags = [diag[k] for k in sorted(diag)]
    dense = [k for k in sorted(ops) if k not in diag]
    stacks = {ks: T for ks, T in stacks.items() if list(ks) == dense}
    gamma = torch.zeros_like(Ht)
    dmat = lops = None

    def stack(xs):                                          # (1 or S, K, ...)
        sets = max(x.shape[0] for x in xs)
        on_host = [not isinstance(x, torch.Tensor) for x in xs]
        if all(on_host) and 16 * sets * int(np.prod(xs[0].shape[1:])) < _LARGE_BYTES:
            wide = [x if x.shape[0] == sets else np.broadcast_to(x, (sets, *x.shape[1:])) for x in xs]
            return torch.as_tensor(np.stack(wide, axis=1), device=dev)
        if not any(on_host):
            return torch.stack([x.to(device=dev, dtype=torch.complex128).expand(sets, *x.shape[1:]) for x in xs], dim=1)
        out = torch.empty((sets, len(xs), *xs[0].shape[1:]), dtype=torch.complex128, device=dev)
        for k, x in enumerate(xs):
            out[:, k] = x if isinstance(x, torch.Tensor) else _as_tensor(x)
        return out

    if dense:
        L = stacks[tuple(dense)] if stacks else stack([ops[k] for k in dense])
        if n <= 64:                                         # one launch: sum L^dag L = V^dag V
            V = L.reshape(L.shape[0], -1, n)
            gamma = gamma + torch.matmul(V.conj().transpose(-1, -2), V)
        else:                                               # its long reduction would idle most CUs
            for k in range(L.shape[1]):
                gamma = gamma + torch.matmul(L[:, k].conj().transpose(-1, -2), L[:, k])
        lops = L.expand(S, *L.shape[1:]).contiguous()
    if diags:
        l = stack(diags)
        lc = l.conj()
        dmat = torch.matmul(l.transpose(-1, -2).contiguous(), lc.resolve_conj().contiguous())
        dmat = dmat.expand(S, n, n).contiguous()
        gamma = gamma + torch.diag_embed((l * lc).sum(dim=1))
    return (Ht - 0.5j * gamma).contiguous(), dmat, lops


class LindbladPropagator:
    """Operator sets for a batch and the kernel call that advances it.

    Parameters
    ----------
    H : (N, N) or (S, N, N) array-like / tensor
    c_ops : list of (N, N) or (S, N, N) jump operators (may be empty/None)
    group : propagated operators per operator set (operator b uses set b // group)
    precision : 'fp32' (FP32 MFMA, default), '3xbf16', 'fp64'
    """

    def __init__(self, H, c_ops=None, group=1, precision="fp32", sandwich=None,
                 force_tiled=False, variant=0):
        """``sandwich``: optional explicit (L, R) lists of (S,N,N) operators contributing
        sum_k L_k X R_k^dag (used instead of folding dense jump operators; H must then
        already be the effective generator).  ``force_tiled`` selects the per-stage tiled
        kernels even for n <= 80."""
        self.dev = device()
        self.force_tiled = bool(force_tiled)
        self.one_sided = False
        self.variant = int(variant)
        self._work = None
        if precision not in _PREC_FLAGS:
            raise ValueError(f"unknown precision {precision!r}; expected one of {sorted(_PREC_FLAGS)}")
        self.precision = precision
        heff, dmat, lops = fold_jump_operators(H, c_ops, self.dev)
        self.nsets, self.n = heff.shape[0], heff.shape[-1]
        self.group = int(group)
        if self.group < 1:
            raise ValueError("group must be >= 1")
        cdt = torch.complex128 if precision == "fp64" else torch.complex64
        self.heff_c128 = heff
        self.heff = heff.to(cdt).contiguous()
        self.dmat = dmat.to(cdt).contiguous() if dmat is not None else None
        self.lops = lops.to(cdt).contiguous() if lops is not None else None
        self.rops = None
        if sandwich is not None:
            Ls, Rs = sandwich
            if len(Ls) != len(Rs):
                raise ValueError("sandwich needs as many left as right factors")
            if self.lops is not None:
                raise ValueError("sandwich terms cannot be combined with dense jump operators")
            if len(Ls):
                self.lops = self._factors(Ls, "L").to(cdt).contiguous()
                self.rops = self._factors(Rs, "R").to(cdt).contiguous()
        self.n_dense = 0 if self.lops is None else self.lops.shape[1]
        self._lib = _lib.load()

    @classmethod
    def from_folded(cls, heff, dmat=None, lops=None, rops=None, group=1, precision="fp32",
                    force_tiled=False, one_sided=False):
        """Build directly from H_eff (S,N,N), D (S,N,N), dense L / R (S,K,N,N) tensors.

        ``one_sided``: drop the X H_eff^dag product, f(X) = -i H_eff X + D o X + sum L X R^dag
        -- with H_eff = i G this steps dX/dt = G X (a Liouville-space generator acting on
        the columns of X; per-stage kernels)."""
        self = object.__new__(cls)
        self.dev = device()
        self.precision = precision
        self.one_sided = bool(one_sided)
        self.force_tiled = bool(force_tiled) or self.one_sided
        self.variant = 0
        self._work = None
        self._lib = _lib.load()
        if precision not in _PREC_FLAGS:
            raise ValueError(f"unknown precision {precision!r}; expected one of {sorted(_PREC_FLAGS)}")
        cdt = torch.complex128 if precision == "fp64" else torch.complex64
        heff = as_c128(heff, self.dev)
        if heff.dim() == 2:
            heff = heff.unsqueeze(0)
        if heff.dim() != 3 or heff.shape[-1] != heff.shape[-2]:
            raise ValueError(f"heff must be (N, N) or (S, N, N), got {tuple(heff.shape)}")
        self.nsets, self.n = heff.shape[0], heff.shape[-1]
        self.group = int(group)
        if self.group < 1:
            raise ValueError("group must be >= 1")
        self.heff_c128 = heff
        self.heff = heff.to(cdt).contiguous()
        self.dmat = _stack_sets(dmat, self.nsets, self.n, self.dev, "dmat").to(cdt).contiguous() \
            if dmat is not None else None
        self.lops = self._op_stack(lops, "lops", cdt)
        self.rops = self._op_stack(rops, "rops", cdt)
        if self.rops is not None and (self.lops is None or self.rops.shape != self.lops.shape):
            raise ValueError("rops needs lops of the same shape")
        self.n_dense = 0 if self.lops is None else self.lops.shape[1]
        return self

    def _factors(self, xs, what):
        """Sandwich factors, (S, N, N) or (N, N) each, as one (S, K, N, N) tensor."""
        if self.nsets == 1 and all(np.shape(x) == (self.n, self.n) for x in xs):
            return as_c128_stack(xs, self.dev).unsqueeze(0)
        return torch.stack([_stack_sets(x, self.nsets, self.n, self.dev, what) for x in xs], dim=1)

    def _op_stack(self, x, what, cdt):
        if x is None:
            return None
        t = as_c128(x, self.dev)
        if t.dim() != 4 or t.shape[0] != self.nsets or t.shape[-2:] != (self.n, self.n):
            raise ValueError(f"{what} has shape {tuple(t.shape)}, expected ({self.nsets}, K, {self.n}, {self.n})")
        return t.to(cdt).contiguous()

    @property
    def batch(self):
        return self.nsets * self.group

    def _resident(self):
        """Does ``step`` run the resident kernel (whose ``variant`` is a launch shape, not
        the tile edge of the per-stage kernels)?"""
        return (not self.force_tiled and not self.one_sided and self.precision == "fp32"
                and self.n <= self.max_n())

    def _tile_variant(self):
        """The ``variant`` field for the per-stage kernels (``apply`` always runs them): a
        tuned tile choice carries over, a resident launch shape does not."""
        return 0 if self._resident() else self.variant

    def tiled(self):
        """The same operator batch on the per-stage kernels (shares the device operators)."""
        t = object.__new__(LindbladPropagator)
        t.__dict__.update(self.__dict__)
        t._work = None
        t.variant = self._tile_variant()
        t.force_tiled = True
        return t

    def adjoint(self):
        """The propagator of the adjoint generator f^dag (same batch layout):
        H_eff -> -H_eff^dag, D -> conj(D), (L, R) -> (L^dag, R^dag)."""
        adj = object.__new__(LindbladPropagator)
        adj.__dict__.update(self.__dict__)
        adj._work = None
        adj.variant = self._tile_variant()
        adj.force_tiled = True
        h = lambda t: t.conj().transpose(-1, -2).resolve_conj().contiguous()
        adj.heff = (-h(self.heff)).contiguous()
        adj.heff_c128 = (-h(self.heff_c128)).contiguous()
        adj.dmat = self.dmat.conj().resolve_conj().contiguous() if self.dmat is not None else None
        adj.lops = h(self.lops) if self.lops is not None else None
        # R = L (rops None) stays implicit: the adjoint's right factors are adj.lops too
        adj.rops = h(self.rops) if self.rops is not None else None
        return adj

    def regrouped(self, group):
        """The same operator sets with ``group`` propagated operators each (shares them)."""
        g = object.__new__(LindbladPropagator)
        g.__dict__.update(self.__dict__)
        g._work = None
        g.group = int(group)
        if g.group < 1:
            raise ValueError("group must be >= 1")
        return g

    def _flags(self):
        return _PREC_FLAGS[self.precision] | (_lib.LIME_F_ONE_SIDED if self.one_sided else 0)

    def _descriptor(self, B):
        d = _lib.LindbladBatch()
        d.batch, d.n, d.group, d.n_dense = B, self.n, self.group, self.n_dense
        d.eop_group = B
        d.flags = self._flags()
        d.variant = self.variant
        d.heff = self.heff.data_ptr()
        d.dmat = self.dmat.data_ptr() if self.dmat is not None else None
        d.lops = self.lops.data_ptr() if self.lops is not None else None
        d.rops = self.rops.data_ptr() if self.rops is not None else None
        return d

    @property
    def operand_dtype(self):
        return torch.complex128 if self.precision == "fp64" else torch.complex64

    def apply(self, x64, *, z=None, y=None, y64=None, acc=None, c_lx=1.0, c_z=1.0, c_acc=1.0,
              stream=None):
        """One generator application V = f(x) (x in the operand precision) with the epilogue
        y = c_lx V + c_z z, y64 = y in the operand precision, acc += c_acc V (all optional)."""
        B, n = self.batch, self.n
        op_dtype = self.operand_dtype
        _check(x64, "x (operand precision)", (B, n, n), op_dtype, self.dev)
        for name, t in (("z", z), ("y", y), ("acc", acc)):
            if t is not None:
                _check(t, name, (B, n, n), torch.complex128, self.dev)
        if y64 is not None:
            _check(y64, "y64 (operand precision)", (B, n, n), op_dtype, self.dev)
        d = self._descriptor(B)
        d.variant = self._tile_variant()
        if self.n_dense > 0:
            need = B * self.n_dense * self.n * self.n * (16 if self.precision == "fp64" else 8)
            if self._work is None or self._work.numel() < need:
                self._work = torch.empty(need, dtype=torch.uint8, device=self.dev)
            d.work, d.work_bytes = self._work.data_ptr(), self._work.numel()
        pair = lambda c: (ctypes.c_double * 2)(complex(c).real, complex(c).imag)
        s = stream if stream is not None else torch.cuda.current_stream(self.dev)
        ptr = lambda t: t.data_ptr() if t is not None else None
        _lib.check(self._lib.lime_lindblad_apply(
            ctypes.byref(d), x64.data_ptr(), ptr(z), ptr(y), ptr(y64), ptr(acc),
            pair(c_lx), pair(c_z), pair(c_acc), ctypes.c_void_p(s.cuda_stream)))

    def variants(self, n_eops=0):
        """Number of launch-shape variants the library offers for this batch."""
        d = self._descriptor(self.batch)
        d.n_eops = n_eops
        d.flags |= (_lib.LIME_F_FORCE_TILED if self.force_tiled else 0)
        return int(self._lib.lime_lindblad_variants(ctypes.byref(d)))

    def max_n(self):
        return self._lib.lime_lindblad_max_n(self.n_dense, _PREC_FLAGS[self.precision])

    def step(self, rho, dt, nsteps, *, eops_t=None, eop_group=None, obs=None, states=None,
             nout=1, step_offset=0, rec_capacity=0, renorm=False, stream=None, stage_states=None,
             heff_steps=None):
        """Advance ``rho`` (B, N, N) complex128 in place by ``nsteps`` RK4 steps (async).

        ``stage_states`` (rec_capacity, 3, B, N, N) complex128 (record-major) receives the
        FP64 stage operands X + h/2 k1, X + h/2 k2, X + h k3 of every recorded step
        (per-stage kernels: the propagator must be ``force_tiled`` for n <= 80).
        ``heff_steps`` (nsteps, nsets, N, N) in the operand precision: the effective
        Hamiltonian of every step (driven systems) in the place of the propagator's own."""
        n, B = self.n, self.batch
        if heff_steps is not None:
            _check(heff_steps, "heff_steps", (int(nsteps), self.nsets, n, n), self.operand_dtype, self.dev)
        _check(rho, "rho", (B, n, n), torch.complex128, self.dev)
        eop_group = int(eop_group or B)
        if eop_group < 1:
            raise ValueError("eop_group must be >= 1")
        n_e = 0
        if eops_t is not None:
            if eops_t.dim() != 4:
                raise ValueError("eops_t must be (E_sets, n_e, N, N)")
            n_e = int(eops_t.shape[1])
            _check(eops_t, "eops_t", (-(-B // eop_group), n_e, n, n), torch.complex128, self.dev)
        if obs is not None:
            if eops_t is None:
                raise ValueError("obs needs eops_t")
            _check(obs, "obs", (B, int(rec_capacity), n_e), torch.complex128, self.dev)
        if states is not None:
            _check(states, "states", (B, int(rec_capacity), n, n), torch.complex128, self.dev)
        if stage_states is not None:
            _check(stage_states, "stage_states", (int(rec_capacity), 3, B, n, n), torch.complex128, self.dev)
        d = _lib.LindbladBatch()
        d.batch, d.n, d.group, d.n_dense = B, n, self.group, self.n_dense
        d.n_eops = n_e
        d.eop_group = eop_group
        d.flags = self._flags() | (_lib.LIME_F_RENORM_TRACE if renorm else 0) \
            | (_lib.LIME_F_FORCE_TILED if self.force_tiled else 0)
        d.variant = self.variant
        d.heff = self.heff.data_ptr()
        d.dmat = self.dmat.data_ptr() if self.dmat is not None else None
        d.lops = self.lops.data_ptr() if self.lops is not None else None
        d.eops_t = eops_t.data_ptr() if eops_t is not None else None
        d.rho = rho.data_ptr()
        d.obs = obs.data_ptr() if obs is not None else None
        d.states = states.data_ptr() if states is not None else None
        d.rops = self.rops.data_ptr() if self.rops is not None else None
        d.stage_states = stage_states.data_ptr() if stage_states is not None else None
        need = int(self._lib.lime_lindblad_workspace_bytes(ctypes.byref(d)))
        if need > 0:
            if self._work is None or self._work.numel() < need:
                self._work = torch.empty(need, dtype=torch.uint8, device=self.dev)
            d.work = self._work.data_ptr()
            d.work_bytes = self._work.numel()
        p = _lib.StepParams()
        p.dt, p.nsteps, p.nout = float(dt), int(nsteps), int(nout)
        p.step_offset, p.rec_capacity = int(step_offset), int(rec_capacity)
        s = stream if stream is not None else torch.cuda.current_stream(self.dev)
        if heff_steps is not None:
            d.heff = heff_steps.data_ptr()
        call = self._lib.lime_lindblad_rk4 if heff_steps is None else self._lib.lime_lindblad_rk4_driven
        _lib.check(call(ctypes.byref(d), ctypes.byref(p), ctypes.c_void_p(s.cuda_stream)))

    def run(self, rho0, dt, nsteps, e_ops=None, nout=1, store_states=False, renorm=False,
            eop_group=None, chunk=None):
        """Propagate ``rho0`` for ``nsteps`` steps, recording after every ``nout`` steps.

        rho0 : (N, N) (broadcast to the batch) or (B, N, N)
        e_ops : list of (N, N) shared observables, or a tensor (E_sets, n_e, N, N) with
                observable set b // eop_group for operator b.
        Returns (rho (B,N,N), obs (B, Nt//nout, n_e) or None, states (B, Nt//nout, N, N) or None),
        all complex128 device tensors.  Records sit at t_r = (r + 1) * nout * dt.
        """
        n, B = self.n, self.batch
        rho = as_c128(rho0, self.dev)
        if rho.dim() == 2:
            rho = rho.unsqueeze(0).expand(B, n, n)
        rho = rho.clone().contiguous()           # the caller's rho0 is never mutated
        eops_t = None
        if e_ops is not None and len(e_ops) > 0:
            if isinstance(e_ops, torch.Tensor) and e_ops.dim() == 4:
                E = as_c128(e_ops, self.dev)
            else:
                E = as_c128_stack(e_ops, self.dev).unsqueeze(0)
            eops_t = E.transpose(-1, -2).contiguous()
            if eop_group is None:
                eop_group = B // E.shape[0]
        nrec = nsteps // nout if nout > 0 else 0
        obs = None
        if eops_t is not None and nrec > 0:
            obs = torch.zeros((B, nrec, eops_t.shape[1]), dtype=torch.complex128, device=self.dev)
        states = None
        if store_states and nrec > 0:
            states = torch.empty((B, nrec, n, n), dtype=torch.complex128, device=self.dev)
        chunk = int(chunk or nsteps)
        done = 0
        while done < nsteps:
            m = min(chunk, nsteps - done)
            self.step(rho, dt, m, eops_t=eops_t, eop_group=eop_group, obs=obs, states=states,
                      nout=nout, step_offset=done, rec_capacity=nrec, renorm=renorm)
            done += m
        return rho, obs, states
