"""The work that users of lime_amd have it do, as cases that can be timed and compared.

``listed()`` names the standing cases, ``draw(rng)`` gives one more of the same ranges.
``prepare(case, seed)`` makes what a program holds before the call, ``run(state)`` is one
pass through the public entry points, ``work(case)`` the bytes and operations that the path
cannot do without, and ``exact(case, seed)`` the same outputs in 64 bits from plain torch.

Kinds
-----
chain      -- ``oqs.Lindblad_solver.evolve`` on one small exciton chain: arrays in, a Result out
driven     -- ``evolve`` with H = [H0, [H1, f1], [H2, f2]] (time-dependent fields)
two_time   -- ``correlation_3op_2t``: a grid of two-time correlations for a 2D spectrum
redfield   -- ``oqs.Redfield_solver.evolve``: Bloch-Redfield in Hilbert space
liouville  -- ``oqs._redfield``: RK4 on vec rho with an explicit Liouville tensor, FP64
absorption -- ``LindbladPropagator.run`` on an ensemble of regression operators, C(t) each step
ensemble   -- ``LindbladPropagator.run`` on an ensemble of density matrices, populations
dense      -- ``LindbladPropagator.run`` with dense jump operators (the compute-bound point)
ragged     -- ``RaggedLindblad.run``: instances of uneven n in one launch
gradient   -- ``ChainAbsorption`` forward and backward behind a spectrum loss
"""
import math

import numpy as np
import torch

GAMMA = 0.01          # on-site dephasing rate of the excitonic kinds
RAGGED_SIZES = tuple(range(16, 257, 16))


def listed():
    return [
        # the smallest call: the 8-site chain of the examples, populations every 10 steps
        dict(name="chain8", kind="chain", n=8, steps=2000, nout=10),
        # a laser-driven system of 33 levels, every step recorded
        dict(name="driven33", kind="driven", n=33, steps=400),
        # a 2D spectrum of 16 sites + ground state on a 128 x 128 grid of times
        dict(name="two_time17", kind="two_time", n=17, steps=128, tau_steps=128),
        # an exciton complex of 24 states with 4 baths
        dict(name="redfield24", kind="redfield", n=24, baths=4, steps=100),
        # lime's Liouville-space RK4 with an explicit tensor, 12 states (144 x 144)
        dict(name="liouville12", kind="liouville", n=12, steps=500),
        # the headline ensemble: 4096 disorder realisations of an 8 x 8 lattice + ground
        # state, three dipole components each
        dict(name="lattice65", kind="absorption", n=65, sets=4096, group=3, steps=96, precision="fp32"),
        # the same ensemble in split-product arithmetic
        dict(name="lattice65_3xbf16", kind="absorption", n=65, sets=4096, group=3, steps=96, precision="3xbf16"),
        # density matrices of a size that is no multiple of any tile, trace renormalised
        dict(name="ensemble100", kind="ensemble", n=100, batch=256, steps=20, observables=4, precision="fp32"),
        # one large dense system, 16 dense jump operators
        dict(name="dense512", kind="dense", n=512, batch=1, jumps=16, steps=10, precision="fp32"),
        # a batch of them in split-product arithmetic: the largest dense work
        dict(name="dense512_3xbf16", kind="dense", n=512, batch=16, jumps=16, steps=5, precision="3xbf16"),
        # uneven systems of 16 .. 256 states, four dense jump operators each
        dict(name="ragged256", kind="ragged", count=256, jumps=4, steps=20, sizes=3),
        # gradient of an absorption spectrum with respect to the parameters of 128 chains
        dict(name="gradient129", kind="gradient", n=129, batch=128, steps=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chain", "driven", "two_time", "redfield", "liouville", "absorption", "ensemble", "dense",
                       "ragged", "gradient"])
    if kind == "chain":
        n = _log(rng, 3, 96)
        return dict(kind=kind, n=n, steps=10 * _log(rng, 10, 200), nout=10)
    if kind == "driven":
        return dict(kind=kind, n=_log(rng, 3, 64), steps=_log(rng, 50, 600))
    if kind == "two_time":
        return dict(kind=kind, n=_log(rng, 3, 49), steps=_log(rng, 16, 128), tau_steps=_log(rng, 16, 128))
    if kind == "redfield":
        return dict(kind=kind, n=_log(rng, 3, 32), baths=rng.randint(1, 5), steps=_log(rng, 20, 200))
    if kind == "liouville":
        return dict(kind=kind, n=_log(rng, 2, 16), steps=_log(rng, 50, 600))
    if kind == "absorption":
        n = _log(rng, 9, 80)
        return dict(kind=kind, n=n, sets=_log(rng, 64, max(64, min(4096, 4096 * 65 ** 3 // (2 * n ** 3)))), group=3,
                    steps=_log(rng, 16, 96), precision=rng.choice(["fp32", "fp32", "3xbf16"]))
    if kind == "ensemble":
        n = _log(rng, 12, 200)
        return dict(kind=kind, n=n, batch=_log(rng, 1, max(2, min(1024, 256 * 100 ** 3 // n ** 3))),
                    steps=_log(rng, 10, 60), observables=rng.randint(1, 6),
                    precision=rng.choice(["fp32", "fp32", "3xbf16", "fp64"]))
    if kind == "dense":
        n = _log(rng, 24, 512)
        kd = _log(rng, 1, 16)
        return dict(kind=kind, n=n, batch=_log(rng, 1, max(2, min(256, 8 * 512 ** 3 // n ** 3))), jumps=kd,
                    steps=rng.randint(3, 10), precision=rng.choice(["fp32", "fp32", "3xbf16", "fp64"]))
    if kind == "ragged":
        return dict(kind=kind, count=_log(rng, 8, 256), jumps=rng.randint(0, 5), steps=10 * rng.randint(1, 3),
                    sizes=rng.randint(0, 1 << 20))
    return dict(kind=kind, n=_log(rng, 24, 160), batch=_log(rng, 2, 128), steps=_log(rng, 32, 128))


# ---------------------------------------------------------------------------- inputs
def _chain_h(eps, J):
    n = len(eps)
    H = np.diag(np.asarray(eps, dtype=np.float64)).astype(np.complex128)
    for i in range(n - 1):
        H[i, i + 1] = H[i + 1, i] = J
    return H


def _sites(n, first, gamma):
    """On-site dephasing operators sqrt(gamma) |i><i|, i = first .. n - 1."""
    ops = []
    for i in range(first, n):
        L = np.zeros((n, n), dtype=np.complex128)
        L[i, i] = math.sqrt(gamma)
        ops.append(L)
    return ops


def _herm(rng, n):
    x = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return (x + x.conj().T) / 2 / math.sqrt(n)


def _pure(rng, n):
    psi = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    psi /= np.linalg.norm(psi)
    return np.outer(psi, psi.conj())


def _ohmic(eta, beta):
    """An Ohmic bath's spectral function with a cut-off at 2."""
    def S(w):
        w = np.asarray(w, dtype=np.float64)
        with np.errstate(divide="ignore", invalid="ignore"):
            v = eta * w * np.exp(-np.abs(w) / 2.0) / (1.0 - np.exp(-beta * w))
        return np.where(np.abs(w) < 1e-12, eta / beta, v)
    return S


def _inputs(case, seed):
    """The inputs of a case, made from the seed alone: NumPy arrays for the kinds that take
    arrays, tensors on the GPU for the ensembles."""
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "chain":
        n = case["n"]
        rho0 = np.zeros((n, n), dtype=np.complex128)
        rho0[0, 0] = 1.0
        return dict(H=_chain_h(rng.normal(0.0, 0.05, n), -0.1), c_ops=_sites(n, 0, 0.02), rho0=rho0, dt=0.05,
                    e_ops=[np.diag(np.eye(n)[i]).astype(np.complex128) for i in range(min(n, 8))])
    if kind == "driven":
        n = case["n"]
        a = np.diag(np.sqrt(np.arange(1, n)), 1).astype(np.complex128) / math.sqrt(n)
        amp = rng.uniform(0.2, 0.4, 2)
        fields = [lambda t, s=amp[0]: s * math.cos(1.1 * t) * math.exp(-((t - 4.0) / 3.0) ** 2),
                  lambda t, s=amp[1]: s * math.sin(0.7 * t)]
        e_ops = [a.conj().T @ a, a + a.conj().T]
        return dict(H0=_herm(rng, n), drives=[a + a.conj().T, 1j * (a.conj().T - a)], fields=fields,
                    c_ops=_sites(n, 0, GAMMA)[:4] + [0.1 * a], rho0=_pure(rng, n), e_ops=e_ops, dt=0.02)
    if kind == "two_time":
        n = case["n"]
        H = np.zeros((n, n), dtype=np.complex128)
        H[1:, 1:] = _chain_h(rng.normal(0.0, 0.05, n - 1), -0.08)
        mu = np.zeros((n, n), dtype=np.complex128)
        mu[1:, 0] = mu[0, 1:] = rng.uniform(-1, 1, n - 1)
        return dict(H=H, c_ops=_sites(n, 1, GAMMA), rho0=_pure(rng, n), ops=[mu, mu, mu], dt=0.05)
    if kind in ("redfield", "liouville"):
        n = case["n"]
        K = case.get("baths", 1)
        return dict(H=_herm(rng, n), a_ops=[_herm(rng, n) for _ in range(K)],
                    spectra=[_ohmic(0.02 + 0.01 * k, 1.0 + 0.5 * k) for k in range(K)], rho0=_pure(rng, n),
                    e_ops=[np.diag(np.eye(n)[i]).astype(np.complex128) for i in range(min(n, 3))], dt=0.05)
    if kind == "ragged":
        ns = np.random.default_rng(case["sizes"]).choice(np.asarray(RAGGED_SIZES), size=case["count"])
        if case["sizes"] % 2 == 0:                      # odd sizes as well as whole tiles
            ns = ns - np.random.default_rng(case["sizes"] + 1).integers(0, 16, case["count"])
        inst = []
        for n in ns:
            n = max(2, int(n))
            Ls = [rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) for _ in range(case["jumps"])]
            inst.append(dict(H=_herm(rng, n) / 2.0, c_ops=[L * (0.1 / np.linalg.norm(L)) for L in Ls],
                             dephasing=GAMMA, rho0=_pure(rng, n)))
        return dict(instances=inst, dt=0.02)
    dev = torch.device("cuda", torch.cuda.current_device())
    if kind == "gradient":
        B, ns = case["batch"], case["n"] - 1
        up = lambda x: torch.as_tensor(x, device=dev)
        mu = rng.standard_normal(ns)
        return dict(eps=up(rng.normal(0.0, 0.05, (B, ns))), J=up(rng.uniform(-0.12, -0.08, (B, ns - 1))),
                    gamma=torch.tensor(0.02, dtype=torch.float64, device=dev), mu=up(mu / np.linalg.norm(mu) * 8.0),
                    target=up(rng.normal(0.0, 1.0, (B, case["steps"])) + 1j * rng.normal(0.0, 1.0, (B, case["steps"]))),
                    dt=0.05)
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    normal = lambda *shape: torch.randn(*shape, dtype=torch.float64, device=dev, generator=g)
    n = case["n"]
    if kind == "absorption":
        R, ns = case["sets"], n - 1
        side = max(1, int(math.isqrt(ns)))               # sites row by row on a lattice of this width
        H = torch.zeros((R, n, n), dtype=torch.complex128, device=dev)
        i = torch.arange(1, n, device=dev)
        H[:, i, i] = (0.05 * normal(R, ns)).to(torch.complex128)
        for p, q in [(s, s + 1) for s in range(ns - 1) if (s + 1) % side] + [(s, s + side) for s in range(ns - side)]:
            H[:, p + 1, q + 1] = H[:, q + 1, p + 1] = -0.08
        mu_v = normal(R, case["group"], ns)
        mu_v = mu_v / mu_v.norm(dim=1, keepdim=True)
        mu = torch.zeros((R * case["group"], n, n), dtype=torch.complex128, device=dev)
        mu[:, 1:, 0] = mu_v.reshape(-1, ns).to(torch.complex128)
        mu[:, 0, 1:] = mu_v.reshape(-1, ns).to(torch.complex128)
        x0 = torch.zeros_like(mu)
        x0[:, :, 0] = mu[:, :, 0]
        return dict(H=H, c_ops=_sites(n, 1, GAMMA), mu=mu, x0=x0, dt=0.05)
    B = case["batch"]
    x = torch.complex(normal(B, n, n), normal(B, n, n))
    H = ((x + x.conj().transpose(-1, -2)) / (4.0 * math.sqrt(n))).resolve_conj().contiguous()
    psi = torch.complex(normal(B, n), normal(B, n))
    psi = psi / psi.norm(dim=1, keepdim=True)
    rho0 = psi.unsqueeze(2) * psi.conj().unsqueeze(1)
    if kind == "ensemble":
        e_ops = [np.diag(np.eye(n)[i]).astype(np.complex128) for i in range(case["observables"])]
        return dict(H=H, c_ops=_sites(n, 0, GAMMA), rho0=rho0.contiguous(), e_ops=e_ops, dt=0.05)
    rho0 = 0.5 * rho0 + 0.5 * torch.eye(n, dtype=torch.complex128, device=dev) / n
    Ls = []
    for _ in range(case["jumps"]):
        L = torch.complex(normal(B, n, n), normal(B, n, n))
        Ls.append(L * (0.05 / L.abs().pow(2).sum(dim=(1, 2), keepdim=True).sqrt()))
    return dict(H=H, c_ops=Ls, rho0=rho0.contiguous(), e_ops=None, dt=0.01)


# ---------------------------------------------------------------------------- the passes
def prepare(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    s["case"] = case
    if kind in ("chain", "two_time"):
        from lime_amd.oqs import Lindblad_solver
        s["solver"] = Lindblad_solver(s["H"], s["c_ops"])
    elif kind == "driven":
        from lime_amd.oqs import Lindblad_solver
        s["solver"] = Lindblad_solver([s["H0"]] + [[h, f] for h, f in zip(s["drives"], s["fields"])], s["c_ops"])
    elif kind in ("redfield", "liouville"):
        from lime_amd.oqs import Redfield_solver
        s["solver"] = Redfield_solver(s["H"], c_ops=s["a_ops"], spectra=s["spectra"])
        s["R"], s["evecs"] = s["solver"].redfield_tensor()
    elif kind == "ragged":
        from lime_amd.ragged import RaggedLindblad
        s["batch"] = RaggedLindblad(s["instances"])
        s["rho0"] = s["batch"].rho.clone()
        del s["instances"]
    elif kind != "gradient":
        from lime_amd.propagator import LindbladPropagator
        s["prop"] = LindbladPropagator(s["H"], s["c_ops"], group=case.get("group", 1), precision=case["precision"])
        del s["H"], s["c_ops"]
    return s


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "chain":
        r = s["solver"].evolve(s["rho0"], s["dt"], case["steps"], e_ops=s["e_ops"], nout=case["nout"])
        return r.observables, np.asarray(r.rholist)
    if kind == "driven":
        r = s["solver"].evolve(s["rho0"], s["dt"], case["steps"], e_ops=s["e_ops"])
        return r.observables, np.asarray(r.rholist)
    if kind == "two_time":
        return s["solver"].correlation_3op_2t(s["rho0"], s["ops"], s["dt"], case["steps"], case["tau_steps"])
    if kind == "redfield":
        r = s["solver"].evolve(s["rho0"], s["dt"], case["steps"], e_ops=s["e_ops"])
        return r.observables, np.asarray(r.rholist)
    if kind == "liouville":
        from lime_amd.oqs import _redfield
        r = _redfield(s["R"], s["rho0"], evecs=s["evecs"], Nt=case["steps"], dt=s["dt"], e_ops=s["e_ops"])
        return r.observables, np.asarray(r.rholist)
    if kind == "absorption":
        E = s["mu"].reshape(-1, 1, case["n"], case["n"])
        rho, obs, _ = s["prop"].run(s["x0"], s["dt"], case["steps"], e_ops=E)
        return rho, obs
    if kind == "ensemble":
        rho, obs, _ = s["prop"].run(s["rho0"], s["dt"], case["steps"], e_ops=s["e_ops"], renorm=True)
        return rho, obs
    if kind == "dense":
        return s["prop"].run(s["rho0"], s["dt"], case["steps"])[0]
    if kind == "ragged":
        s["batch"].rho.copy_(s["rho0"])
        s["batch"].run(s["dt"], case["steps"], chunk=10)
        return s["batch"].rho
    from lime_amd.adjoint import ChainAbsorption, spectrum_loss
    eps, J, gamma = (s[k].detach().clone().requires_grad_(True) for k in ("eps", "J", "gamma"))
    C = ChainAbsorption.apply(eps, J, gamma, s["mu"], s["dt"], case["steps"])
    spectrum_loss(C, s["target"], s["dt"]).sum().backward()
    return C, eps.grad, J.grad, gamma.grad


# ---------------------------------------------------------------------------- its size
def _sizes(case):
    ns = np.random.default_rng(case["sizes"]).choice(np.asarray(RAGGED_SIZES), size=case["count"])
    if case["sizes"] % 2 == 0:
        ns = ns - np.random.default_rng(case["sizes"] + 1).integers(0, 16, case["count"])
    return np.maximum(ns, 2).astype(np.float64)


def work(case):
    """One generator application takes 2 complex products of n^3 (8 real operations each), a
    sandwich term 2 more, a step 4 applications; Liouville space takes one matrix-vector
    product of n^2 x n^2 per stage.  Operators are counted in the arithmetic's operand size
    (8 bytes an element, 16 in FP64), states and records in 16 bytes."""
    kind, steps = case["kind"], case["steps"]
    n = float(case.get("n", 0))
    nn = n * n
    if kind == "chain":
        rec = steps // case["nout"]
        return dict(bytes=16 * (nn * (2 + rec) + nn) + 16 * rec * min(n, 8), flops=64 * n ** 3 * steps)
    if kind == "driven":
        return dict(bytes=16 * (nn * (4 + 5) + steps * (nn + 2)), flops=64 * n ** 3 * 2 * steps)
    if kind == "two_time":
        t, u = steps, case["tau_steps"]
        return dict(bytes=16 * (5 * nn + t * u), flops=64 * n ** 3 * (t + t * u))
    if kind == "redfield":
        return dict(bytes=16 * (nn * (2 + 2 * case["baths"]) + steps * (nn + 3)),
                    flops=64 * n ** 3 * (1 + 2 * case["baths"]) * steps)
    if kind == "liouville":
        return dict(bytes=16 * (nn * nn + steps * (nn + 3)), flops=32 * nn * nn * steps)
    if kind == "absorption":
        B = case["sets"] * case["group"]
        return dict(bytes=B * nn * (16 * 3) + case["sets"] * nn * 8 * 2 + 16 * B * steps, flops=64 * n ** 3 * B * steps)
    if kind == "ensemble":
        op = 16 if case["precision"] == "fp64" else 8
        return dict(bytes=case["batch"] * (nn * (32 + 2 * op) + 16 * steps * case["observables"]),
                    flops=64 * n ** 3 * case["batch"] * steps)
    if kind == "dense":
        op = 16 if case["precision"] == "fp64" else 8
        return dict(bytes=case["batch"] * nn * (32 + op * (1 + case["jumps"])),
                    flops=64 * n ** 3 * (1 + case["jumps"]) * case["batch"] * steps)
    if kind == "ragged":
        ns = _sizes(case)
        return dict(bytes=float((ns ** 2).sum()) * (32 + 8 * (2 + case["jumps"])),
                    flops=64 * float((ns ** 3).sum()) * (1 + case["jumps"]) * steps)
    # forward, recomputation of the stage operands and four adjoint applications per step
    return dict(bytes=case["batch"] * (nn * 8 * 2 + 16 * steps * 2 + 8 * 4 * n), flops=64 * n ** 3 * case["batch"] * steps * 3)


# ---------------------------------------------------------------------------- 64 bits
def _dag(x):
    return x.conj().transpose(-1, -2).resolve_conj().contiguous()


def _field(heff, d=None, Ls=(), Rs=None):
    """f(X) = -i (H X - X H^dag) + D o X + sum L X R^dag in complex128 (batched)."""
    hd = _dag(heff)
    pairs = [(L, _dag(R)) for L, R in zip(Ls, Ls if Rs is None else Rs)]

    def f(X):
        v = -1j * (torch.matmul(heff, X) - torch.matmul(X, hd))
        if d is not None:
            v = v + d * X
        for L, rd in pairs:
            v = v + torch.matmul(torch.matmul(L, X), rd)
        return v
    return f


def _fold(H, c_ops):
    """(H_eff, D, dense jump operators), all complex128 on the GPU."""
    G = torch.zeros_like(H)
    D, dense = None, []
    for c in c_ops:
        L = torch.as_tensor(c, dtype=torch.complex128, device=H.device)
        l = torch.diagonal(L, dim1=-2, dim2=-1)
        if torch.equal(L, torch.diag_embed(l)):
            G = G + torch.diag_embed((l.abs() ** 2).to(torch.complex128))
            t = l.unsqueeze(-1) * l.conj().unsqueeze(-2)
            D = t if D is None else D + t
        else:
            G = G + torch.matmul(_dag(L), L)
            dense.append(L)
    return H - 0.5j * G, D, dense


def _rk4(f, X, dt):
    a = f(X)
    b = f(X + 0.5 * dt * a)
    c = f(X + 0.5 * dt * b)
    return X + (dt / 6.0) * (a + 2 * b + 2 * c + f(X + dt * c))


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    dt, steps = s["dt"], case["steps"]
    dev = torch.device("cuda", torch.cuda.current_device())
    up = lambda x: torch.as_tensor(x, dtype=torch.complex128, device=dev)
    down = lambda x: x.cpu().numpy()

    def series(f, X, E, nout=1, back=None):
        obs, states = [], []
        for k in range(steps):
            X = _rk4(f, X, dt)
            if (k + 1) % nout == 0:
                obs.append((E * X.transpose(-1, -2)).sum(dim=(-1, -2)))
                states.append(X if back is None else back(X))
        return down(torch.stack(obs)), down(torch.stack(states))

    if kind == "chain":
        he, D, Ls = _fold(up(s["H"]), s["c_ops"])
        return series(_field(he, D, Ls), up(s["rho0"]), up(np.stack(s["e_ops"])), case["nout"])
    if kind == "driven":
        he, D, Ls = _fold(up(s["H0"]), s["c_ops"])
        Hd = [up(h) for h in s["drives"]]
        E, X, t = up(np.stack(s["e_ops"])), up(s["rho0"]), 0.0
        obs, states = [], []
        for _ in range(steps):
            t += dt
            h = he
            for f, d in zip(s["fields"], Hd):
                h = h - f(t) * d
            X = _rk4(_field(h, D, Ls), X, dt)
            obs.append((E * X.transpose(-1, -2)).sum(dim=(-1, -2)))
            states.append(X)
        return down(torch.stack(obs)), down(torch.stack(states))
    if kind == "two_time":
        f = _field(*_fold(up(s["H"]), s["c_ops"]))
        A, Bo, Co = (up(o) for o in s["ops"])
        X, grid = up(s["rho0"]), []
        for _ in range(steps):
            X = _rk4(f, X, dt)
            grid.append(torch.matmul(torch.matmul(Co, X), A))
        X, out = torch.stack(grid), []
        for _ in range(case["tau_steps"]):
            X = _rk4(f, X, dt)
            out.append((Bo * X.transpose(-1, -2)).sum(dim=(-1, -2)))
        return down(torch.stack(out, dim=1))
    if kind in ("redfield", "liouville"):
        E, V = np.linalg.eigh(s["H"])
        W = E[:, None] - E[None, :]
        A = [V.conj().T @ a @ V for a in s["a_ops"]]
        Lam = [S(-W) * a for S, a in zip(s["spectra"], A)]
        G = np.diag(E).astype(np.complex128) - 1j * sum(a @ l for a, l in zip(A, Lam))
        f = _field(up(G), None, [up(x) for x in A + Lam], [up(x) for x in Lam + A])
        Vt = up(V)
        Vd = _dag(Vt)
        e = up(np.stack([V.conj().T @ o @ V for o in s["e_ops"]]))
        return series(f, up(V.conj().T @ s["rho0"] @ V), e, back=lambda X: torch.matmul(torch.matmul(Vt, X), Vd))
    if kind == "ragged":
        # instances of one size together, put back in the batch's order
        out = [None] * len(s["instances"])
        by_n = {}
        for i, c in enumerate(s["instances"]):
            by_n.setdefault(c["H"].shape[0], []).append(i)
        for n, idx in by_n.items():
            inst = [s["instances"][i] for i in idx]
            Ls = [up(np.stack([c["c_ops"][k] for c in inst])) for k in range(case["jumps"])]
            he, _, dense = _fold(up(np.stack([c["H"] for c in inst])), Ls)
            eye = torch.eye(n, dtype=torch.complex128, device=dev)
            f = _field(he - 0.5j * GAMMA * eye, GAMMA * eye, dense)
            X = up(np.stack([c["rho0"] for c in inst]))
            for _ in range(steps):
                X = _rk4(f, X, dt)
            for j, i in enumerate(idx):
                out[i] = X[j].reshape(-1)
        return torch.cat(out)
    if kind == "gradient":
        return _exact_gradient(s, case)
    he, D, Ls = _fold(s["H"], s["c_ops"])
    g = case.get("group", 1)
    if g > 1:
        he, D = he.repeat_interleave(g, 0), D if D.dim() == 2 else D.repeat_interleave(g, 0)
    f = _field(he, D, Ls)
    X = s["x0"] if kind == "absorption" else s["rho0"]
    E = None
    if kind == "absorption":
        E = s["mu"].unsqueeze(1)
    elif s["e_ops"]:
        E = up(np.stack(s["e_ops"])).unsqueeze(0)
    obs = []
    for _ in range(steps):
        X = _rk4(f, X, dt)
        if kind == "ensemble":
            X = X / torch.diagonal(X, dim1=-2, dim2=-1).real.sum(-1).reshape(-1, 1, 1)
        if E is not None:
            obs.append((E * X.transpose(-1, -2).unsqueeze(1)).sum(dim=(-1, -2)))
    return X if E is None else (X, torch.stack(obs, dim=1))


def _exact_gradient(s, case):
    """Automatic differentiation of the unrolled RK4 steps, each one recomputed in the backward pass."""
    from torch.utils.checkpoint import checkpoint
    n, dt = case["n"], s["dt"]
    eps, J, gamma = (s[k].detach().clone().requires_grad_(True) for k in ("eps", "J", "gamma"))
    B, dev = eps.shape[0], eps.device
    mu = torch.zeros((n, n), dtype=torch.complex128, device=dev)
    mu[1:, 0] = mu[0, 1:] = s["mu"].to(torch.complex128)
    site = torch.zeros(n, dtype=torch.float64, device=dev)
    site[1:] = 1.0
    pad = torch.nn.functional.pad

    def step(X, eps, J, gamma):
        H = torch.diag_embed(pad(eps, (1, 0))) + torch.diag_embed(pad(J, (1, 0)), offset=1) + torch.diag_embed(pad(J, (1, 0)), offset=-1)
        D = torch.diag_embed(gamma * site)
        he = torch.complex(H, -0.5 * D.expand_as(H))
        hd = he.conj().transpose(-1, -2).resolve_conj().contiguous()
        f = lambda x: -1j * (torch.matmul(he, x) - torch.matmul(x, hd)) + D * x
        return _rk4(f, X, dt)

    X = torch.zeros((B, n, n), dtype=torch.complex128, device=dev)
    X[:, :, 0] = mu[:, 0]
    C = []
    for _ in range(case["steps"]):
        X = checkpoint(step, X, eps, J, gamma, use_reentrant=False)
        C.append((mu * X.transpose(-1, -2)).sum(dim=(-1, -2)))
    C = torch.stack(C, dim=1)
    S, St = (torch.fft.fft(x, dim=-1) * dt for x in (C, s["target"]))
    ((S.real - St.real) ** 2).sum().backward()
    return C.detach(), eps.grad, J.grad, gamma.grad
