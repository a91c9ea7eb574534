"""Ragged batches: many independent Lindblad systems of uneven dimension.

lime propagates one system at a time (oqs.py:1590-1688).  ``RaggedLindblad`` takes a list
of instances of different n and advances all of them together.  The instances are packed
into three pools (complex64 operators, complex128 states, complex64 per-stage workspace).
Two organisations step them, with the same results bit for bit:

* one persistent launch (``lime_lindblad_rk4_ragged``): a grid of workgroups drains the
  instances, ordered by cost n^3 (1 + K_d), through an atomic queue, each instance on one
  workgroup for every step of the call;
* one launch per phase of a stage (``lime_lindblad_rk4_ragged_tiles``): every tile of every
  instance is a workgroup of its own, so few or large instances fill the GPU too.

The autotuner (``lime_amd.autotune.tune_ragged``) times both, with their launch shapes, on
the batch; ``capture``/``run`` put the launches in a hipGraph (torch.cuda.CUDAGraph) and
replay it.

``RaggedClasses`` is the earlier organisation, kept as the comparison point: size classes,
one operator batch each on the per-class fused kernels, all captured into one graph.

An instance is a dict with ``H`` (n, n), ``rho0`` (n, n), optional ``c_ops`` (list of
(n, n) jump operators) and optional ``dephasing`` (scalar or length-n rates gamma_i of
L_i = sqrt(gamma_i)|i><i|, given compactly instead of n dense matrices).
"""
import ctypes

import numpy as np
import torch

from . import autotune
from .propagator import LindbladPropagator, device


XCDS = 8                 # accelerator dies of the GPU, each with its own L2
TILE_EDGES = (32, 64)    # output tiles of the per-phase launches
# Steps of a captured graph of per-phase launches.  A graph of all steps grows with them (8 nodes each) and
# its capture is time: 8 systems of n = 17 .. 64, 4000 steps, first run / again 315 / 259 ms, by 32 264 / 251.
GRAPH_STEPS = 64


def fold_host(inst):
    """(H_eff, D, dense L list) of one instance, complex128 NumPy."""
    H = np.asarray(inst["H"], dtype=np.complex128)
    n = H.shape[0]
    gam_d = np.zeros(n)
    D = np.zeros((n, n), dtype=np.complex128)
    G = np.zeros((n, n), dtype=np.complex128)
    if inst.get("dephasing") is not None:
        g = np.broadcast_to(np.asarray(inst["dephasing"], dtype=np.float64), (n,))
        gam_d += g
        D[np.arange(n), np.arange(n)] += g
    dense = []
    for L in inst.get("c_ops") or []:
        L = np.asarray(L, dtype=np.complex128)
        d = np.diagonal(L)
        if np.count_nonzero(L) == np.count_nonzero(d):            # diagonal jump operator
            gam_d += np.abs(d) ** 2
            D += np.outer(d, d.conj())
        else:
            G += L.conj().T @ L
            dense.append(L)
    G[np.arange(n), np.arange(n)] += gam_d
    return H - 0.5j * G, D, dense


def tile_lists(sizes, kd, cost, edge):
    """(stage, left) workgroup lists of ``lime_lindblad_rk4_ragged_tiles``: int32 (count, 2)
    arrays of (instance, tile) and (instance, k * tiles + tile).

    Instances are dealt to the 8 XCDs, the most expensive first, each to the XCD with the
    least work so far; list entry b belongs to XCD b % 8, so an instance's tiles share one
    L2 and every XCD starts with its largest instances.  (-1, -1) pads the shorter lists."""
    tiles = ((np.asarray(sizes, dtype=np.int64) + edge - 1) // edge) ** 2
    load = np.zeros(XCDS)
    mine = [[] for _ in range(XCDS)]
    for i in np.argsort(-np.asarray(cost), kind="stable"):
        x = int(np.argmin(load))
        load[x] += cost[i]
        mine[x].append(i)

    def interleave(items):
        per = []
        for ids in mine:
            ids = np.asarray(ids, dtype=np.int64)
            c = items[ids]
            e = np.empty((int(c.sum()), 2), dtype=np.int32)
            e[:, 0] = np.repeat(ids, c)
            e[:, 1] = np.arange(len(e)) - np.repeat(np.cumsum(c) - c, c)
            per.append(e)
        out = np.full((max(len(e) for e in per), XCDS, 2), -1, dtype=np.int32)
        for x, e in enumerate(per):
            out[:len(e), x] = e
        return out.reshape(-1, 2)

    return interleave(tiles), interleave(tiles * np.asarray(kd, dtype=np.int64))


class RaggedLindblad:
    """A list of instances of uneven n advanced together (FP32 MFMA, FP64 state): one
    persistent launch, or one launch per phase of a stage, whichever the autotuner measured
    faster on the batch (the same results, bit for bit)."""

    def __init__(self, instances, tune=True, dt_tune=0.01, verbose=False, max_groups=0):
        from . import _lib
        self.dev = device()
        self._lib = _lib.load()
        self.count = len(instances)
        self.sizes = np.array([np.asarray(i["H"]).shape[0] for i in instances])
        rec = np.zeros(self.count, dtype=[("n", "<i4"), ("n_dense", "<i4"), ("heff", "<i8"),
                                          ("dmat", "<i8"), ("lops", "<i8"), ("rho", "<i8"),
                                          ("work", "<i8")])
        assert rec.dtype.itemsize == ctypes.sizeof(_lib.RaggedInstance)
        ops, rhos = [], []
        o_ops = o_rho = o_work = 0
        cost = np.zeros(self.count)
        self.kd = np.zeros(self.count, dtype=np.int64)
        for i, inst in enumerate(instances):
            heff, dmat, dense = fold_host(inst)
            n, kd = heff.shape[0], len(dense)
            r0 = np.asarray(inst["rho0"], dtype=np.complex128)
            if r0.shape != (n, n):
                raise ValueError(f"instance {i}: rho0 has shape {r0.shape}, H is {n} x {n}")
            rec[i] = (n, kd, o_ops, -1, -1, o_rho, o_work)
            ops.append(heff.ravel())
            o_ops += n * n
            if np.any(dmat != 0):
                rec[i]["dmat"] = o_ops
                ops.append(dmat.ravel())
                o_ops += n * n
            if kd:
                rec[i]["lops"] = o_ops
                for L in dense:
                    ops.append(L.ravel())
                o_ops += kd * n * n
            rhos.append(r0.ravel())
            o_rho += n * n
            o_work += (3 + kd) * n * n
            cost[i] = float(n) ** 3 * (1 + kd)
            self.kd[i] = kd
        self.work_units = float(cost.sum())
        self.rec = rec
        self.ops = torch.as_tensor(np.concatenate(ops).astype(np.complex64), device=self.dev)
        self.rho = torch.as_tensor(np.concatenate(rhos), device=self.dev).contiguous()
        self.work = torch.empty(o_work, dtype=torch.complex64, device=self.dev)
        self.inst = torch.as_tensor(rec.view(np.uint8), device=self.dev)
        order = np.argsort(-cost, kind="stable").astype(np.int32)
        self.order = torch.as_tensor(order, device=self.dev)
        self.queue = torch.zeros(2, dtype=torch.int32, device=self.dev)
        self.max_groups = int(max_groups)
        self.cost = cost
        self._lists = {}
        self.variant = 0
        self.graph = None
        if tune:
            from . import autotune
            autotune.tune_ragged(self, dt_tune, verbose=verbose)
        if self.variant >= self.variants():       # a choice from the cache was not timed here: a first step
            self._tile_lists(TILE_EDGES[self.variant - self.variants()])     # may be one that is captured

    def variants(self):
        """Launch shapes of the persistent kernel."""
        return int(self._lib.lime_ragged_variants())

    def launches(self):
        """Values of ``variant`` the autotuner times: the persistent launch shapes, then one
        launch per phase of a stage with 32 x 32 and with 64 x 64 tiles (not with a cap on
        the persistent workgroups)."""
        return self.variants() + (0 if self.max_groups else len(TILE_EDGES))

    def _tile_lists(self, edge):
        """Device lists of ``lime_lindblad_rk4_ragged_tiles`` for a tile edge (made once)."""
        if edge not in self._lists:
            from . import _lib
            stage, left = (torch.as_tensor(x, device=self.dev) for x in tile_lists(self.sizes, self.kd, self.cost, edge))
            t = _lib.RaggedTiles()
            t.tile, t.stage_count, t.stage = edge, stage.shape[0], stage.data_ptr()
            t.left_count, t.left = left.shape[0], left.data_ptr()
            self._lists[edge] = (t, stage, left)
        return self._lists[edge][0]

    @property
    def flops_per_step(self):
        """Canonical algorithmic FLOPs of one RK4 step of the whole batch: 64 n^3 (1 + K_d)."""
        return 64.0 * self.work_units

    def step(self, dt, nsteps, stream=None):
        """Advance every instance by ``nsteps`` RK4 steps (async): one persistent launch
        (``variant`` < ``variants()``), or one launch per phase of each stage."""
        from . import _lib
        r = _lib.RaggedBatch()
        tiled = self.variant - self.variants()
        r.count, r.max_groups = self.count, self.max_groups
        r.inst, r.order = self.inst.data_ptr(), self.order.data_ptr()
        r.ops, r.rho, r.work, r.queue = (self.ops.data_ptr(), self.rho.data_ptr(),
                                         self.work.data_ptr(), self.queue.data_ptr())
        p = _lib.StepParams()
        p.dt, p.nsteps = float(dt), int(nsteps)
        s = stream if stream is not None else torch.cuda.current_stream(self.dev)
        if 0 <= tiled < self.launches() - self.variants():     # what is not offered the library refuses
            tiles = self._tile_lists(TILE_EDGES[tiled])
            _lib.check(self._lib.lime_lindblad_rk4_ragged_tiles(ctypes.byref(r), ctypes.byref(tiles),
                                                                ctypes.byref(p), ctypes.c_void_p(s.cuda_stream)))
            return
        r.variant = self.variant
        _lib.check(self._lib.lime_lindblad_rk4_ragged(ctypes.byref(r), ctypes.byref(p),
                                                      ctypes.c_void_p(s.cuda_stream)))

    step_eager = step

    def capture(self, dt, nsteps):
        """Capture one launch of ``nsteps`` steps of every instance into a graph."""
        saved = self.rho.clone()
        self.step(dt, 1)                          # kernel loaded, attributes set
        torch.cuda.synchronize(self.dev)
        self.rho.copy_(saved)
        torch.cuda.synchronize(self.dev)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            self.step(dt, nsteps)
        self.graph, self.graph_steps, self.graph_dt = g, nsteps, dt
        return g

    def run(self, dt, nsteps, chunk=None):
        """Advance every instance by ``nsteps`` steps by replaying the captured launch(es): all steps in
        one replay, or with a launch per phase (8 a step) ``GRAPH_STEPS`` of them, unless ``chunk`` says
        how many."""
        if nsteps < 1:
            return
        whole = nsteps if self.variant < self.variants() else min(nsteps, GRAPH_STEPS)
        chunk = int(chunk or whole)
        if self.graph is None or self.graph_steps != chunk or self.graph_dt != dt:
            self.capture(dt, chunk)
        done = 0
        while done + chunk <= nsteps:
            self.graph.replay()
            done += chunk
        if done < nsteps:
            self.step(dt, nsteps - done)

    def states(self):
        """Current operators as a list in the original instance order (NumPy)."""
        r = self.rho.cpu().numpy()
        return [r[o:o + n * n].reshape(n, n) for n, o in zip(self.rec["n"], self.rec["rho"])]


class RaggedClasses:
    """Size classes on the per-class fused kernels, all captured into one graph."""

    def __init__(self, instances, precision="fp32", tune=True, dt_tune=0.01, verbose=False):
        self.dev = device()
        self.precision = precision
        self.sizes = np.array([np.asarray(i["H"]).shape[0] for i in instances])
        by_n = {}
        for idx, inst in enumerate(instances):
            by_n.setdefault(int(self.sizes[idx]), []).append(idx)
        self.classes = []
        for n, idxs in sorted(by_n.items(), key=lambda kv: -(kv[0] ** 3) * len(kv[1])):
            folded = [fold_host(instances[i]) for i in idxs]
            kd = {len(f[2]) for f in folded}
            if len(kd) != 1:
                raise ValueError(f"instances of n = {n} differ in their number of dense jump operators")
            kd = kd.pop()
            heff = np.stack([f[0] for f in folded])
            dmat = np.stack([f[1] for f in folded])
            lops = np.stack([np.stack(f[2]) for f in folded]) if kd else None
            prop = LindbladPropagator.from_folded(heff, dmat, lops, precision=precision)
            rho = torch.as_tensor(np.stack([np.asarray(instances[i]["rho0"], dtype=np.complex128)
                                            for i in idxs]), device=self.dev).contiguous()
            self.classes.append({"n": n, "idx": idxs, "prop": prop, "rho": rho,
                                 "cost": float(n) ** 3 * (1 + kd) * len(idxs)})
        if tune:
            for c in self.classes:
                autotune.tune(c["prop"], c["rho"], dt_tune, verbose=verbose)
        self.graph = None
        self.graph_steps = None

    @property
    def flops_per_step(self):
        """Canonical algorithmic FLOPs of one RK4 step of the whole batch: 64 n^3 (1 + K_d)."""
        return sum(64.0 * c["n"] ** 3 * (1 + c["prop"].n_dense) * len(c["idx"]) for c in self.classes)

    def _launch_all(self, dt, nsteps):
        main = torch.cuda.current_stream(self.dev)
        for c in self.classes:
            s = c.setdefault("stream", torch.cuda.Stream(self.dev))
            s.wait_stream(main)
            with torch.cuda.stream(s):
                c["prop"].step(c["rho"], dt, nsteps, stream=s)
            main.wait_stream(s)

    def step_eager(self, dt, nsteps):
        self._launch_all(dt, nsteps)

    def capture(self, dt, nsteps):
        """Capture ``nsteps`` RK4 steps of every class into one graph."""
        saved = [c["rho"].clone() for c in self.classes]
        self._launch_all(dt, 1)                  # workspaces and kernel attributes exist
        torch.cuda.synchronize(self.dev)
        for c, r in zip(self.classes, saved):    # the warm-up step is undone
            c["rho"].copy_(r)
        torch.cuda.synchronize(self.dev)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            self._launch_all(dt, nsteps)
        self.graph, self.graph_steps, self.graph_dt = g, nsteps, dt
        return g

    def run(self, dt, nsteps, chunk=None):
        """Advance every instance by ``nsteps`` steps by replaying the captured graph."""
        if nsteps < 1:
            return
        chunk = int(chunk or nsteps)
        if self.graph is None or self.graph_steps != chunk or self.graph_dt != dt:
            self.capture(dt, chunk)
        done = 0
        while done + chunk <= nsteps:
            self.graph.replay()
            done += chunk
        if done < nsteps:
            self.step_eager(dt, nsteps - done)

    def states(self):
        """Current operators as a list in the original instance order (NumPy)."""
        out = [None] * len(self.sizes)
        for c in self.classes:
            r = c["rho"].cpu().numpy()
            for k, i in enumerate(c["idx"]):
                out[i] = r[k]
        return out
