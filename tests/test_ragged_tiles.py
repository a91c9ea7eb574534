"""The per-phase launches of a ragged batch: their workgroup lists (on the CPU) and their
results against the persistent launch (on the GPU)."""
import numpy as np
import pytest

from lime_amd.ragged import XCDS, tile_lists

SIZES = (1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 129)


@pytest.mark.parametrize("edge", [32, 64])
@pytest.mark.parametrize("sizes,kd", [(SIZES, [k % 3 for k in range(len(SIZES))]), ((256,), (0,)), ((40, 40), (2, 0))])
def test_lists_hold_every_tile_once_and_keep_an_instance_on_one_xcd(sizes, kd, edge):
    cost = [float(n) ** 3 * (1 + k) for n, k in zip(sizes, kd)]
    for which, lst in zip(("stage", "left"), tile_lists(sizes, kd, cost, edge)):
        assert lst.dtype == np.int32 and lst.shape[1] == 2 and len(lst) % XCDS == 0
        seen = {}
        for b, (i, item) in enumerate(lst.tolist()):
            if i < 0:
                continue
            seen.setdefault(i, []).append((item, b % XCDS))
        for i, (n, k) in enumerate(zip(sizes, kd)):
            tiles = (-(-n // edge)) ** 2
            got = seen.get(i, [])
            assert sorted(t for t, _ in got) == list(range(tiles * (1 if which == "stage" else k)))
            assert len({x for _, x in got}) <= 1


def _instances(seed):
    rng = np.random.default_rng(seed)
    c = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    out = []
    for k, n in enumerate(SIZES):
        x, psi = c(n, n), c(n)
        Ls = [0.1 * c(n, n) / n for _ in range(k % 3)]
        out.append(dict(H=(x + x.conj().T) / (4 * np.sqrt(n)), c_ops=Ls, dephasing=0.01 if k % 2 else None,
                        rho0=np.outer(psi, psi.conj()) / np.vdot(psi, psi).real))
    return out


@pytest.mark.gpu
def test_per_phase_launches_equal_the_persistent_launch_eager_and_replayed():
    torch = pytest.importorskip("torch")
    from lime_amd.ragged import RaggedLindblad
    inst = _instances(5)
    ref = RaggedLindblad(inst, tune=False)
    for v in range(ref.variants(), ref.launches()):
        rb = RaggedLindblad(inst, tune=False)
        rb.variant = v
        rb.capture(0.02, 3)
        want = RaggedLindblad(inst, tune=False)
        for _ in range(2):
            rb.graph.replay()
            want.step(0.02, 3)
            torch.cuda.synchronize()
            assert torch.equal(rb.rho, want.rho), v
        rb.step(0.02, 2)
        want.step(0.02, 2)
        assert torch.equal(rb.rho, want.rho), v
    assert RaggedLindblad(inst, tune=False, max_groups=1).launches() == ref.variants()


@pytest.mark.gpu
def test_a_run_of_many_steps_captures_a_bounded_graph():
    torch = pytest.importorskip("torch")
    from lime_amd.ragged import GRAPH_STEPS, RaggedLindblad
    inst = _instances(6)[2:7]
    steps = 2 * GRAPH_STEPS + 5
    for v in (5, 6):
        want, rb = (RaggedLindblad(inst, tune=False) for _ in range(2))
        want.run(0.005, steps)
        assert want.graph_steps == steps               # the persistent launch is one node
        rb.variant = v
        assert rb.variants() <= v < rb.launches()
        rb.run(0.005, steps)
        assert rb.graph_steps == GRAPH_STEPS
        assert torch.equal(rb.rho, want.rho)
        rb.run(0.005, 3, chunk=3)
        want.run(0.005, 3)
        assert rb.graph_steps == 3 and torch.equal(rb.rho, want.rho)


def test_a_run_of_no_steps_ends():
    from lime_amd.ragged import RaggedClasses, RaggedLindblad
    for cls in (RaggedLindblad, RaggedClasses):
        assert object.__new__(cls).run(0.01, 0) is None
