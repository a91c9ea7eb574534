"""The cached launch choices of ragged batches: one per batch shape and cap on workgroups."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")


class Timed(Exception):
    pass


class _States:
    def clone(self):                                   # the tuner saves the states before it times
        raise Timed


class _Batch:
    def __init__(self, sizes, kd, max_groups=0):
        self.sizes, self.kd, self.max_groups = np.array(sizes), np.array(kd, dtype=np.int64), max_groups
        self.count, self.variant, self.rho = len(sizes), 0, _States()
        self.work_units = float((self.sizes.astype(float) ** 3 * (1 + self.kd)).sum())

    def launches(self):
        return 5 if self.max_groups else 7


@pytest.fixture
def cache(monkeypatch):
    from lime_amd import autotune
    entries = {}
    monkeypatch.setattr(autotune, "_load", lambda: entries)
    monkeypatch.setattr(autotune, "_version", lambda: "v")
    return entries


def _remember(entries, batch, variant):
    """What the tuner stores for a batch: under the key that it looks up."""
    from lime_amd import autotune
    seen = []

    class Probe(dict):
        def __contains__(self, key):
            seen.append(key)
            return False
    load, autotune._load = autotune._load, lambda: Probe()
    try:
        with pytest.raises(Timed):
            autotune.tune_ragged(batch, 0.01)
    finally:
        autotune._load = load
    entries[seen[0]] = {"variant": variant}


def test_a_capped_batch_keeps_its_cap(cache):
    from lime_amd import autotune
    sizes, kd = (16, 32, 100), (2, 0, 1)
    _remember(cache, _Batch(sizes, kd), 6)
    capped = _Batch(sizes, kd, max_groups=4)
    with pytest.raises(Timed):
        autotune.tune_ragged(capped, 0.01)
    _remember(cache, capped, 1)
    for batch, want in ((_Batch(sizes[::-1], kd[::-1]), 6), (_Batch(sizes, kd, max_groups=4), 1)):
        assert autotune.tune_ragged(batch, 0.01)[0] == want and batch.variant == want
    with pytest.raises(Timed):
        autotune.tune_ragged(_Batch(sizes, kd, max_groups=2), 0.01)


def test_batches_of_one_sum_are_told_apart(cache):
    from lime_amd import autotune
    few, many = _Batch((20,), (0,)), _Batch((10,) * 8, (0,) * 8)
    many.count = few.count                             # by the sum n^3 (1 + K_d) alone
    _remember(cache, few, 2)
    with pytest.raises(Timed):
        autotune.tune_ragged(many, 0.01)
    dense = _Batch((10, 10), (3, 3))
    _remember(cache, dense, 3)
    with pytest.raises(Timed):
        autotune.tune_ragged(_Batch((10, 10), (6, 0)), 0.01)


def test_a_stored_choice_that_the_batch_does_not_offer_is_timed_again(cache):
    from lime_amd import autotune
    batch = _Batch((16, 16), (0, 0))
    _remember(cache, batch, 7)
    with pytest.raises(Timed):
        autotune.tune_ragged(batch, 0.01)


@pytest.mark.gpu
def test_uncapped_then_capped_and_the_reverse(tmp_path, monkeypatch):
    from lime_amd import autotune
    from lime_amd.ragged import RaggedLindblad
    monkeypatch.setattr(autotune, "_CACHE_PATH", str(tmp_path / "tune.json"))
    rng = np.random.default_rng(2)
    inst = []
    for n in (8, 40, 70):
        x = rng.standard_normal((n, n))
        inst.append(dict(H=(x + x.T) / n + 0j, c_ops=[x / n ** 2], dephasing=0.01, rho0=np.eye(n) / n + 0j))
    for first in (0, 1):
        monkeypatch.setattr(autotune, "_cache", {})
        for cap in (first, 1 - first):
            rb = RaggedLindblad(inst, max_groups=cap)
            assert 0 <= rb.variant < rb.launches()
        assert len(autotune._cache) == 2
        assert all(len(v["ms"]) == (5 if k.endswith(":g1") else 7) for k, v in autotune._cache.items())


@pytest.mark.parametrize("variant,max_groups", [(-1, 0), (7, 0), (8, 0), (5, 1), (6, 3)])
def test_a_launch_that_is_not_offered_is_refused(variant, max_groups):
    """By the library, before any GPU work: the sizes are checked first."""
    from types import SimpleNamespace

    from lime_amd import _lib
    from lime_amd.ragged import RaggedLindblad
    rb = object.__new__(RaggedLindblad)
    rb._lib = _lib.load()
    rb.count, rb.variant, rb.max_groups = 1, variant, max_groups
    rb.inst = rb.order = rb.ops = rb.rho = rb.work = rb.queue = torch.zeros(1)
    rb.sizes, rb.kd, rb.cost, rb._lists, rb.dev = np.array([4]), np.array([0]), np.array([64.0]), {}, "cpu"
    with pytest.raises(_lib.LimeError, match="variant"):
        rb.step(0.01, 1, stream=SimpleNamespace(cuda_stream=0))


@pytest.mark.gpu
def test_the_first_step_of_a_batch_with_a_cached_choice_can_be_captured(cache):
    """The workgroup lists are there before the first step: a copy to the GPU cannot be captured."""
    from lime_amd import autotune
    from lime_amd.ragged import RaggedLindblad
    rng = np.random.default_rng(3)
    inst = []
    for n in (8, 33, 70):
        x = rng.standard_normal((n, n))
        inst.append(dict(H=(x + x.T) / n + 0j, c_ops=[x / n ** 2], dephasing=0.01, rho0=np.eye(n) / n + 0j))
    want = RaggedLindblad(inst, tune=False)
    for variant in (want.variants(), want.variants() + 1):
        want.variant = variant
        want.step(0.02, 1)                             # the kernels are loaded
        want.rho.copy_(RaggedLindblad(inst, tune=False).rho)
        cache[autotune.ragged_key(want)] = {"variant": variant}
        rb = RaggedLindblad(inst)
        assert rb.variant == variant and len(rb._lists) == 1
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            rb.step(0.02, 2)
        for _ in range(3):
            g.replay()
            want.step(0.02, 2)
            torch.cuda.synchronize()
            assert torch.equal(rb.rho, want.rho)
