"""Device memory that calls keep between them: scratch buffers of at most 64 MiB per
device for all contexts, as many as calls were under way at a time, and none of a
replicate's for launches that its batch does not make."""
import threading
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _used():
    free, total = api.device_memory()
    return total - free


def _context(n, slots, seed):
    sim = api.Simulation(api.make_config(n, 0.1, 1.0, seed=seed, traits=1, max_alleles=slots))
    rng = np.random.default_rng(seed)
    sim.set_synthetic(rng.uniform(0, 1, slots), np.arange(slots) / 2**32, np.zeros((slots, 1)),
                      seed=seed)
    return sim


def test_contexts_share_scratch():
    sims = [_context(20_000, 8192, s) for s in range(12)]  # about 14 MB of partials a call
    first = sims[0].allele_counts()
    before = _used()
    for s in sims[1:]:
        s.allele_counts()
        s.traits()
    assert _used() - before <= 4 * MIB
    again = sims[0].allele_counts()
    assert all(np.array_equal(a, b) for a, b in zip(first, again))
    for s in sims:
        s.close()


def test_as_many_buffers_as_threads():
    start = _used()
    sims = [_context(20_000, 8192, s) for s in range(12)]
    want = [s.allele_counts() for s in sims]
    one = _used()
    with ThreadPoolExecutor(4) as pool:
        for _ in range(3):
            got = list(pool.map(lambda s: s.allele_counts(), sims))
            for a, b in zip(want, got):
                assert all(np.array_equal(x, y) for x, y in zip(a, b))
    assert _used() - one <= 3 * 64 * MIB
    for s in sims:
        s.close()
    assert _used() - start <= 8 * MIB


def test_threads_with_contexts_of_their_own():
    sims = [_context(5000, 4096, s) for s in range(4)]
    sample = np.arange(0, 10_000, 40, dtype=np.uint32)
    want = [(s.allele_counts(), s.allele_counts(sample), s.pairwise_differences(sample), s.traits())
            for s in sims]
    errors = []

    def work(s, w):
        for _ in range(5):
            got = (s.allele_counts(), s.allele_counts(sample), s.pairwise_differences(sample),
                   s.traits())
            for a, b in zip(got, w):
                a, b = (a, b) if isinstance(a, tuple) else ((a,), (b,))
                if not all(np.array_equal(x, y) for x, y in zip(a, b)):
                    errors.append(s)

    threads = [threading.Thread(target=work, args=p) for p in zip(sims, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for s in sims:
        s.close()


def test_replicates_hold_no_pieces():
    # 16 traits: a balanced launch of a replicate's own would keep up to 33 MB for its
    # pieces, which a batch never makes
    cfgs = [api.make_config(4000, 0.01, 1.0, seed=1, replicate=r, traits=16, sigma=0.1,
                            max_alleles=4096) for r in range(8)]
    batch = api.Batch(cfgs)
    lone = api.Simulation(cfgs[0])
    per = [batch.replicate(r).device_bytes() for r in range(8)]
    assert max(per) < lone.device_bytes() - 3 * MIB
    rng = np.random.default_rng(2)
    rows = rng.integers(0, 2**63, (8000, 32), dtype=np.int64).view(np.uint64)
    eff = rng.integers(-2**20, 2**20, (2048, 16)) * 2.0**-24
    for s in (lone, *[batch.replicate(r) for r in range(8)]):
        s.set_population(rows, np.arange(2048) / 2**32, eff)
    assert max(batch.replicate(r).device_bytes() for r in range(8)) == max(per)
    assert np.array_equal(batch.replicate(3).traits(), lone.traits())
    batch.run(2, mode="graph")
    lone.run(2)
    assert np.array_equal(batch.replicate(0).traits(), lone.traits())
    batch.run(2, mode="sequential")  # replicates' own launches
    lone.run(2)
    assert np.array_equal(batch.replicate(0).traits(), lone.traits())
    batch.close()
    lone.close()
