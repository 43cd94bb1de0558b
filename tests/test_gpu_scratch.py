"""Device memory that calls keep between them: one scratch allocation of at most 64 MiB
per device for all contexts."""
import threading

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
