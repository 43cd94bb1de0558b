"""Pairwise differences at the edges of the 64-row tiles and 32-word chunks,
with one word range per tile and with several, against numpy's counts (whole
numbers: equal)."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alleles", [40, 2000, 2100, 9000])
@pytest.mark.parametrize("rows", [2, 63, 64, 65, 129, 700])
def test_pairwise_edges(rows, alleles):
    rng = np.random.default_rng(rows + alleles)
    n, words = 400, (alleles + 511) // 512 * 8
    bits = rng.uniform(0, 1, (2 * n, words * 64)) < rng.uniform(0, 1, (2 * n, 1))
    bits[:, alleles:] = False
    pop = np.packbits(bits.astype(np.uint8), axis=1, bitorder="little").view(np.uint64)
    sim = api.Simulation(api.make_config(n, 0.1, 1.0, traits=1, max_alleles=alleles))
    sim.set_population(pop, np.arange(alleles) / 2**32, np.zeros((alleles, 1)))
    sample = rng.integers(0, 2 * n, rows).astype(np.uint32)  # rows may repeat
    x = bits[sample].astype(np.float32)
    counts = x.sum(axis=1)
    differ = counts[:, None] + counts[None, :] - 2 * (x @ x.T)  # exact: below 2^24
    want = differ[np.triu_indices(rows, 1)].astype(np.uint32)
    assert np.array_equal(sim.pairwise_differences(sample), want)


def test_pairwise_whole_population():
    # 5000 rows: 3160 tiles, one word range each
    n = 2500
    rng = np.random.default_rng(5)
    pop = rng.integers(0, 2**63, (2 * n, 16), dtype=np.int64).view(np.uint64)
    sim = api.Simulation(api.make_config(n, 0.1, 1.0, traits=1, max_alleles=1024))
    sim.set_population(pop, np.arange(1024) / 2**32, np.zeros((1024, 1)))
    x = np.unpackbits(pop.view(np.uint8), axis=1).astype(np.float32)
    counts = x.sum(axis=1)
    differ = counts[:, None] + counts[None, :] - 2 * (x @ x.T)
    want = differ[np.triu_indices(2 * n, 1)].astype(np.uint32)
    assert np.array_equal(sim.pairwise_differences(np.arange(2 * n, dtype=np.uint32)), want)
