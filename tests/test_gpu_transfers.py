"""Results on either side of the sizes where their way to the caller changes:
32 KB (pinned stage or the caller's pages) and 64 MiB (kept scratch memory or
its own), and the two flags of the shape with their one odd value at either end."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,traits,alleles", [(2048, 1, 8192), (2049, 1, 8193), (4096, 2, 100),
                                              (4097, 2, 8191), (135000, 32, 300)])
def test_downloads(n, traits, alleles):
    rng = np.random.default_rng(n)
    words = (alleles + 511) // 512 * 8
    bits = rng.uniform(0, 1, (64, words * 64)) < 0.5
    bits[:, alleles:] = False
    some = np.packbits(bits.astype(np.uint8), axis=1, bitorder="little").view(np.uint64)
    pick = rng.integers(0, 64, 2 * n)
    k = rng.integers(-2**20, 2**20, (alleles, traits))
    key = rng.integers(0, 2**32, alleles)
    fitness = rng.uniform(0.1, 1.0, n)
    sim = api.Simulation(api.make_config(n, 0.1, 1.0, traits=traits, max_alleles=alleles))
    sim.set_population(some[pick], key / 2**32, k * 2.0**-24, fitness)
    sums = bits[:, :alleles].astype(np.float64) @ k.astype(np.float64)  # exact: below 2^53
    assert np.array_equal(sim.traits() * 2.0**24, sums[pick])
    assert np.array_equal(sim.fitness(), fitness)
    pos, eff, _ = sim.alleles()
    assert np.array_equal(pos, key / 2**32) and np.array_equal(eff * 2.0**24, k)
    fixed, lost = sim.free_space()
    used = bits[np.unique(pick)]
    assert np.array_equal(fixed, np.flatnonzero(used[:, :alleles].all(axis=0)))
    assert np.array_equal(lost, np.flatnonzero(~used[:, :alleles].any(axis=0)))


@pytest.mark.parametrize("at", [0, 1, 63, 16384, 70000 - 1])
def test_shape_flags(at):
    n, alleles = 70000, 500
    sim = api.Simulation(api.make_config(n, 0.1, 1.0, traits=1, max_alleles=512))
    rows = np.zeros((2 * n, 8), np.uint64)
    rows[0] = 1
    pos, eff, fitness = np.arange(alleles) / 2**32, np.zeros((alleles, 1)), np.full(n, 0.5)
    sim.set_population(rows, pos, eff, fitness)
    s = sim.shape()
    assert s.all_neutral == 1 and s.fitness_constant == 1
    fitness[at] = 0.25
    eff[min(at, alleles - 1)] = 2.0**-24
    sim.set_population(rows, pos, eff, fitness)
    s = sim.shape()
    assert s.all_neutral == 0 and s.fitness_constant == 0
    fitness[:] = 0.5
    fitness[at] = np.nan
    sim.set_population(rows, pos, eff, fitness)
    assert sim.shape().fitness_constant == 0
