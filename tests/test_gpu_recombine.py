"""The recombination at the edges of its groups, tables and tiles, bit for bit
against the CPU oracle: gamete counts around a group of 64 and its quarters,
rows of half a 16-word tile to several tiles of every wave, groups cut short by
their events (more than 768) or their new mutations (more than 192), more
than 64 events per gamete, positions at both ends of the key range, and row
chunks and column ranges from one to more than there are groups or tiles."""
import numpy as np
import pytest

import oracle
from clotho_amd import api
from tests.parity_util import compare_gametes, compare_state

pytestmark = pytest.mark.gpu


def _population(n, alleles, seed):
    rng = np.random.default_rng(seed)
    words = (alleles + 511) // 512 * 8
    bits = rng.uniform(0, 1, (2 * n, words * 64)) < 0.5
    bits[:, alleles:] = False
    bits[:, rng.integers(0, alleles, 3)] = True  # fixed columns
    rows = np.packbits(bits.astype(np.uint8), axis=1, bitorder="little").view(np.uint64)
    key = rng.integers(0, 2**32, alleles)
    key[:4] = 0, 2**32 - 1, 2**32 - 1, 2**31
    return rows, key / 2**32, np.round(rng.normal(0, 0.2, (alleles, 1)) * 2**24) / 2**24


@pytest.mark.parametrize("mu,rho", [(0.2, 5.0), (8.0, 25.0), (0.5, 60.0)])
@pytest.mark.parametrize("alleles", [60, 1000, 4700])
@pytest.mark.parametrize("n", [1, 8, 31, 32, 33, 100])
def test_groups_and_tiles(n, alleles, mu, rho):
    cfg = api.make_config(n, mu, rho, seed=n + alleles, traits=1, neutral_p=0.3, sigma=0.1,
                          fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0, max_alleles=1 << 13)
    sim, orc = api.Simulation(cfg), oracle.OracleSim(cfg)
    rows, pos, eff = _population(n, alleles, 7 * n + alleles)
    for x in (sim, orc):
        x.set_population(rows, pos, eff)
    default = sim.launch_shape()["recombine_chunks"]
    for g, chunks in enumerate((default, 1, min(3, 2 * n // 8 or 1), default)):
        sim.set_launch_shape(recombine_chunks=chunks)
        sim.run(1, graph=g == 3)
        orc.step()
        compare_gametes(sim, orc, f"generation {g + 1}, {chunks} chunks")
        compare_state(sim, orc, f"generation {g + 1}, {chunks} chunks")


@pytest.mark.parametrize("large", [False, True])
def test_batch_kernels(large):
    # a batch of few groups recombines by groups throughout; in one of more
    # than 16 groups per resident block the rows up to 256 words take a
    # lookup per event: every replicate equals a lone context
    specs = [(60, 100, 4.0), (33, 1600, 60.0), (50, 2100, 5.0), (40, 16384, 3.0), (41, 16500, 3.0)]
    if large:
        specs.append((420_000, 500, 2.0))  # 13,125 groups
    cfgs, pops = [], []
    for r, (n, alleles, rho) in enumerate(specs):
        cfgs.append(api.make_config(n, 20.0 / n, rho, seed=r, replicate=r, traits=1, neutral_p=0.2,
                                    sigma=0.1, fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0,
                                    max_alleles=alleles + 2048))
        rows, pos, eff = _population(min(n, 100), alleles, r)
        pops.append((rows[np.arange(2 * n) % len(rows)], pos, eff))
    batch = api.Batch(cfgs)
    for r, pop in enumerate(pops):
        batch.replicate(r).set_population(*pop)
    batch.run(2, mode="graph")
    batch.run(1, mode="eager")
    for r, cfg in enumerate(cfgs):
        lone = api.Simulation(cfg)
        lone.set_population(*pops[r])
        lone.run(3)
        compare_gametes(batch.replicate(r), lone, f"replicate {r}")
        compare_state(batch.replicate(r), lone, f"replicate {r}")
        lone.close()
    batch.close()


@pytest.mark.parametrize("alleles", [60, 1000, 4700])
@pytest.mark.parametrize("n,rho", [(20_000, 4.4), (20_000, 4.5), (13_001, 0.5)])
def test_large_capacity_few_events(n, rho, alleles):
    # two populations of 131,072 slots exceed the cache: up to rho^2 n = 4e5
    # (rho = 4.47 at n = 20,000) recombination takes a lookup per event and row
    cfg = api.make_config(n, 0.01, rho, seed=alleles, traits=1, neutral_p=0.3, sigma=0.1,
                          fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0, max_alleles=1 << 17)
    sim, orc = api.Simulation(cfg), oracle.OracleSim(cfg)
    rows, pos, eff = _population(100, alleles, alleles)
    rows = rows[np.arange(2 * n) % len(rows)]
    for x in (sim, orc):
        x.set_population(rows, pos, eff)
    for g in range(3):
        sim.run(1, graph=g == 2)
        orc.step()
        if g == 1:
            sim.autotune()
    compare_gametes(sim, orc, "generation 3")
    compare_state(sim, orc, "generation 3")
