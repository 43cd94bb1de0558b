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
