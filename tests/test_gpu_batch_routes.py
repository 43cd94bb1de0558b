"""Batches on either side of the sizes where their recombination changes its kernel:
few groups of gametes, many with few and with many events, wide rows, and row
chunks chosen for a replicate; every replicate equals a lone context bit for bit."""
import numpy as np
import pytest

from clotho_amd import api
from tests.parity_util import compare_gametes, compare_state

pytestmark = pytest.mark.gpu


def _population(n, alleles, seed):
    rng = np.random.default_rng(seed)
    words = (alleles + 511) // 512 * 8
    some = rng.integers(0, 2**63, (64, words), dtype=np.int64).view(np.uint64)
    used = np.zeros(words * 64, np.uint8)
    used[:alleles] = 1
    some &= np.packbits(used, bitorder="little").view(np.uint64)
    eff = np.round(rng.normal(0, 0.2, (alleles, 1)) * 2**24) / 2**24
    return some[rng.integers(0, 64, 2 * n)], rng.integers(0, 2**32, alleles) / 2**32, eff


# sizes with 4,608 groups are those of 147,456 individuals
@pytest.mark.parametrize("sizes,rho", [
    ([(300, 500), (200, 20_000), (90_000, 400), (55_000, 3000)], 1.0),   # 4,549 groups
    ([(300, 500), (200, 20_000), (90_000, 400), (60_000, 3000)], 1.0),   # 4,705, by event
    ([(300, 500), (200, 20_000), (90_000, 400), (60_000, 3000)], 4.0),   # by groups
    ([(100, 500), (75_000, 8000), (75_000, 7000), (400, 20_000)], 4.0),  # wide: by event
    ([(100, 500), (75_000, 900), (75_000, 700), (400, 20_000)], 70.0 / 2),  # over 64 events
])
def test_routes(sizes, rho):
    cfgs, pops = [], []
    for r, (n, alleles) in enumerate(sizes):
        cfgs.append(api.make_config(n, 20.0 / n, rho, seed=r, replicate=r, traits=1, neutral_p=0.2,
                                    sigma=0.1, fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0,
                                    max_alleles=alleles + 1024))
        pops.append(_population(n, alleles, r))
    batch = api.Batch(cfgs)
    for r, pop in enumerate(pops):
        batch.replicate(r).set_population(*pop)
    batch.replicate(1).set_launch_shape(recombine_chunks=3)
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


@pytest.mark.parametrize("mode", ["graph", "eager", "sequential"])
def test_width_looked_at_within_a_run(mode):
    # 8 x 12,500 from no alleles to about 110 words, where rho = 4 changes the rule
    cfgs = [api.make_config(12_500, 0.06, 4.0, seed=9, replicate=r, traits=1, neutral_p=0.3,
                            sigma=0.1, fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0,
                            max_alleles=1 << 14) for r in range(8)]
    batch = api.Batch(cfgs)
    batch.run(66, mode=mode)
    batch.run(2, mode=mode)
    for r in (0, 7):
        alone = api.Simulation(cfgs[r])
        for _ in range(17):
            alone.run(4, graph=True)
        rep = batch.replicate(r)
        assert rep.shape().words == alone.shape().words >= 100
        np.testing.assert_array_equal(rep.rows(), alone.rows())
        np.testing.assert_array_equal(rep.traits(), alone.traits())
        for a, b in zip(rep.free_space(), alone.free_space()):
            np.testing.assert_array_equal(a, b)
