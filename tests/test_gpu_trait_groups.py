"""The population's exact traits on either side of the row widths where their launch
changes: rows of up to eight groups of 16 words in whole blocks, wider ones cut
along the sites, and for more than 16 traits one row tile per wave up to 256
words and two beyond, also where a population grows across; against numpy's
exact sums over the rows and effects that the library reports."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu


def _check(sim, when):
    rows, (_, eff, _) = sim.rows(), sim.alleles()
    bits = np.unpackbits(rows.view(np.uint8), axis=1, bitorder="little")[:, : len(eff)]
    # effects are multiples of 2^-24 below 2^6: sums below 2^53 units are exact
    assert np.array_equal(sim.traits(), bits.astype(np.float64) @ eff), when


def _population(rng, n, alleles, traits):
    words = (alleles + 511) // 512 * 8
    some = rng.integers(0, 2**63, (50, words), dtype=np.int64).view(np.uint64)
    used = np.zeros(words * 64, np.uint8)
    used[:alleles] = 1
    some &= np.packbits(used, bitorder="little").view(np.uint64)
    rows = some[rng.integers(0, 50, 2 * n)]
    eff = rng.integers(-2**21, 2**21, (alleles, traits)) * 2.0**-24
    return rows, rng.integers(0, 2**32, alleles) / 2**32, eff


@pytest.mark.parametrize("traits", [1, 3, 6, 11, 17, 32])
@pytest.mark.parametrize("n,alleles", [(40, 500), (33, 8192), (33, 8193), (700, 16_384),
                                       (700, 16_900), (3000, 1000), (40_000, 400)])
def test_widths(n, alleles, traits):
    rng = np.random.default_rng(n + alleles + traits)
    sim = api.Simulation(api.make_config(n, 2.0 / n, 1.0, seed=3, traits=traits, neutral_p=0.0,
                                         sigma=0.1, max_alleles=alleles + 512))
    sim.set_population(*_population(rng, n, alleles, traits))
    _check(sim, "upload")
    sim.run(1)
    sim.run(2, graph=True)
    _check(sim, "generation 3")
    sim.close()


@pytest.mark.parametrize("traits", [4, 20])
def test_growing_width(traits):
    # 15,900 sites of 248 words to more than 256 words, captured launches throughout
    rng = np.random.default_rng(traits)
    n = 100
    sim = api.Simulation(api.make_config(n, 1.0, 1.0, seed=3, traits=traits, neutral_p=0.0,
                                         sigma=0.1, max_alleles=24_576))
    sim.set_population(*_population(rng, n, 15_900, traits))
    widths = []
    for g in range(10):
        sim.run(2, graph=True)
        widths.append(sim.shape().words)
        _check(sim, f"generation {2 * g + 2}")
    assert widths[0] <= 256 < widths[-1]
    small = _population(rng, n, 900, traits)
    sim.set_population(*small)  # and narrow again
    sim.run(3, graph=True)
    _check(sim, "narrow again")
    sim.close()


def test_batch_many_traits():
    cfgs = [api.make_config(n, 2.0 / n, 1.0, seed=5, replicate=r, traits=20, neutral_p=0.0,
                            sigma=0.1, max_alleles=a + 1024)
            for r, (n, a) in enumerate([(30, 400), (200, 3000), (65, 17_000)])]
    batch = api.Batch(cfgs)
    rng = np.random.default_rng(9)
    for r, (n, a) in enumerate([(30, 400), (200, 3000), (65, 17_000)]):
        batch.replicate(r).set_population(*_population(rng, n, a, 20))
    batch.run(3, mode="graph")
    for r in range(3):
        _check(batch.replicate(r), f"replicate {r}")
    batch.close()


@pytest.mark.parametrize("traits", [2, 4, 8, 16, 20])
@pytest.mark.parametrize("n", [150, 8192, 8193, 10_241])
def test_few_groups(n, traits):
    # 3, 4, 5 and 8 groups of 16 words, whole or cut by the number of rows
    rng = np.random.default_rng(n + traits)
    sim = api.Simulation(api.make_config(n, 2.0 / n, 1.0, seed=3, traits=traits, neutral_p=0.0,
                                         sigma=0.1, max_alleles=8704))
    for alleles in (3072, 4096, 4100, 8192):
        sim.set_population(*_population(rng, n, alleles, traits))
        _check(sim, f"{alleles} alleles")
        sim.run(1)
        _check(sim, f"{alleles} alleles, a generation on")
    sim.close()
