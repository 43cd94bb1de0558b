"""The exact traits where the FP32 accumulators are fullest.  Effects of
-16 (32^6 - 1) / 31 have six digits of -16, so that a row with every site set takes
the sums of six digit planes to -2^23 units of 1/8, the last value that a float
holds in such units, at the end of a segment of 2^19 sites; single units are
added beside sums that are nearly there.  In the fixed launch shapes one wave sums
whole segments, in the balanced one shares of them."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu

SEGMENT = 1 << 19
FULL = -16 * (32**6 - 1) // 31  # -554,189,328


@pytest.mark.parametrize("sites", [SEGMENT, SEGMENT + 2048])
@pytest.mark.parametrize("traits", [1, 2, 4, 5, 16, 20])
def test_full_accumulators(traits, sites):
    rng = np.random.default_rng(traits + sites)
    n = 9
    k = np.full((sites, traits), FULL, np.int64)
    # one digit unit up or down in a random plane: before the end of the segment,
    # so that it is added beside a nearly full sum, and scattered
    late = np.arange(SEGMENT - 3000, SEGMENT)
    some = rng.integers(0, sites, 500)
    for t in range(1, traits):  # the first trait stays at the limit
        k[late, t] = rng.choice([-1, 1], late.size) * 32 ** rng.integers(0, 6, late.size)
        k[some, t] = rng.integers(-1, 2, some.size) * 32 ** rng.integers(0, 6, some.size)
    words = (sites + 511) // 512 * 8
    bits = np.zeros((2 * n, words * 64), np.uint8)
    bits[:, :sites] = 1
    bits[1, : SEGMENT // 2] = 0
    bits[2, :sites] = rng.integers(0, 2, sites)
    bits[3, late] = rng.integers(0, 2, late.size)
    bits[4, rng.integers(0, sites, 1000)] = 0
    rows = np.packbits(bits, axis=1, bitorder="little").view(np.uint64)
    want = bits[:, :sites].astype(np.float64) @ k.astype(np.float64)  # below 2^53: exact
    sim = api.Simulation(api.make_config(n, 1.0, 1.0, traits=traits, max_alleles=sites))
    for v in range(1, sim.launch_shape()["traits_variants"] + 1):
        sim.set_launch_shape(traits_variant=v)
        sim.set_population(rows, np.arange(sites) / 2**32, k * 2.0**-24)
        assert np.array_equal(sim.traits() * 2.0**24, want), f"shape {v}"
    sim.close()
