"""The exact traits at the edges of their digit planes, tiles and row blocks,
against numpy's exact integer sums: every trait class (1-2, 3-4, 5-8, 9-16, 17-32
traits) with effects of one to seven base-32 digits, row counts around the
row blocks and below one of them, widths of half a 16-word group to several
groups, and rows of more than the 512 groups that are summed at a time."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu

# largest |k| of 1 .. 7 balanced base-32 digits, and the first of the next
EDGES = [15 * (32**p - 1) // 31 for p in range(1, 7)]


def _exact(rows, k):
    """Integer sums (below 2^53: exact in float64 in any order)."""
    out = np.empty((rows.shape[0], k.shape[1]))
    for r in range(0, rows.shape[0], 256):
        bits = np.unpackbits(rows[r:r + 256].view(np.uint8), axis=1, bitorder="little")
        out[r:r + 256] = bits[:, : k.shape[0]].astype(np.float64) @ k.astype(np.float64)
    return out


def _rows(rng, h, sites, p=0.4):
    words = (sites + 511) // 512 * 8
    bits = rng.uniform(0, 1, (h, words * 64)) < p
    bits[:, sites:] = False
    bits[0, :sites] = True  # a full row: the largest sums
    return np.packbits(bits.astype(np.uint8), axis=1, bitorder="little").view(np.uint64)


@pytest.mark.parametrize("most", [3, *[e + d for e in EDGES for d in (0, 1)], 2**30 - 1])
@pytest.mark.parametrize("traits", [1, 2, 3, 8, 11, 16, 32])
def test_population_traits_at_digit_edges(traits, most):
    rng = np.random.default_rng(traits * 1000 + most % 997)
    n, sites = 170, 1100
    rows = _rows(rng, 2 * n, sites)
    k = rng.integers(-most, most + 1, (sites, traits))
    k[0], k[-1] = most, -most  # the bound itself, at the first and last site
    sim = api.Simulation(api.make_config(n, 1.0, 1.0, traits=traits, max_alleles=2048))
    pos = np.arange(sites) / 2**32
    sim.set_population(rows, pos, k * 2.0**-24)
    assert np.array_equal(sim.traits() * 2.0**24, _exact(rows, k))
    # every launch shape of the class
    for v in range(1, sim.launch_shape()["traits_variants"] + 1):
        sim.set_launch_shape(traits_variant=v)
        sim.set_population(rows, pos, k * 2.0**-24)
        assert np.array_equal(sim.traits() * 2.0**24, _exact(rows, k)), f"shape {v}"


@pytest.mark.parametrize("h", [1, 15, 17, 255, 257, 319, 321, 1281])
@pytest.mark.parametrize("sites", [60, 512, 1024, 1500, 9000])
@pytest.mark.parametrize("traits", [1, 4, 9])
def test_contraction_row_blocks(h, sites, traits):
    rng = np.random.default_rng(h * 7 + sites + traits)
    rows = _rows(rng, h, sites)
    k = rng.integers(-(2**30 - 1), 2**30, (sites, traits))
    k[0, 0] = 2**30 - 1
    z, _ = api.trait_contract(rows, k * 2.0**-24, api.TRAITS_EXACT_I8)
    assert np.array_equal(z * 2.0**24, _exact(rows, k))


@pytest.mark.parametrize("traits", [1, 5])
def test_contraction_past_one_segment(traits):
    """Rows of 517 groups: the sums of two segments are added in 64 bits."""
    rng = np.random.default_rng(traits)
    h, sites = 70, 529_000
    rows = _rows(rng, h, sites)
    k = rng.integers(2**29, 2**30, (sites, traits))  # one sign: the largest partial sums
    z, _ = api.trait_contract(rows, k * 2.0**-24, api.TRAITS_EXACT_I8)
    assert np.array_equal(z * 2.0**24, _exact(rows, k))
