"""The exact contraction's launch forms against numpy's exact integer sums: blocks of
one and of two row tiles per wave, the balanced launch cut along the sites and
uncut, at each trait class's tile counts, one group of sites to the last of few
groups and past it, and row counts around the blocks and at the sizes where the
form changes."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu


def _check(h, sites, traits, seed):
    rng = np.random.default_rng(seed)
    words = (sites + 511) // 512 * 8
    some = rng.integers(0, 2**63, (97, words), dtype=np.int64).view(np.uint64) << np.uint64(1)
    used = np.zeros(words * 64, np.uint8)
    used[:sites] = 1
    some &= np.packbits(used, bitorder="little").view(np.uint64)
    some[0] = np.packbits(used, bitorder="little").view(np.uint64)
    pick = rng.integers(0, 97, h)
    pick[[0, -1]] = 0
    most = 2**30 - 1
    k = rng.integers(-most, most + 1, (sites, traits))
    k[0, 0] = most
    bits = np.unpackbits(some.view(np.uint8), axis=1, bitorder="little")[:, :sites]
    want = (bits.astype(np.float64) @ k.astype(np.float64))[pick]  # below 2^53: exact
    z, _ = api.trait_contract(some[pick], k * 2.0**-24, api.TRAITS_EXACT_I8)
    assert np.array_equal(z * 2.0**24, want)


@pytest.mark.parametrize("traits", [2, 4, 6, 8, 9, 11, 16])
@pytest.mark.parametrize("h,sites", [(65, 60), (1000, 1024), (129, 1025), (3000, 3000), (64, 8192),
                                     (500, 8193), (40_001, 500), (70_001, 1500), (5000, 12_288)])
def test_forms(h, sites, traits):
    _check(h, sites, traits, h + sites + traits)


def test_uncut_round():
    # 625 row blocks of 320 rows for a round of 768
    _check(200_000, 9300, 2, 5)
