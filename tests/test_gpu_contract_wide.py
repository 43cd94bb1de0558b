"""The exact contraction over rows whose digit planes take more than 4 GB: bits
set past the last site do not count, however far past it they are."""
import numpy as np
import pytest

from clotho_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("traits,words,h", [(16, 800_000, 2), (1, 5_600_000, 1)])
def test_bits_far_past_the_sites(traits, words, h):
    # 86,016 bytes of planes per 16 words at 16 traits, 12,288 at one
    rng = np.random.default_rng(words)
    sites = 2000
    k = rng.integers(2**29, 2**30, (sites, traits))  # one sign: nothing cancels
    rows = np.zeros((h, words), np.uint64)
    rows[:, : sites // 64] = rng.integers(0, 2**63, (h, sites // 64), dtype=np.int64).view(np.uint64)
    bits = np.unpackbits(rows[:, : (sites + 63) // 64].copy().view(np.uint8), axis=1,
                         bitorder="little")[:, :sites]
    want = bits.astype(np.int64) @ k
    rows[:, words - 32_768:] = 2**64 - 1
    z, _ = api.trait_contract(rows, k * 2.0**-24, api.TRAITS_EXACT_I8)
    # effects of 2^29 .. 2^30 units: the quantisation keeps the 2^-24 grid or a finer one
    assert np.array_equal(z * 2.0**24, want.astype(np.float64))
