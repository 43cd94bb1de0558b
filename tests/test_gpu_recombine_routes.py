"""The recombination where its kernel follows the population's width: a lookup per
event and row for wide rows of many individuals with few events, groups of
gametes for the others, changing at the start of a run with eager and captured
launches alike; bit for bit against the CPU oracle."""
import numpy as np
import pytest

import oracle
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
    some[:, 0] |= np.uint64(5)  # two fixed columns
    key = rng.integers(0, 2**32, alleles)
    key[:3] = 0, 2**32 - 1, 2**31
    eff = np.round(rng.normal(0, 0.2, (alleles, 1)) * 2**24) / 2**24
    return some[rng.integers(0, 64, 2 * n)], key / 2**32, eff


def _pair(n, rho, slots):
    cfg = api.make_config(n, 3.0 / n, rho, seed=7, traits=1, neutral_p=0.3, sigma=0.1,
                          fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0, max_alleles=slots)
    return api.Simulation(cfg), oracle.OracleSim(cfg)


def _steps(sim, orc, generations, graph, when):
    sim.run(generations, graph=graph)
    for _ in range(generations):
        orc.step()
    compare_gametes(sim, orc, when)
    compare_state(sim, orc, when)


@pytest.mark.parametrize("rho", [0.0, 0.5, 4.4])
def test_width_decides(rho):
    # two populations of n = 4,200: 384 words 52 MB, 144 words 19 MB, 8 words 1 MB;
    # by event from 20 MB + 50 MB rho on
    sim, orc = _pair(4200, rho, 1 << 15)
    for alleles, graph in ((60, True), (24_400, True), (9000, False), (24_100, False), (500, True)):
        for x in (sim, orc):
            x.set_population(*_population(4200, alleles, alleles))
        _steps(sim, orc, 2, graph, f"rho {rho}, {alleles} alleles")
        # the first run after an upload sees its width: 17 chunks of 512 rows by
        # event, as many as there are groups otherwise
        by_event = 2 * 8 * 8400 * ((alleles + 511) // 512 * 8) > (20 + 50 * rho) * 1e6
        assert sim.launch_shape()["recombine_chunks"] == (17 if by_event else 132)


def test_chosen_chunks_stay():
    sim, orc = _pair(4200, 0.5, 1 << 15)
    for x in (sim, orc):
        x.set_population(*_population(4200, 400, 1))
    sim.set_launch_shape(recombine_chunks=37)
    for alleles in (400, 24_000):
        for x in (sim, orc):
            x.set_population(*_population(4200, alleles, alleles))
        _steps(sim, orc, 1, alleles > 400, f"{alleles} alleles")
        assert sim.launch_shape()["recombine_chunks"] == 37


def test_tuned_by_event():
    sim, orc = _pair(4200, 0.5, 1 << 15)
    for x in (sim, orc):
        x.set_population(*_population(4200, 24_000, 3))
    _steps(sim, orc, 1, False, "before")
    sim.autotune()
    _steps(sim, orc, 2, True, "tuned")


@pytest.mark.parametrize("chunks", [1, 3, 8, 13])
def test_blocks_without_work(chunks):
    # the grid has several blocks per chunk for wide rows; rows of up to 32 words have
    # work in one of them only
    sim, orc = _pair(700, 1.5, 1 << 15)
    sim.set_launch_shape(recombine_chunks=chunks)
    for alleles, graph in ((300, True), (1900, False), (2400, True), (100, True)):
        for x in (sim, orc):
            x.set_population(*_population(700, alleles, alleles))
        _steps(sim, orc, 2, graph, f"{chunks} chunks, {alleles} alleles")


@pytest.mark.parametrize("graph", [True, False])
def test_width_looked_at_within_a_run(graph):
    # 0 words at the start, about 270 at generation 64: by event from there on
    cfg = api.make_config(4200, 0.2, 0.0, seed=5, traits=1, neutral_p=0.3, sigma=0.1,
                          fitness=api.FIT_GAUSSIAN_FIXED, env_sigma=1.0, max_alleles=1 << 15)
    sim, orc = api.Simulation(cfg), oracle.OracleSim(cfg)
    assert sim.launch_shape()["recombine_chunks"] == 132
    _steps(sim, orc, 67, graph, "from no alleles")
    assert sim.launch_shape()["recombine_chunks"] == 17


@pytest.mark.parametrize("words", [152, 192, 200])
def test_capacity_beyond_the_width(words):
    # by event with 3 and 4 live column tiles of 64
    sim, orc = _pair(4200, 0.0, 1 << 18)
    for x in (sim, orc):
        x.set_population(*_population(4200, 64 * words - 100, words))
    _steps(sim, orc, 2, True, f"{words} words")
    assert sim.launch_shape()["recombine_chunks"] == 17


def test_saved_chunks_by_phases():
    # chunks tuned by event, given to a context that has no population yet; the
    # phases of a generation called one by one
    sim, orc = _pair(4200, 0.5, 1 << 15)
    sim.set_launch_shape(recombine_chunks=17)
    for alleles in (400, 24_000, 300):
        for x in (sim, orc):
            x.set_population(*_population(4200, alleles, alleles))
        for _ in range(2):
            for phase in ("draw", "recombine_mutate", "traits", "free_space", "fitness", "commit"):
                assert getattr(api.lib(), "clotho_phase_" + phase)(sim.ctx) == 0
            orc.step()
        compare_gametes(sim, orc, f"{alleles} alleles")
        compare_state(sim, orc, f"{alleles} alleles")
        _steps(sim, orc, 1, True, f"{alleles} alleles, a run")
        assert sim.launch_shape()["recombine_chunks"] == 17
