"""Timed workloads of the offspring pipeline, through its public entry points.

Each case is a plain dict; prepare() builds what a user's program holds before
the call (contexts, batches, device buffers), run() is one pass of the
program, and work() is what that pass cannot do without.  Populations start
from synthetic standing variation with the neutral 1/f spectrum and run a few
generations of burn-in, so that passes see the slot turnover of a steady
state.  New mutations enter at about the rate that keeps the number of
segregating columns where it starts (or at the case's own rate).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from clotho_amd import api

FITNESS = {
    "constant": api.FIT_CONSTANT,
    "gaussian": api.FIT_GAUSSIAN,
    "quadratic": api.FIT_QUADRATIC,
    "gaussian_fixed": api.FIT_GAUSSIAN_FIXED,
    "stabilizing": api.FIT_MV_STABILIZING,
}


def _generations(name, n, slots, capacity, mu, rho, traits, fitness, gens, graph, **more):
    case = {"name": name, "kind": "generations", "n": n, "slots": slots, "capacity": capacity,
            "mu": mu, "rho": rho, "traits": traits, "fitness": fitness, "gens": gens,
            "graph": graph, "sigma": 0.1, "env": 0.0, "compact": False, "intermediates": 0,
            "burn": 30, "rows": False}
    case.update(more)
    return case


def listed():
    return [
        # one generation of a very small population and its whole state read
        # back: an interactive or teaching-size run, all launches and latency
        _generations("step_n200", 200, 3072, 8192, 0.5, 1.0, 1, "gaussian_fixed", 1, True,
                     env=1.0, rows=True),
        # the plain configuration: 1,000 diploid, random mating, one mutation
        # and one crossover per gamete, 100 generations launched one by one
        _generations("plain_n1000", 1000, 24576, 65536, 1.0, 1.0, 1, "constant", 100, False,
                     rows=True),
        # an ordinary quantitative-trait run of odd size: four traits,
        # N-scaled quadratic fitness, a logging period of 20 generations with
        # its population statistics
        _generations("period_n12345_t4", 12345, 20000, 28672, 0.035, 2.5, 4, "quadratic", 20,
                     False),
        # the single-population configuration the throughput is quoted on: a
        # logging period of 20 generations at 100,000 diploid
        _generations("period_n100k", 100_000, 50_176, 61_440, 0.0088, 5.0, 1, "gaussian_fixed",
                     20, True, env=1.0, burn=10),
        # a large 16-trait population under stabilising selection with its
        # fixed and lost columns compacted away every generation
        _generations("period_n250k_t16_compact", 250_000, 131_072, 163_840, 0.009, 10.0, 16,
                     "stabilizing", 10, True, sigma=0.002, compact=True, burn=3),
        # 256 replicates of uneven size advanced together
        {"name": "batch_256", "kind": "batch", "replicates": 256, "n_low": 1000, "n_high": 50000,
         "rho_low": 0.5, "rho_high": 5.0, "mu_low": 0.0005, "mu_high": 0.005, "capacity": 16384,
         "traits": 1, "gens": 50, "burn": 300, "graph": True},
        # a small parameter sweep: two dozen small replicates, three traits
        {"name": "batch_24_t3", "kind": "batch", "replicates": 24, "n_low": 200, "n_high": 3000,
         "rho_low": 0.5, "rho_high": 12.0, "mu_low": 0.01, "mu_high": 0.1, "capacity": 8192,
         "traits": 3, "gens": 50, "burn": 200, "graph": True},
        # analysis of one large population: margins over all rows, margins and
        # pairwise differences of a row sample
        {"name": "statistics_n100k", "kind": "statistics", "n": 100_000, "slots": 50_176,
         "sample": 1000},
        # the exact contraction on a caller's own device buffers: one small
        # odd-sized call, and the precision workload's shape
        {"name": "contract_h3001_t3", "kind": "contract", "h": 3001, "sites": 4000, "traits": 3},
        {"name": "contract_h200k_t16", "kind": "contract", "h": 200_000, "sites": 65_536,
         "traits": 16},
        # a split-BF16 contraction of host genotypes, the whole call
        {"name": "host_bf16_h20k_t8", "kind": "host_contract", "h": 20_000, "sites": 16_384,
         "traits": 8, "mode": "bf16", "terms": 3},
        # the base engine's loop: the caller draws mate pairs and mutations,
        # the library recombines, adds the mutations and evaluates fitness
        {"name": "base_engine_n5000", "kind": "base_engine", "n": 5000, "slots": 8192,
         "capacity": 20480, "mu": 0.02, "rho": 2.0, "traits": 1},
    ]


def _log_uniform(rng, low, high):
    return int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))


def draw(rng):
    kind = rng.choice(["generations", "generations", "generations", "batch", "statistics",
                       "contract", "contract", "host_contract", "base_engine"])
    if kind == "generations":
        n = _log_uniform(rng, 100, 150_000)
        traits = rng.choice([1, 1, 2, 3, 4, 5, 8, 11, 16, 20])
        # rows of at most about 2 GB per population
        slots = _log_uniform(rng, 600, min(131_072, 8_000_000_000 // n))
        mu = 0.9 * slots / (4.0 * n * (math.log(2 * n) + 0.6))
        compact = rng.random() < 0.3
        words = (slots + 511) // 512 * 8
        gens = max(1, min(60, int(6e9 / (48.0 * words * n * (1 + traits / 8)))))
        case = _generations("", n, slots, slots * 3 // 2 + 4096, mu,
                            round(math.exp(rng.uniform(math.log(0.3), math.log(22))), 3), traits,
                            rng.choice(sorted(FITNESS)), gens, rng.random() < 0.5,
                            compact=compact,
                            intermediates=0 if compact else rng.choice([0, 0, 0, 2]),
                            sigma=rng.choice([0.002, 0.1]), env=rng.choice([0.0, 1.0]),
                            burn=rng.choice([3, 20]), rows=n * words < 600_000)
    elif kind == "batch":
        top = _log_uniform(rng, 500, 20_000)
        case = {"kind": kind, "replicates": rng.randint(3, 160), "n_low": max(20, top // 40),
                "n_high": top, "rho_low": 0.3, "rho_high": rng.choice([1.0, 5.0, 14.0]),
                "mu_low": 20.0 / top, "mu_high": 150.0 / top, "capacity": 16384,
                "traits": rng.choice([1, 1, 2, 6, 16]), "gens": 30, "burn": 100,
                "graph": rng.random() < 0.7}
    elif kind == "statistics":
        n = _log_uniform(rng, 300, 100_000)
        case = {"kind": kind, "n": n, "slots": _log_uniform(rng, 600, 60_000),
                "sample": rng.randint(2, min(2 * n, 2500))}
    elif kind == "contract":
        case = {"kind": kind, "h": _log_uniform(rng, 500, 200_000),
                "sites": _log_uniform(rng, 500, 65_536), "traits": rng.randint(1, 16)}
    elif kind == "host_contract":
        case = {"kind": kind, "h": _log_uniform(rng, 500, 20_000),
                "sites": _log_uniform(rng, 500, 16_384), "traits": rng.randint(1, 16),
                "mode": rng.choice(["bf16", "exact_i8"]), "terms": rng.choice([2, 3])}
    else:
        n = _log_uniform(rng, 100, 8000)
        slots = _log_uniform(rng, 600, 16_384)
        case = {"kind": kind, "n": n, "slots": slots, "capacity": slots * 3 // 2 + 4096,
                "mu": 0.8 * slots / (4.0 * n * (math.log(2 * n) + 0.6)),
                "rho": round(rng.uniform(0.5, 8.0), 3), "traits": rng.choice([1, 2, 4])}
    case.pop("name", None)
    return case


# ---- inputs ---------------------------------------------------------------


def _standing_variation(n, slots, traits, sigma, seed):
    """Column frequencies P(f) ~ 1/f on [1/H, 1 - 1/H], uniform positions
    k 2^-32, effects on the 2^-24 grid."""
    rng = np.random.default_rng(seed)
    a, b = 1.0 / (2 * n), 1.0 - 1.0 / (2 * n)
    freqs = a * (b / a) ** rng.uniform(0, 1, slots)
    positions = np.floor(rng.uniform(0, 1, slots) * 2**32) / 2**32
    effects = np.round(rng.normal(0, sigma, (slots, traits)) * 2**24) / 2**24
    return freqs, positions, effects


def _population(case, seed, **config):
    sim = api.Simulation(api.make_config(case["n"], seed=seed, quantum_log2=-24, **config))
    sim.set_synthetic(*_standing_variation(case["n"], case["slots"], config["traits"],
                                           config["sigma"], seed), seed=seed)
    return sim


def _genotypes(case, seed):
    """Device genotypes (column frequencies in multiples of 1/256) and int32
    effects of the whole range the contraction takes."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    h, sites, traits = case["h"], case["sites"], case["traits"]
    words = (sites + 511) // 512 * 8

    def bits(*shape):
        return torch.randint(-2**63, 2**63 - 1, shape, generator=g, device="cuda",
                             dtype=torch.int64)

    rows = torch.zeros((h, words), dtype=torch.int64, device="cuda")
    for _ in range(8):
        level = bits(1, words)
        r = bits(h, words)
        rows = (rows & r) | (r & level) | (rows & level)  # level bit set: or, else and
    full, part = sites // 64, sites % 64
    if part:
        rows[:, full] &= (1 << part) - 1
        full += 1
    rows[:, full:] = 0
    effects = torch.randint(-(2**30 - 1), 2**30, (sites, traits), generator=g, device="cuda",
                            dtype=torch.int32)
    return rows, effects


def _host_genotypes(case, seed):
    rng = np.random.default_rng(seed)
    words = (case["sites"] + 511) // 512 * 8
    rows = rng.integers(0, 2**64, (case["h"], words), dtype=np.uint64)
    rows &= rng.integers(0, 2**64, (1, words), dtype=np.uint64) | rng.integers(
        0, 2**64, (case["h"], words), dtype=np.uint64)
    used = np.zeros(words * 64, np.uint8)
    used[: case["sites"]] = 1
    rows &= np.packbits(used, bitorder="little").view(np.uint64)[None, :]
    return rows, rng.standard_normal((case["sites"], case["traits"]))


MODES = {"bf16": api.TRAITS_MFMA_BF16, "exact_i8": api.TRAITS_EXACT_I8}


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "generations":
        sim = _population(case, seed, mu=case["mu"], rho=case["rho"], traits=case["traits"],
                          fitness=FITNESS[case["fitness"]], neutral_p=0.0, sigma=case["sigma"],
                          env_sigma=case["env"], max_alleles=case["capacity"],
                          compact=case["compact"], intermediates=case["intermediates"])
        sim.run(case["burn"], graph=case["graph"])
        state["sim"] = sim
        if case["rows"]:
            state["rows"] = np.zeros(2 * case["n"] * ((case["capacity"] + 511) // 512 * 8),
                                     np.int64)
    elif kind == "batch":
        rng = np.random.default_rng(42)  # the sweep's parameters; the seed draws the histories
        low, high = case["n_low"], case["n_high"]
        r = case["replicates"]
        sizes = np.exp(rng.uniform(np.log(low), np.log(high), r)).astype(np.int64)
        rho = rng.uniform(case["rho_low"], case["rho_high"], r)
        mu = rng.uniform(case["mu_low"], case["mu_high"], r)
        batch = api.Batch([
            api.make_config(int(sizes[i]), float(mu[i]), float(rho[i]), seed=seed, replicate=i,
                            traits=case["traits"], fitness=api.FIT_GAUSSIAN_FIXED, neutral_p=0.0,
                            sigma=0.1, env_sigma=1.0, quantum_log2=-24,
                            max_alleles=case["capacity"]) for i in range(r)])
        state["mode"] = "graph" if case["graph"] else "eager"
        batch.run(case["burn"], mode=state["mode"])
        state["batch"] = batch
    elif kind == "statistics":
        state["sim"] = _population(case, seed, mu=0.01, rho=1.0, traits=1, sigma=0.1,
                                   max_alleles=case["slots"])
        state["sample"] = api.sample_rows(seed, 1, 0, 2 * case["n"], case["sample"])
    elif kind == "contract":
        state["rows"], state["effects"] = _genotypes(case, seed)
        state["sums"] = torch.zeros((case["h"], case["traits"]), dtype=torch.int64,
                                    device="cuda")
    elif kind == "host_contract":
        state["rows"], state["effects"] = _host_genotypes(case, seed)
    else:
        sim = _population(case, seed, mu=case["mu"], rho=case["rho"], traits=case["traits"],
                          fitness=api.FIT_GAUSSIAN_FIXED, sigma=0.1, env_sigma=0.5,
                          max_alleles=case["capacity"], host_mutations=True)
        sim.evaluate_fitness()
        state["sim"] = sim
        state["rng"] = np.random.default_rng(seed)
    return state


# ---- one pass -------------------------------------------------------------
# Lists that a program keeps in buffers of the allele capacity (free slots,
# columns, allele attributes) are returned in arrays of that size.


def _in_capacity(case, *lists):
    out = []
    for x in lists:
        buf = np.zeros((case["capacity"],) + x.shape[1:], x.dtype)
        buf[: len(x)] = x
        out.append(buf)
    return out


def _run_generations(case, state):
    sim = state["sim"]
    sim.run(case["gens"], graph=case["graph"])
    out = {"traits": sim.traits(), "fitness": sim.fitness()}
    out["fixed"], out["lost"] = _in_capacity(case, *sim.free_space())
    if case["rows"]:  # into the caller's buffer, at the rows' present width
        rc = api.lib().clotho_download_population(sim.ctx, state["rows"].ctypes.data,
                                                  state["rows"].size)
        if rc:
            raise RuntimeError(f"download failed ({rc})")
        out["rows"] = state["rows"]
    else:  # the period's statistics: carriers per column, alleles per row
        columns, out["alleles"] = sim.allele_counts()
        out["columns"], out["positions"], out["effects"], out["ages"] = _in_capacity(
            case, columns, *sim.alleles())
    return out


def _run_base_engine(case, state):
    sim, rng, n = state["sim"], state["rng"], case["n"]
    sim.set_parents(rng.integers(0, n, 2 * n).astype(np.uint32))
    sim.run(1)
    m = int(rng.poisson(case["mu"] * 2 * n))
    rows = rng.integers(0, 2 * n, m).astype(np.uint32)
    positions = np.floor(rng.uniform(0, 1, m) * 2**32) / 2**32
    effects = np.round(rng.normal(0, 0.1, (m, case["traits"])) * 2**24) / 2**24
    slots = sim.add_mutations(rows, positions, effects)
    sim.evaluate_fitness()
    slots, fixed, lost = _in_capacity(case, slots, *sim.free_space())
    return {"slots": slots, "traits": sim.traits(), "fitness": sim.fitness(), "fixed": fixed,
            "lost": lost}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "generations":
        return _run_generations(case, state)
    if kind == "batch":
        batch = state["batch"]
        batch.run(case["gens"], mode=state["mode"])
        reps = [batch.replicate(r) for r in range(len(batch))]
        return {"traits": np.concatenate([s.traits() for s in reps]),
                "fitness": np.concatenate([s.fitness() for s in reps])}
    if kind == "statistics":
        sim, sample = state["sim"], state["sample"]
        columns, alleles = sim.allele_counts()
        sample_columns, sample_alleles = sim.allele_counts(sample)
        return {"columns": columns, "alleles": alleles, "sample_columns": sample_columns,
                "sample_alleles": sample_alleles,
                "differences": sim.pairwise_differences(sample)}
    if kind == "contract":
        rows, effects, sums = state["rows"], state["effects"], state["sums"]
        rc = api.lib().clotho_trait_contract_exact_noalloc(
            rows.data_ptr(), rows.shape[0], rows.shape[1], effects.data_ptr(), effects.shape[0],
            effects.shape[1], sums.data_ptr(),
            C.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(f"contraction failed ({rc})")
        return sums
    if kind == "host_contract":
        return api.trait_contract(state["rows"], state["effects"], MODES[case["mode"]],
                                  split_terms=case["terms"])[0]
    return _run_base_engine(case, state)


def work(case):
    """Bytes: every population read and written once per generation, traits
    and fitness once.  Operations: one multiply and add per (row, site,
    trait) of the contractions."""
    kind = case["kind"]
    if kind == "batch":
        # mean of the log-uniform sizes; about 600 segregating sites each
        low, high = case["n_low"], case["n_high"]
        h = 2.0 * case["replicates"] * (high - low) / math.log(high / low)
        words, t, gens = 16, case["traits"], case["gens"]
        return {"bytes": gens * h * (16.0 * words + 8 * t + 4),
                "flops": gens * 2.0 * h * words * 64 * t}
    if kind in ("contract", "host_contract"):
        h, s, t = float(case["h"]), case["sites"], case["traits"]
        words = (s + 511) // 512 * 8
        return {"bytes": h * (8 * words + 8 * t) + 4 * s * t, "flops": 2 * h * s * t}
    h = 2.0 * case["n"]
    words = (case["slots"] + 511) // 512 * 8
    if kind == "statistics":
        m = case["sample"]
        return {"bytes": 8 * words * (h + m) + 4 * (h + 2 * 64 * words + m + m * (m - 1) / 2),
                "flops": 0}
    gens, t = case.get("gens", 1), case["traits"]
    return {"bytes": gens * h * (16.0 * words + 8 * t + 4),
            "flops": gens * 2.0 * h * words * 64 * t}


def exact(case, seed):
    """The contractions' sums in 64 bits.  The simulations draw from the
    library's own streams and have no plain restatement."""
    if case["kind"] == "contract":
        rows, effects = _genotypes(case, seed)
        k = effects.double()
        shifts = torch.arange(64, device="cuda")
        out = torch.empty((rows.shape[0], k.shape[1]), dtype=torch.int64, device="cuda")
        step = max(1, (1 << 26) // (rows.shape[1] * 64))
        for r in range(0, rows.shape[0], step):
            bits = ((rows[r:r + step, :, None] >> shifts) & 1).reshape(-1, rows.shape[1] * 64)
            # integer sums below 2^53: exact in any order
            out[r:r + step] = (bits[:, : case["sites"]].double() @ k).long()
        return out
    if case["kind"] == "host_contract":
        rows, effects = _host_genotypes(case, seed)
        out = np.empty((rows.shape[0], effects.shape[1]))
        for r in range(0, rows.shape[0], 1000):
            bits = np.unpackbits(rows[r:r + 1000].view(np.uint8), axis=1, bitorder="little")
            out[r:r + 1000] = bits[:, : case["sites"]].astype(np.float64) @ effects
        return out
    return None
