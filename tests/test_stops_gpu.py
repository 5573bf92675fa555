"""Stops at every generation of a run's first batches, whatever their lengths: on a
batch's first and last generation and inside, while the next batches' draws are
made beside it.  The threshold is the oracle's best fitness where it drops at
that generation, from the first seed whose run drops there.  One handle takes
all runs, so that each starts from what a stopped one left behind.  Bar: the
oracle's generation, random state, statistics, DSF and fitnesses, bit for bit.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,T,G,last,kw,run", [
    (8, 9, 16, 130, {}, {}),                                       # trials beside the chains, serial walk
    (62, 17, 12, 70, {}, {}),                                      # the same, walk of many members
    (63, 5, 70, 70, {}, {}),
    (200, 17, 20, 70, {}, {}),
    (130, 33, 12, 70, {}, {}),                                     # selection by wavefronts
    (9, 20, 33, 70, dict(normalize=True, renormalize=True), {}),   # trial phase, repeated selection
    (24, 18, 31, 70, dict(spectra_type="bdsf"), {}),               # folds
    (24, 17, 20, 70, {}, dict(split_loop=True)),
])
def test_stops_at_every_generation(P, T, G, last, kw, run):
    print(f"[gpu] stops P={P} T={T} G={G} {kw} {run}", flush=True)
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    freq = ob.frequency_grid(G, 48.0)
    N = 3 * last

    def oracle(seed, n, stop):
        return ob.run(ob.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, number_of_generations=n, population_size=P,
                                      stop_minimum_fitness=stop, **kw), seed)

    drops = {}  # generation: seed, best fitness there
    for seed in range(1, 100):
        m = oracle(seed, last + 2, 0.0)["minimum"]
        for g in range(last + 1):
            if g not in drops and (g == 0 or m[g] < m[g - 1]):
                drops[g] = seed, float(m[g])
        if len(drops) == last + 1:
            break
    assert len(drops) == last + 1
    with da.Engine(da.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, population_size=P, **kw)) as e:
        for g, (seed, stop) in drops.items():
            o, s = oracle(seed, N, stop), e.run(seed, N, stop, **run)
            assert o["generation"] == s["generation"] == g
            assert s["rng"] == o["rng"], g
            for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
                assert gc.bit_diff(s[k], o[k]) is None, (g, k, gc.bit_diff(s[k], o[k]))
