"""Populations around the limits of the plain path's top of a generation and
trial phase, against the oracle, bit for bit: the best fitness by one scan or
in parallel (32 members), the statistics' windows (1056), the copy of the
members' buffer indices in LDS (11264), blocks shared out across members, and
renormalized trials with more and fewer members than workgroups.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,G,kw", [
    (32, 70, {}), (33, 70, {}), (248, 65, {}), (249, 130, {}), (1056, 40, {}), (1057, 40, {}), (2113, 20, {}),
    (11264, 4, {}), (11265, 4, {}), (500, 150, dict(zero_temperature=True)),
    (247, 70, dict(normalize=True, renormalize=True)), (249, 129, dict(normalize=True, renormalize=True)),
    (1000, 33, dict(normalize=True, renormalize=True)), (11265, 3, dict(normalize=True, renormalize=True)),
    (20, 321, dict(normalize=True, renormalize=True, allow_negative=True)),
])
def test_population_sizes_match_oracle(P, G, kw):
    print(f"[gpu] population P={P} G={G} {kw}", flush=True)
    T, seed, N = 5, 7, 8 if P > 1100 else 14
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    freq = ob.frequency_grid(G, 48.0)
    o = ob.run(ob.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, number_of_generations=N, population_size=P,
                               stop_minimum_fitness=0.0, **kw), seed)
    with da.Engine(da.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, population_size=P, **kw)) as e:
        g = e.run(seed, N, 0.0)
    assert g["rng"] == o["rng"]
    for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
        assert gc.bit_diff(g[k], o[k]) is None, (k, gc.bit_diff(g[k], o[k]))
