"""The wide random walk (populations of 20 to 4096 with equal redraw
probabilities) and its serial form, against the oracle's stream: every
member's draws change the returned random state and the results, so both are
compared bit for bit.  Populations around the 63 members of a block, redraw
probabilities from none to all (every draw a test; every test followed by a
value), unequal ones (serial), and one and two signs.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [19, 20, 21, 62, 63, 64, 65, 126, 127, 300, 512])
@pytest.mark.parametrize("tau", [(0.1, 0.1), (0.0, 0.0), (1.0, 1.0), (0.5, 0.5), (0.97, 0.97), (0.1, 0.3)])
def test_walk_matches_oracle(P, tau):
    print(f"[gpu] walk P={P} redraw {tau}", flush=True)
    t = np.linspace(0.0, 0.37, 4)
    isf = 0.55 * np.exp(-1.7 * t) + 0.45 * np.exp(-0.4 * t)
    freq = ob.frequency_grid(6, 48.0)
    for zero_t, seed in ((False, 3), (True, 4)):
        kw = dict(population_size=P, zero_temperature=zero_t, self_adapting_crossover_probability=tau[0],
                  self_adapting_differential_weight_probability=tau[1])
        N = 26 if P > 100 else 60
        o = ob.run(ob.make_problem(t, isf, 1e-2 * isf, freq, 1.35, number_of_generations=N, stop_minimum_fitness=0.0,
                                   **kw), seed)
        with da.Engine(da.make_problem(t, isf, 1e-2 * isf, freq, 1.35, **kw)) as e:
            g = e.run(seed, N, 0.0)
        assert g["rng"] == o["rng"]
        for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
            assert gc.bit_diff(g[k], o[k]) is None, (k, gc.bit_diff(g[k], o[k]))
