"""The plain path where the workgroups form the trials beside the chains, at the
edges of its ring (8 chunks of 128 positions, three feeders, two chunks of each
in flight), with the second sign beginning at every place of a chunk, against
the oracle.  Bar: bit-exact.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,T,G,kw", [
    (4, 2, 64, {}), (4, 16, 128, {}), (5, 17, 192, {}), (6, 9, 256, {}), (7, 33, 320, {}), (8, 20, 384, {}),
    (8, 33, 447, {}), (8, 5, 448, {}), (9, 16, 512, {}), (12, 7, 513, {}), (4, 40, 575, {}), (4, 3, 576, {}),
    (5, 15, 577, {}), (8, 12, 640, {}), (6, 6, 1087, {}), (4, 18, 1216, {}), (62, 65, 96, {}), (63, 20, 129, {}),
    (200, 17, 70, {}), (9, 12, 1024, dict(zero_temperature=True)), (9, 12, 1025, dict(zero_temperature=True)),
    (8, 10, 1151, dict(zero_temperature=True)), (10, 12, 321, dict(allow_negative=True)),
    (10, 12, 512, dict(normalize=True, model="hyperbolic")),
])
def test_fed_chains_match_oracle(P, T, G, kw):
    print(f"[gpu] fed chains P={P} T={T} G={G} {kw}", flush=True)
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    freq = ob.frequency_grid(G, 48.0)
    N, seed = 14, 23
    o = ob.run(ob.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, number_of_generations=N, population_size=P,
                               stop_minimum_fitness=0.0, **kw), seed)
    with da.Engine(da.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, population_size=P, **kw)) as e:
        for _ in range(2):  # the second run starts from what the first left in the buffers
            g = e.run(seed, N, 0.0)
            for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
                assert gc.bit_diff(g[k], o[k]) is None, (k, gc.bit_diff(g[k], o[k]))
            assert g["rng"] == o["rng"]
        # a stop on the way ends both forms at the same generation
        stop = float(np.nextafter(o["minimum"][6], np.inf))
        s = e.run(seed, N, stop)
        assert s["generation"] <= 6 and gc.bit_diff(s["minimum"], o["minimum"][:s["generation"] + 1]) is None
