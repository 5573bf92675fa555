"""Initial populations drawn and normalized on the device, against the oracle.

Two-generation runs: the first statistics entry is the initial population's
fitness, and the returned random state shows where the draws ended.  Genome
lengths around the edges of the sub-streams (64 per member in the engine, 3,
6 or 12 in the batch) and of the fold's 128-position blocks; odd lengths end
each sign with a fused element.  Bar: bit-exact.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu

KEYS = ("minimum", "mean", "squared_mean", "dsf", "fitness")


@pytest.mark.parametrize("G", [2, 3, 16, 31, 32, 33, 63, 64, 65, 127, 128, 129, 192, 193, 511, 1000])
@pytest.mark.parametrize("kw", [dict(), dict(normalize=True), dict(zero_temperature=True, normalize=True),
                                dict(allow_negative=True, normalize=True), dict(spectra_type="bdsf", normalize=True)],
                         ids=["plain", "normalized", "zero_t", "negative", "bdsf"])
def test_initial_population_matches_oracle(G, kw):
    print(f"[gpu] initial population G={G} {kw}", flush=True)
    tau = np.linspace(0.0, 0.37, 7)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    freq = ob.frequency_grid(G, 48.0)

    def check(got, o, who):
        for k in KEYS:
            assert gc.bit_diff(got[k], o[k]) is None, (who, k, gc.bit_diff(got[k], o[k]))
        assert got["rng"] == o["rng"], who

    # 5 members leave padded rows; 20 and 40 take two and four member tiles in the batch
    for P, seed in ((5, 3), (20, 4), (40, 5)):
        o = ob.run(ob.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, number_of_generations=2, population_size=P,
                                   stop_minimum_fitness=0.0, **kw), seed)
        p = da.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, population_size=P, **kw)
        with da.Engine(p) as e:
            check(e.run(seed, 2, 0.0), o, ("engine", P))
            e.run(seed + 1, 4, 0.0)  # another population in the same buffers, then the first again
            check(e.run(seed, 2, 0.0), o, ("engine again", P))
        with da.Batch([p, p, p]) as b:
            check(b.run([seed + 7, seed, seed + 8], 2, 0.0)[1], o, ("batch", P))
