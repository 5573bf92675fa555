"""Two engines at once, from two host threads: their persistent workgroups share the
CUs, and each run is what it is alone.
"""
import threading

import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc

pytestmark = pytest.mark.gpu


# 248 workgroups each (the most a handle takes), and one of them with trials beside the chains
@pytest.mark.parametrize("shapes", [((512, 65, 96), (512, 65, 96)), ((62, 65, 600), (512, 33, 200))])
def test_two_engines_at_once(shapes):
    print(f"[gpu] two engines {shapes}", flush=True)

    def engine(P, T, G):
        tau = np.linspace(0.0, 0.37, T)
        isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
        return da.Engine(da.make_problem(tau, isf, 1e-2 * isf, da.frequency_grid(G, 48.0), 1.35, population_size=P))

    engines = [engine(*s) for s in shapes]
    try:
        alone = [e.run(3 + i, 200, 0.0) for i, e in enumerate(engines)]
        start, got = threading.Barrier(2), [[], []]

        def work(i):
            start.wait()
            for _ in range(5):
                got[i].append(engines[i].run(3 + i, 200, 0.0))

        threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        for e in engines:
            e.close()
    for i in (0, 1):
        assert len(got[i]) == 5
        for g in got[i]:
            assert g["rng"] == alone[i]["rng"]
            for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
                assert gc.bit_diff(g[k], alone[i][k]) is None, (i, k)
