"""Results brought back in pieces: best rows of more instances than one piece
(2^22 doubles) holds, and histories on both sides of the length from which one is
copied by itself (2^17 doubles for the three).  Bar: the oracle's, bit for bit.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


def problem(module, T, G, **kw):
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    return module.make_problem(tau, isf, 1e-2 * isf, module.frequency_grid(G, 48.0), 1.35, population_size=4, **kw)


def same(got, want):
    assert got["generation"] == want["generation"] and got["rng"] == want["rng"]
    for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
        assert gc.bit_diff(got[k], want[k]) is None, (k, gc.bit_diff(got[k], want[k]))


def test_rows_of_many_instances():
    G, n, N = 8192, 260, 4  # 256 rows of 2 x 8192 fill a piece
    print(f"[gpu] readback of {n} rows", flush=True)
    with da.Batch([problem(da, 3, G)] * n) as b:
        outs = b.run(list(range(1, n + 1)), N, 0.0)
    for i in (0, 1, 255, 256, 259):
        same(outs[i], ob.run(problem(ob, 3, G, number_of_generations=N, stop_minimum_fitness=0.0), i + 1))


@pytest.mark.parametrize("N", [43690, 43691, 200000])
def test_histories_of_stopped_runs(N):
    print(f"[gpu] histories of {N}", flush=True)
    stop = float(ob.run(problem(ob, 5, 9, number_of_generations=40, stop_minimum_fitness=0.0), 1)["minimum"][30])
    lengths = [N, 300, N]
    with da.Batch([problem(da, 5, 9)] * 3) as b, da.Engine(problem(da, 5, 9)) as e:
        outs = b.run([1, 2, 3], lengths, [stop, 0.0, stop])
        alone = e.run(1, N, stop)
    for seed, length, threshold, got in zip((1, 2, 3), lengths, (stop, 0.0, stop), outs):
        same(got, ob.run(problem(ob, 5, 9, number_of_generations=length, stop_minimum_fitness=threshold), seed))
    same(alone, outs[0])
