"""Detailed-balance folds at the edges of their blocks of 128 positions (16 units
of K): genome lengths around one, two and three blocks, the fused last element of
odd ones on a block's first position and last but one, with and without the -1st
moment.  Fused evolution and split loop against the oracle, bit for bit.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G", [120, 127, 128, 129, 136, 255, 256, 257, 383, 384, 385])
@pytest.mark.parametrize("nfm", [False, True])
def test_folds_at_block_edges(G, nfm):
    P, T = (6, 17) if G % 2 else (9, 32)
    print(f"[gpu] fold blocks P={P} T={T} G={G} nfm={nfm}", flush=True)
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    freq = ob.frequency_grid(G, 48.0)
    kw = dict(spectra_type="bdsf", use_negative_first_moment=nfm, population_size=P)
    N, seed = 30, 11
    o = ob.run(ob.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, number_of_generations=N, stop_minimum_fitness=0.0,
                               **kw), seed)
    with da.Engine(da.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, **kw)) as e:
        for split in (False, True):
            g = e.run(seed, N, 0.0, split_loop=split)
            assert g["rng"] == o["rng"]
            for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
                assert gc.bit_diff(g[k], o[k]) is None, (split, k, gc.bit_diff(g[k], o[k]))
