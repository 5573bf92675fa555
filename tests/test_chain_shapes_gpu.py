"""The plain path's chains and selection at the edges of their tiles, against
the oracle: genome lengths around one, two and three 128-position chunks (the
K ring holds two), timeslices around the 16-row tiles, members around the
groups of four, both forms of the selection (repeated by every workgroup while
P x T is at most 4096, by one wavefront per member above).  Bar: bit-exact.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc
import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,T,G,kw", [
    (4, 2, 2, {}), (5, 15, 64, {}), (7, 16, 65, {}), (8, 17, 63, {}), (4, 33, 128, {}), (9, 31, 129, {}),
    (6, 5, 191, {}), (12, 48, 192, {}), (8, 65, 193, {}), (4, 3, 256, {}), (13, 64, 321, {}),
    (8, 20, 127, dict(zero_temperature=True)), (8, 20, 385, dict(zero_temperature=True)),
    (63, 65, 70, {}), (64, 64, 70, {}), (64, 65, 70, {}), (65, 63, 40, dict(normalize=True)), (130, 31, 33, {}),
    # bdsf folds: chunks of 32 positions, odd lengths fuse the last, both forms of the -1st moment's sum
    (4, 2, 2, dict(spectra_type="bdsf")), (6, 17, 31, dict(spectra_type="bdsf")),
    (5, 16, 32, dict(spectra_type="bdsf", use_negative_first_moment=True)),
    (9, 33, 33, dict(spectra_type="bdsf", use_negative_first_moment=True)),
    (8, 65, 127, dict(spectra_type="bdsf", use_negative_first_moment=True, normalize=True)),
    (13, 18, 257, dict(spectra_type="bdsf", model="hyperbolic")),
    (70, 66, 129, dict(spectra_type="bdsf", use_negative_first_moment=True)),
    (66, 600, 40, dict(spectra_type="bdsf", use_negative_first_moment=True)),
    (5, 1101, 21, dict(spectra_type="bdsf", use_negative_first_moment=True)),
    (130, 33, 33, {}), (10, 20, 255, dict(first_moment=1.5)),
    (6, 20, 64, dict(normalize=True, third_moment=900.0, third_moment_error=9.0)),
    (5, 9, 193, dict(normalize=True, renormalize=True, first_moment=1.5, third_moment=900.0, third_moment_error=9.0)),
    (300, 7, 65, dict(normalize=True, renormalize=True, first_moment=1.5)),
    (11, 18, 129, dict(normalize=True, renormalize=True, zero_temperature=True)), (512, 8, 20, {}), (5, 1100, 20, {}), (300, 2, 12, dict(allow_negative=True)),
])
def test_plain_path_shapes_match_oracle(P, T, G, kw):
    print(f"[gpu] plain path P={P} T={T} G={G} {kw}", flush=True)
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    freq = ob.frequency_grid(G, 48.0)
    N, seed = 30, 11
    o = ob.run(ob.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, number_of_generations=N, population_size=P,
                               stop_minimum_fitness=0.0, **kw), seed)
    with da.Engine(da.make_problem(tau, isf, 1e-2 * isf, freq, 1.35, population_size=P, **kw)) as e:
        g = e.run(seed, N, 0.0)
        if "bdsf" in kw.values():
            split = e.run(seed, N, 0.0, split_loop=True)
            assert gc.bit_diff(g["minimum"], split["minimum"]) is None and g["rng"] == split["rng"]
    for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
        assert gc.bit_diff(g[k], o[k]) is None, (k, gc.bit_diff(g[k], o[k]))
    assert g["rng"] == o["rng"]
