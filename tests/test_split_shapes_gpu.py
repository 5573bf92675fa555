"""The split loop's kernels at the edges of their tiles: members around the 16
of a tile and the 1 to 4 tiles of a wavefront, timeslices around the 16-row
tiles and the 4096 residuals of a selection's window, genomes around the
128-position blocks of the trials and operands.

At FP64 the split loop is the fused kernel bit for bit.  At FP32 and BF16x3 the
statistics after one generation, whose trials come from the same population,
differ from FP64's by the contraction's rounding: each model ISF is a sum of at
most 2 G positive terms in slices of at least 8 k-blocks, off by less than
2 G 2^-24 = 2^-13 of itself at these sizes (BF16x3's dropped terms are below
2^-16 of it), and the data lie 30% or more from it, so that chi^2 and its mean
are off by less than 2 (1/0.3 + 1) 2^-13 = 1.1e-3 and its mean square by twice
that.  An operand or slice out of place moves them by order 1.
"""
import numpy as np
import pytest

import deac_amd as da
import golden_cases as gc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,T,G,kw", [
    (4, 2, 2, {}), (5, 15, 63, {}), (15, 16, 64, {}), (16, 17, 65, {}), (17, 33, 127, {}), (33, 31, 128, {}),
    (48, 32, 129, {}), (49, 65, 191, {}), (64, 48, 193, {}), (65, 18, 257, {}), (130, 9, 320, {}),
    (20, 40, 201, dict(zero_temperature=True)), (9, 20, 333, dict(spectra_type="bdsf")),
    (18, 20, 100, dict(normalize=True, renormalize=True)),
    (5, 4096, 12, {}), (5, 4097, 12, {}), (4, 4500, 9, {}),
])
def test_split_loop_shapes(P, T, G, kw):
    print(f"[gpu] split loop P={P} T={T} G={G} {kw}", flush=True)
    tau = np.linspace(0.0, 0.37, T)
    isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
    far = 100.0 * isf  # data that no member of the first generations comes near
    norm = kw.get("normalize", False)
    p = da.make_problem(tau, isf if norm else far, 1e-2 * isf, da.frequency_grid(G, 48.0), 1.35, population_size=P, **kw)
    with da.Engine(p) as e:
        fused = e.run(5, 20, 0.0)
        split = e.run(5, 20, 0.0, split_loop=True)
        for k in ("minimum", "mean", "squared_mean", "dsf", "fitness"):
            assert gc.bit_diff(fused[k], split[k]) is None, k
        assert fused["rng"] == split["rng"]
        for precision in ("fp32", "bf16x3"):
            low = e.run(5, 20, 0.0, precision=precision)
            assert low["rng"] == fused["rng"]
            for k, tol in (("minimum", 1.1e-3), ("mean", 1.1e-3), ("squared_mean", 2.2e-3)):
                for g in (0, 1):
                    assert abs(low[k][g] / fused[k][g] - 1.0) < tol, (precision, k, g, low[k][g], fused[k][g])
            assert np.all(np.diff(low["minimum"]) <= 0.0)
