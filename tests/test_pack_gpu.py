"""Operand layouts packed on the device: deac_model_isf at sizes around the
tiles of 16 timeslices and genomes and the k-blocks of every precision, and
stacks of several upload blocks, against a plain float64 product.

FP64 chains round each of L fused products once: |error| <= L 2^-53 sum|K S|,
doubled for the kernel matrix numpy builds (its exp rounds differently in the
last place).  FP32 rounds K and S to 24 bits and sums in FP32: (L + 4) 2^-24;
BF16x3 keeps 16 bits of each factor's 24 and drops lo.lo: 2^-15 on top.
"""
import numpy as np
import pytest

import deac_amd as da

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("T,G,N", [(2, 2, 1), (15, 3, 15), (16, 16, 16), (17, 33, 17), (33, 63, 65), (5, 129, 40),
                                   (64, 511, 3), (3, 70000, 40)])
def test_model_isf_sizes(T, G, N, precision):
    print(f"[gpu] model_isf T={T} G={G} N={N} {precision}", flush=True)
    tau = np.linspace(0.0, 0.37, T)
    f = np.exp(-tau)
    w = np.linspace(0.0, 30.0, G)
    beta = 1.0 / 1.35
    df = np.empty(G)
    df[1:-1] = 0.5 * (w[2:] - w[:-2])
    df[0], df[-1] = 0.5 * (w[1] - w[0]), 0.5 * (w[-1] - w[-2])
    K = np.concatenate([df * np.exp(-np.outer(tau, w)), df * np.exp(np.outer(tau - beta, w))], axis=1)
    S = np.random.default_rng(T + G + N).random((N, 2 * G))
    e, chi, _ = da.model_isf(da.make_problem(tau, f, 1e-2 * f, w, 1.35), S, precision)
    size = S @ np.abs(K.T)
    eps = {"fp64": 2 * 2 * G * 2.0 ** -53, "fp32": (2 * G + 4) * 2.0 ** -24,
           "bf16x3": (2 * G + 4) * 2.0 ** -24 + 2.0 ** -15}[precision]
    assert np.all(np.abs(e - S @ K.T) <= eps * size)
    d = (f - e) / (1e-2 * f)
    assert np.allclose(chi, np.sum(d * d, axis=1) / T, rtol=T * 2.0 ** -52)
