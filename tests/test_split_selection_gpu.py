"""The mixed split loop's selection where few timeslices meet many slices: each
workgroup adds a member's slices in runs, one after the other, of no more runs
than the slices fill.  A generation's other kernels read K and the genomes, so
that fewer timeslices never take longer by more than the runs do; twice is
allowed for.
"""
import numpy as np
import pytest

import deac_amd as da

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,G", [(8, 4096), (33, 8000)])
@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
def test_few_timeslices_take_no_longer(P, G, precision):
    us = {}
    for T in (2, 8, 33, 257):
        print(f"[gpu] split selection P={P} G={G} T={T} {precision}", flush=True)
        tau = np.linspace(0.0, 0.37, T)
        isf = 0.55 * np.exp(-1.7 * tau) + 0.45 * np.exp(-0.4 * tau)
        p = da.make_problem(tau, isf, 1e-2 * isf, da.frequency_grid(G, 48.0), 1.35, population_size=P)
        with da.Engine(p) as e:
            e.run(5, 40, 0.0, precision=precision)
            us[T] = min(e.run(5, 150, 0.0, precision=precision)["loop_ms"] for _ in range(3)) / 149 * 1e3
    assert max(us.values()) < 2.0 * us[257], us
