"""Kernels at the sizes where their tiles and dispatch rules have edges,
against the CPU oracle or a float64 direct sum."""
import numpy as np
import pytest

from phyflow_amd import workloads as W
from phyflow_amd.cpp.blobs.kernels import gauss

pytestmark = pytest.mark.gpu
F64, F32C = gauss.PREC_F64, gauss.PREC_F32C


@pytest.mark.parametrize("order", [2, 11, 12, 15, 16, 19, 20, 23, 24, 31, 32, 40])
def test_multipole_orders(order, O):
    """Orders on both sides of each compiled power count.  One-box separation
    (ws = 1): the expansions of two boxes of side s at distance 2 s converge as
    (r / (2 - r))^k, r = sqrt(1/2); leaves of 0 to some 150 points."""
    n = 6001
    s = W.uniform_system(n, seed=order)
    x, y, w = s["x"] ** 2, s["y"], s["w"]  # uneven leaves
    xopt, cutoff = W.oseen_params(s["sigma"] * 0.1)
    ref = O.direct_oseen(x, y, w, x, y, xopt, cutoff)
    got = gauss.fmm2d_gpu(x, y, w, x, y, 35, xopt, cutoff, 1e-6, prec=F64, order=order, leaf=32)
    r = 0.5 ** 0.5
    assert O.rel_l2(got, ref) <= (r / (2 - r)) ** (order + 1) + 1e-12
    got = gauss.fmm2d_gpu(x, y, w, x, y, 35, xopt, cutoff, 1e-6, prec=F32C, order=order, leaf=32)
    assert O.rel_l2(got, ref) <= (r / (2 - r)) ** (order + 1) + 1e-6


@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 1025, 2047, 2048, 2049, 70001])
def test_population_control_chunks(n, O):
    """Chunks of 2048 and waves of 64 blobs at their edges; few, most, all and
    none of the blobs under the thresholds; values that are not finite stay."""
    from phyflow_amd.blobs.base.regrid import PopulationControl
    rng = np.random.default_rng(n)
    x, y = rng.random(n), rng.random(n)
    for lo, hi, total in ((-12, -3, 1e-7), (-14, -9, 1e-9), (-7, -3, 1e-8), (-30, -20, 1.0)):
        w = 10.0 ** rng.uniform(lo, hi, n) * rng.choice([-1.0, 1.0], n)
        got = PopulationControl(x, y, w, 1e-8, total)
        ref = O.population_control(x, y, w, 1e-8, total)
        for a, b in zip(got, ref[:3]):
            assert np.array_equal(a, b)
    w = 10.0 ** rng.uniform(-12, -3, n)
    w[n // 2] = np.nan
    w[n // 3] = np.inf
    got = PopulationControl(x, y, w, 1e-8, 1e300)
    assert np.array_equal(got[0], x[~(np.abs(w) < 1e-8)])
