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
