"""The adjoint's reverse pass (forward, multipliers with the scalars' sums, inverse of P and Q along
the last axis) against the oracle's reverse mode at lengths of every count of elements per thread, odd
and uncompiled ones, one line per tile, 3D, with and without the source's scalars, and segments
shorter than the run.  FP64: loss 1e-12, gradients 1e-10 relative (the path's bars)."""
import numpy as np
import pytest

import gopf_amd as G
from gopf_amd import workloads as W
from oracle import parser as P
from oracle.engine import OracleSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wanted", [["mk"], ["m2", "m4", "mk"]], ids=["implicit", "all"])
@pytest.mark.parametrize("dims", [[100, 12], [24, 20], [9, 15], [400, 8], [512, 6], [11, 64], [20, 20, 20], [9, 9, 9]])
def test_adjoint_sizes(oracle_lib, dims, wanted):
    n = int(np.prod(dims))
    c0, tgt, scal = W.ch_initial(5, n), W.ch_initial(6, n), W.ch_scalars(1.0, 1.0)
    pm, om = G.Model(), P.Model()
    pm.AddField("conc", c0)
    om.add_field("conc", n)
    for k, v in scal.items():
        pm.AddScalar(k, v)
        om.add_scalar(k, v)
    pm.AddEquation(W.CH_EQUATION)
    om.add_equation(W.CH_EQUATION)
    pm.Init()
    om.init()
    Jo, go, gso = OracleSolver(om, dims, {"conc": c0}, 0.05).adjoint(11, tgt, wanted)
    s = G.Solver(pm, dims, 0.05)
    for _ in range(2):   # the second run finds the storage of the first
        s.SetField(0, c0)
        J, g0, gs = s.Adjoint(11, tgt, wanted, checkpoint_every=4)
        assert abs(J - Jo) <= 1e-12 * abs(Jo)
        assert np.abs(g0 - go).max() <= 1e-10 * np.abs(go).max()
        for k in wanted:
            assert abs(gs[k] - gso[k]) <= 1e-10 * abs(gso[k]), (k, gs[k], gso[k])
