"""The fused step with tabulated update multipliers against the oracle, where the table, its chunked
loads and the untuned launch layout can go wrong: lines of every count of elements per thread,
tiles with one line or with lines past the end, an axis of two points, a filter set after the first
steps (the table is rebuilt), the energy monitor, a mean that moves (k = 0 from the table).
FP64 to 1e-10 max relative, FP32 to 1e-5 relative L2.
"""
import numpy as np
import pytest

import gopf_amd as G
from gopf_amd import workloads as W
from oracle import engine as E
from oracle import parser as P

pytestmark = pytest.mark.gpu

AC = "dconc/dt = m2*conc - m4*conc^3 + mk*LAP conc"     # not conserved: the mean moves


def models(dims, eq, seed):
    n = int(np.prod(dims))
    c0 = 0.5 + 0.1 * (np.random.default_rng(seed).random(n) - 0.5)
    pm, om = G.Model(), P.Model()
    pm.AddField("conc", c0)
    om.add_field("conc", n)
    for k, v in W.ch_scalars(1.0, 1.0).items():
        pm.AddScalar(k, v)
        om.add_scalar(k, v)
    pm.AddEquation(eq)
    om.add_equation(eq)
    pm.Init()
    om.init()
    return pm, om, c0


def close(got, ref, precision):
    if precision == "fp64":
        return np.abs(got - ref).max() <= 1e-10 * np.abs(ref).max()
    return np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("eq", [W.CH_EQUATION, AC], ids=["ch", "ac"])
@pytest.mark.parametrize("dims", [[2, 16], [100, 12], [112, 20], [400, 10], [250, 64], [512, 30], [33, 50], [768, 8],
                                  [448, 10], [20, 20, 20], [24, 24, 24], [9, 9, 9]])
def test_fused_step_with_table(dims, eq, precision):
    pm, om, c0 = models(dims, eq, 3)
    s = G.Solver(pm, dims, 0.05, precision=precision)
    assert s.fused
    o = E.OracleSolver(om, dims, {"conc": c0}, 0.05)
    s.MonitorEnergy(W.CH_BULK_POLY, 1.0)
    s.Propagate(13)
    o.stepper_propagate(13)
    assert close(s.Field(0).real, o.field("conc").real, precision)
    energy, mass = s.EnergySeries()
    assert energy.size == 13 and abs(mass[0] - c0.sum()) <= 1e-6 * abs(c0.sum())
    # a filter from here on
    s.SetFilter(G.NewVandeven(4))
    f = E.OracleSolver(om, dims, {"conc": o.field("conc").real}, 0.05, filter_order=4)
    s.Propagate(5)
    f.stepper_propagate(5)
    assert close(s.Field(0).real, f.field("conc").real, precision)


@pytest.mark.parametrize("precision,bound", [("fp64", 1e-12), ("fp32", 1e-6)])
@pytest.mark.parametrize("dims", [[448, 448], [128, 128, 128]])
def test_monitor_leaves_the_fields_alone(dims, precision, bound):
    """The monitored passes have their own launch layout (blocks of up to 256 threads): the fields
    are those of the unmonitored run, and a slot is the energy of the step's initial state."""
    pm, _, _ = models(dims, W.CH_EQUATION, 4)
    a, b = (G.Solver(pm, dims, 0.05, precision=precision) for _ in range(2))
    a.MonitorEnergy(W.CH_BULK_POLY, 1.0)
    want = []
    for _ in range(3):
        want.append(b.Energy(0, W.CH_BULK_POLY, 1.0))
        b.Propagate(1)
    a.Propagate(3)
    energy, mass = a.EnergySeries()
    x, y = a.Field(0).real, b.Field(0).real
    if dims == [448, 448] and precision == "fp64":  # computed against tabulated multipliers
        assert np.abs(x - y).max() <= 1e-14 * np.abs(y).max()
    else:
        assert np.array_equal(x, y)
    for k in range(3):
        assert abs(energy[k] - want[k][0]) <= bound * abs(want[k][0]), k
        assert abs(mass[k] - want[k][1]) <= bound * abs(want[k][1]), k


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_table_follows_the_update_axis(precision):
    """A layout with another update axis, set after the table was built for the first one, gives the
    run that has it from the start, bit for bit."""
    dims = [20, 20, 20]
    pm, _, _ = models(dims, W.CH_EQUATION, 5)
    layout = dict(zip(G.Solver.TUNING_KEYS, (8, 8, 8, 8, "z", 0, 1, 1, 0, 0)))
    for axis, other in (("z", "y"), ("y", "z")):
        a, b = (G.Solver(pm, dims, 0.05, precision=precision) for _ in range(2))
        a.SetTuning({**layout, "update_axis": axis})
        b.SetTuning({**layout, "update_axis": other})
        b.Prepare(20)
        b.SetTuning({**layout, "update_axis": axis})
        for s in (a, b):
            s.Propagate(20)
        assert np.array_equal(a.Field(0).real, b.Field(0).real), axis
