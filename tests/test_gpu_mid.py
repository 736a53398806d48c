"""The general path's middle pass (forward, stage, inverse along the last axis in one launch)
against the oracle: lengths with and without a compiled schedule, one line term and several, terms
with a LAP power, a constant term, a field's own and another field's spectrum as a term, filter
(a volume constraint's multiplier: test_gpu_terms.py).
FP64 to the path's parity bound (1e-10 max relative), FP32 to 1e-5 relative L2.
"""
import numpy as np
import pytest

import gopf_amd as G
from oracle import engine as E
from oracle import parser as P

pytestmark = pytest.mark.gpu

MODELS = {
    # one line term per field (the precipitate's form)
    "single": (["alpha", "beta"], {"kap": 0.2}, ["dalpha/dt = PAA + kap*LAP alpha", "dbeta/dt = PBB + kap*LAP beta"],
               {"PAA": [(0.3, {"alpha": 1, "beta": 0}), (-0.2, {"alpha": 2, "beta": 1})],
                "PBB": [(-0.4, {"alpha": 0, "beta": 1}), (0.1, {"alpha": 1, "beta": 2})]}),
    # several line terms with LAP powers
    "lap": (["conc", "etaa"], {"m2": 0.4, "kap": 0.3, "gam": 0.05},
            ["dconc/dt = m2*LAP conc^2 - m2*LAP conc^3 - kap*LAP^2 conc", "detaa/dt = PEE - gam*etaa + kap*LAP etaa"],
            {"PEE": [(0.2, {"conc": 1, "etaa": 1})]}),
    # another field's spectrum, and a field's own, as explicit terms
    "cross": (["aaa", "bbb"], {"kap": 0.2, "cpl": 0.3}, ["daaa/dt = cpl*bbb + PAA + kap*LAP aaa",
                                                         "dbbb/dt = cpl*aaa - PBB + kap*LAP bbb"],
              {"PAA": [(0.1, {"aaa": 2, "bbb": 0})], "PBB": [(0.2, {"aaa": 0, "bbb": 3})]}),
    # a bare scalar: the same value at every k, without a brick
    "constant": (["aaa", "bbb"], {"kap": 0.2, "src": 0.3}, ["daaa/dt = src + PAA + kap*LAP aaa", "dbbb/dt = src - PBB"],
                 {"PAA": [(0.1, {"aaa": 2, "bbb": 0})], "PBB": [(0.2, {"aaa": 0, "bbb": 3})]}),
}


def pair(name, dims, seed):
    fields, scal, eqs, polys = MODELS[name]
    n = int(np.prod(dims))
    rng = np.random.default_rng(seed)
    pm, om, init = G.Model(), P.Model(), {}
    for f in fields:
        init[f] = 0.4 + 0.2 * rng.random(n)
        pm.AddField(f, init[f])
        om.add_field(f, n)
    for k, v in scal.items():
        pm.AddScalar(k, v)
        om.add_scalar(k, v)
    for k, poly in polys.items():
        pm.RegisterPolynomial(k, poly)
        om.register_polynomial(k, poly)
    for e in eqs:
        pm.AddEquation(e)
        om.add_equation(e)
    pm.Init()
    om.init()
    return pm, om, init


# the filter enters through the factor table only: one model covers it
@pytest.mark.parametrize("name,filter_order", [(n, 0) for n in sorted(MODELS)] + [("single", 4)])
@pytest.mark.parametrize("dims", [[9, 15], [2, 16], [40, 24], [100, 12], [12, 400], [11, 11, 11], [24, 24, 24]])
@pytest.mark.parametrize("stepper", ["euler", "rk4"])
def test_middle_pass_matches_oracle(name, filter_order, stepper, dims):
    pm, om, init = pair(name, dims, 5)
    o = E.OracleSolver(om, dims, init, 0.02, stepper, filter_order=filter_order)
    o.solver_propagate(6)
    for precision, bound in (("fp64", 1e-10), ("fp32", 1e-5)):
        s = G.Solver(pm, dims, 0.02, stepper=stepper, precision=precision, filter_order=filter_order)
        s.Propagate(6)
        for f in init:
            got, ref = s.Field(f).real, o.field(f).real
            if precision == "fp64":
                assert np.abs(got - ref).max() <= bound * np.abs(ref).max(), (precision, f)
            else:
                assert np.linalg.norm(got - ref) <= bound * np.linalg.norm(ref), (precision, f)
