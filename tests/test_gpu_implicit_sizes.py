"""ImplicitEuler through the middle pass at the sizes where its row pass and the Arnoldi sweeps can
go wrong: odd and uncompiled lengths, one to a few hundred reduction blocks, one and two fields,
every stencil, a restart shorter than the Krylov space, 3D.

Both sides solve the residual to 1e-12 in max norm; a step's root is then within a few 1e-12 over
the smallest singular value of the Jacobian (above 1/2 here), so the fields agree to 1e-9.
"""
import numpy as np
import pytest

import gopf_amd as G
from oracle import parser as P
from oracle.implicit import ImplicitEulerOracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,nfields,stencil,restart", [
    ([9, 15], 1, 6, 30), ([33, 20], 1, 2, 30), ([16, 100], 1, 4, 3), ([60, 48], 2, 6, 30), ([256, 16], 1, 8, 30),
    ([7, 9], 2, 1, 30), ([10, 10, 10], 1, 6, 4), ([12, 12, 12], 2, 6, 30), ([320, 250], 1, 6, 30)])
def test_implicit_sizes(dims, nfields, stencil, restart):
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    names = ["aaa", "bbb"][:nfields]
    fields = {f: 0.5 + 0.1 * (rng.random(n) - 0.5) for f in names}
    eqs = ["daaa/dt = m2*LAP aaa - m6*LAP aaa^2 + m4*LAP aaa^3 - mk*LAP^2 aaa"]
    polys = {}
    if nfields == 2:
        eqs.append("dbbb/dt = MIX + mk*LAP bbb")
        polys["MIX"] = [(0.3, {"aaa": 1, "bbb": 1}), (-0.2, {"aaa": 0, "bbb": 2})]
    pm, om = G.Model(), P.Model()
    for f, x in fields.items():
        pm.AddField(f, x)
        om.add_field(f, n)
    for k, v in {"m2": 2.0, "m6": 6.0, "m4": 4.0, "mk": 1.0}.items():
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
    s = G.Solver(pm, dims, 0.1, stepper="implicitEuler")
    # a forward difference (stencil 1) is off by 1e-3 per Newton update: more of them, same root
    s.SetNewtonKrylov(Tol=1e-12, Stencil=stencil, Restart=restart)
    o = ImplicitEulerOracle(om, dims, {k: v.astype(complex) for k, v in fields.items()}, 0.1, f_tol=1e-12)
    for _ in range(2):
        s.Propagate(1)
        o.step()
        assert s.NewtonStats()["converged"]
    for f in names:
        ref = o.field(f).real
        assert np.abs(s.Field(f).real - ref).max() <= 1e-9 * np.abs(ref).max(), f


def test_long_vectors():
    """Vectors of more than half a million values take more than 256 reduction blocks: two
    independent fields of one equation and start, solved together, against one alone (256 blocks)."""
    dims = [448, 640]
    n = int(np.prod(dims))
    x = 0.5 + 0.1 * (np.random.default_rng(8).random(n) - 0.5)
    got = []
    for names in (["aaa"], ["aaa", "bbb"]):
        m = G.Model()
        for f in names:
            m.AddField(f, x)
        for k, v in {"m2": 2.0, "m6": 6.0, "m4": 4.0, "mk": 1.0}.items():
            m.AddScalar(k, v)
        for f in names:
            m.AddEquation(f"d{f}/dt = m2*LAP {f} - m6*LAP {f}^2 + m4*LAP {f}^3 - mk*LAP^2 {f}")
        m.Init()
        s = G.Solver(m, dims, 0.1, stepper="implicitEuler")
        s.SetNewtonKrylov(Tol=1e-12)
        s.Propagate(2)
        assert s.NewtonStats()["converged"]
        got += [s.Field(f).real for f in names]
    for g in got[1:]:
        assert np.abs(g - got[0]).max() <= 1e-9 * np.abs(got[0]).max()
