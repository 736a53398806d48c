"""Every compiled 2^a 3, radix-5 and radix-7 schedule (their stages join the odd factor to a power
of two by the prime-factor map) against numpy's FP64 transform, along the contiguous and the
strided axis, both ways.

Bound: a transform of length n has at most about 2 log2(n) roundings in a value's chain, each
half an ulp of values of the size of the result's root mean square: 2 eps log2(n) relative L2.

Launch layouts kept from when some of these lengths took fewer threads per line stay admissible.
"""
import numpy as np
import pytest

import gopf_amd as G
from gopf_amd import workloads as W

pytestmark = pytest.mark.gpu

LENGTHS = [12, 24, 48, 96, 192, 384, 768, 80, 100, 160, 200, 250, 320, 400, 500, 640, 800, 1000, 1280, 1600, 2000,
           2560, 112, 224, 448, 896]


@pytest.mark.parametrize("precision,eps", [("fp64", 2.0 ** -52), ("fp32", 2.0 ** -23)])
@pytest.mark.parametrize("n", LENGTHS)
def test_compiled_schedules_match_numpy(n, precision, eps):
    rng = np.random.default_rng(n)
    for dims in ([3, n], [n, 5]):
        x = rng.standard_normal(dims) + 1j * rng.standard_normal(dims)
        ft = G.FourierTransform(dims, precision=precision)
        tol = 2.0 * eps * np.log2(n * min(dims))
        for call, ref in ((ft.FFT, np.fft.fftn(x)), (ft.IFFT, np.fft.ifftn(x) * x.size)):
            got = call(x.reshape(-1).copy()).reshape(dims)
            assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), (dims, precision)


def ch_model(n):
    m = G.Model()
    m.AddField("conc", 0.5 + 0.1 * (np.random.default_rng(1).random(n) - 0.5))
    for k, v in W.ch_scalars(1.0, 1.0).items():
        m.AddScalar(k, v)
    m.AddEquation(W.CH_EQUATION)
    m.Init()
    return m


# (side, schedule, precision, the most lines a layout could name with the lengths' former threads per
# line, lines that run now): 512 threads per block, and 160 KiB of LDS for 1000 in FP64
@pytest.mark.parametrize("side,schedule,precision,named,now", [
    (500, 0, "fp64", 16, 8), (500, 1, "fp32", 16, 8), (1000, 0, "fp32", 8, 4), (1000, 0, "fp64", 4, 4),
    (384, 0, "fp32", 32, 16), (768, 0, "fp32", 16, 8), (200, 0, "fp32", 32, 16), (256, 0, "fp32", 32, 32)])
def test_layouts_stored_for_fewer_threads_per_line(side, schedule, precision, named, now):
    dims = [side, side]
    m = ch_model(side * side)
    a, b = (G.Solver(m, dims, 0.05, precision=precision) for _ in range(2))
    layout = dict(zip(G.Solver.TUNING_KEYS, (named, 0, 4, 0, "y", schedule, 1, 1, 0, 0)))
    a.SetTuning(layout)
    assert a.Tuning()["rows_fused"] == now
    with pytest.raises(G.GpfError, match="not admissible"):
        b.SetTuning({**layout, "rows_fused": 2 * named})
    for s in (a, b):
        s.Propagate(3)
    x, y = a.Field(0).real, b.Field(0).real
    tol = 1e-13 if precision == "fp64" else 1e-6   # the row schedules differ by roundings
    assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y)
    t = G.Batch(ch_model(16), [(dims, 2)], 0.05, precision=precision, autotune=False)
    stored = {"classes": [{"rows_tw": named, "update_tw": 4, "rows_schedule": schedule}], "grouped_threads": 0}
    t.SetLayout(stored)
    assert t.Tuning()["classes"][0]["rows_tw"] == now
    stored["classes"][0]["rows_tw"] = 2 * named
    with pytest.raises(G.GpfError, match="not admissible"):
        t.SetLayout(stored)
