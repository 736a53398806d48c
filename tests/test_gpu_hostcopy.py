"""Whole fields to and from the device in chunks: sizes of one chunk, of a ragged last chunk, and of
more than the pinned ring holds.  A multi-field FP64 solver keeps the arrays themselves, so reading
back what was set is exact, repeated and from several threads; the transform is compared with
numpy's to 1e-13 * sqrt(N) of the largest value.
"""
import threading

import numpy as np
import pytest

import gopf_amd as G

pytestmark = pytest.mark.gpu


def solver(dims):
    m = G.Model()
    n = int(np.prod(dims))
    for f in ("conc", "etaa"):
        m.AddField(f, np.zeros(n))
    m.AddScalar("kap", 0.1)
    m.AddEquation("dconc/dt = kap*LAP conc")
    m.AddEquation("detaa/dt = kap*LAP etaa")
    m.Init()
    return G.Solver(m, dims, 0.1)


# one copy, the largest of them (3.5 MB) and a little more, chunks on three threads and on several, each
# with a ragged last one; 33 MB, past the ring
@pytest.mark.parametrize("dims", [[16, 16], [128, 128], [112, 160], [400, 250], [500, 512], [448, 1024], [500, 1000],
                                  [800, 768], [160, 160, 160]])
def test_round_trip_exact(dims):
    print("round trip", dims, flush=True)
    s = solver(dims)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    for _ in range(2):
        x = {f: rng.standard_normal(n) for f in ("conc", "etaa")}
        for f, v in x.items():
            s.SetField(f, v)
        for f, v in x.items():
            assert np.array_equal(np.asarray(s.Field(f)).real.ravel(), v)


@pytest.mark.parametrize("dims", [[200, 640], [1000, 640]])  # one copy; chunks on four threads each
def test_threads(dims):
    n = int(np.prod(dims))
    solvers = [solver(dims) for _ in range(4)]
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for _ in range(3):
            x = rng.standard_normal(n)
            solvers[k].SetField("etaa", x)
            if not np.array_equal(np.asarray(solvers[k].Field("etaa")).real.ravel(), x):
                bad.append(k)

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


@pytest.mark.parametrize("precision, tol", [("fp64", 1e-13), ("fp32", 2e-6)])
@pytest.mark.parametrize("dims", [[96, 96], [320, 400], [580, 400], [96, 100, 128]])
def test_transform(dims, precision, tol):
    print("transform", dims, precision, flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(3)
    ft = G.FourierTransform(dims, precision=precision)
    for _ in range(2):
        x = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        got = x.copy()
        ft.FFT(got)
        ref = np.fft.fftn(x.reshape(dims)).ravel()
        scale = np.sqrt(n) if precision == "fp64" else 1.0
        assert np.abs(got - ref).max() < tol * scale * np.abs(ref).max()
