"""Every compiled 2^a 3, radix-5 and radix-7 schedule (their stages join the odd factor to a power
of two by the prime-factor map) against numpy's FP64 transform, along the contiguous and the
strided axis, both ways.

Bound: a transform of length n has at most about 2 log2(n) roundings in a value's chain, each
half an ulp of values of the size of the result's root mean square: 2 eps log2(n) relative L2.
"""
import numpy as np
import pytest

import gopf_amd as G

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
