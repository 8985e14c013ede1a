"""FP32 transforms of data towards the ends of FP32's exponent range.  Scaling
by a power of two is exact, so a trafo or adjoint of scaled data is the scaled
result, bit for bit, unless something leaves the normal range.  At 2^100 (2^27
below the largest value) nothing does.  At 2^-104 the grid, whose values the
deconvolution factors bring to 2^-124 and more, and the results stay in it;
products with the window's smallest values do not, and are off by half a step
of 2^-149: 14^3 of them are less than 2e-8 of a result of 2^-110.  A trafo with
m = 3 and more has factors above 2^-12, and meets that bound at 2^-116 too.
3-D sets of some and of several nodes per cell, and 2-D ones."""
import numpy as np
import pytest

import nfft_amd as nf
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("N,n,M", [([10, 12, 9], [20, 24, 18], 9000), ([10, 12, 9], [20, 24, 18], 60000),
                                   ([20, 30], [40, 60], 9000)],
                         ids=["3d", "3d-dense", "2d"])
def test_scaled_data(N, n, M, m):
    NN = int(np.prod(N))
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision="single", fftw_flags=nf.FFTW_ESTIMATE)
    try:
        p.x[:] = W.uniform(M, len(N), seed=m)
        p.precompute()
        fh, y = W.complex_normal(NN, seed=3).astype(np.complex64), W.complex_normal(M, seed=4).astype(np.complex64)

        def run(s):
            p.f_hat[:] = fh * np.float32(s)
            p.trafo()
            f = p.f.astype(np.complex128) / s
            p.f[:] = y * np.float32(s)
            p.adjoint()
            return f, p.f_hat.astype(np.complex128) / s

        one, small, large, tiny = run(1.0), run(2.0 ** -104), run(2.0 ** 100), run(2.0 ** -116)
    finally:
        p.finalize()
    off = [np.linalg.norm(b - a) / np.linalg.norm(a) for a, b in zip(one, small)]
    if m > 2:
        off.append(np.linalg.norm(tiny[0] - one[0]) / np.linalg.norm(one[0]))
    print("m=%d: trafo, adjoint at 2^-104, trafo at 2^-116:" % m, *("%.2e" % v for v in off))
    assert np.array_equal(one[0], large[0]) and np.array_equal(one[1], large[1])
    assert max(off) <= 2e-8
