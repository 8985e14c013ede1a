"""Fewer and more FFT lines per workgroup than by default (what FFTW_MEASURE
plans time), also along the long strided axes that wide workgroups take: the
values do not depend on it, bit for bit (a line's butterflies are the same
whichever workgroup runs it)."""
import numpy as np
import pytest

import nfft_amd as nf
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT


def run(N, n, precision):
    p = nf.Plan(N, 40, n=n, m=4, flags=FLAGS, precision=precision, fftw_flags=nf.FFTW_ESTIMATE)
    try:
        p.x[:] = W.uniform(40, len(N), seed=1)
        p.precompute()
        p.f_hat[:] = W.complex_normal(int(np.prod(N)), seed=2)
        p.trafo()
        return p.f.copy()
    finally:
        p.finalize()


@pytest.mark.gpu
@pytest.mark.parametrize("precision,n", [("single", [600, 7200]), ("single", [4096, 512]), ("single", [1 << 22]),
                                         ("double", [600, 7000]), ("double", [96, 100, 90])])
def test_lines_per_workgroup(precision, n, monkeypatch):
    N = [t // 2 for t in n]
    ref = run(N, n, precision)
    for k in (-4, -2, -1, 1, 3):
        monkeypatch.setenv("NFFT_HIP_FFT_LINES", str(k))
        assert np.array_equal(run(N, n, precision), ref), k
