"""FFT lengths over the radices of the passes (2 .. 13, 15, 16; one to four
stages, remainders of lines per workgroup) and the wide workgroups that long
strided axes take, against the definition evaluated by numpy in FP64
(separable products over a few nodes).

Tolerances: FP64, m = 8 on twice oversampled grids, 1e-12, as in the other
parity tests (window error 1e-14); FP32, m = 4, 1e-5.
"""
import numpy as np
import pytest

import nfft_amd as nf
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT
TOL = {"double": 1e-12, "single": 1e-5}


def errors(N, n, precision, M=48):
    p = nf.Plan(N, M, n=n, m=8 if precision == "double" else 4, flags=FLAGS, precision=precision)
    try:
        p.x[:] = W.uniform(M, len(N), seed=len(N))
        p.precompute()
        x = p.x.astype(np.float64).reshape(M, len(N)).copy()
        p.f_hat[:] = W.complex_normal(int(np.prod(N)), seed=5)
        fh = p.f_hat.astype(np.complex128).reshape(N).copy()
        p.trafo()
        f = p.f.astype(np.complex128).copy()
        p.f[:] = W.complex_normal(M, seed=6)
        y = p.f.astype(np.complex128).copy()
        p.adjoint()
        h = p.f_hat.astype(np.complex128).reshape(N).copy()
    finally:
        p.finalize()
    E = [np.exp(-2j * np.pi * np.outer(x[:, t], np.arange(N[t]) - N[t] // 2)) for t in range(len(N))]
    z = fh
    if len(N) == 1:
        f0, h0 = E[0] @ fh, E[0].conj().T @ y
    else:
        f0 = ((E[0] @ z) * E[1]).sum(1)
        h0 = (E[0].conj() * y[:, None]).T @ E[1].conj()
    return (np.linalg.norm(f - f0) / np.linalg.norm(f0), np.linalg.norm(h - h0) / np.linalg.norm(h0))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("n", [20, 22, 26, 42, 48, 66, 90, 98, 128, 150, 180, 208, 240, 256, 330, 512, 768,
                               1000, 1024, 1170, 1350, 1536, 1890, 2016, 2048])
def test_single_axis(n, precision):
    et, ea = errors([n // 2], [n], precision)
    print("n=%d %s: trafo %.2e adjoint %.2e" % (n, precision, et, ea))
    assert et < TOL[precision] and ea < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2574, 3432, 3750, 4050, 4056, 4096])
def test_single_axis_longest_fp32(n):
    et, ea = errors([n // 2], [n], "single")
    print("n=%d: trafo %.2e adjoint %.2e" % (n, et, ea))
    assert et < TOL["single"] and ea < TOL["single"]


@pytest.mark.gpu
@pytest.mark.parametrize("precision,n", [("single", [600, 7200]), ("single", [1024, 4096]),
                                         ("double", [600, 7000]), ("double", [768, 4608])])
def test_wide_workgroups(precision, n):
    """Strided axes of which fewer than 64 bytes of adjacent lines fit the
    ordinary workgroup, on grids large enough to fill the CUs with wide ones;
    the last group of lines is partly empty at 7200 and 7000."""
    et, ea = errors([t // 2 for t in n], n, precision)
    print("n=%s %s: trafo %.2e adjoint %.2e" % (n, precision, et, ea))
    assert et < TOL[precision] and ea < TOL[precision]
