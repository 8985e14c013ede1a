"""3-D plans whose first axis is the shortest that the fast path takes
(n0 = 2m + 3) and a little longer, with nodes in its last cells, against the
FP64 oracle.

Tolerances as for the other 3-D kernels: FP64 1e-12, FP32 2e-6."""
import numpy as np
import pytest

import nfft_amd as nf
import oracle as O
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT
TOL = {"double": 1e-12, "single": 2e-6}


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("more", [0, 1, 2])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6])
def test_short_first_axis(m, more, precision):
    n = [2 * m + 3 + more, 20, 18]
    N = [m + 1 + more // 2, 10, 9]
    x = np.concatenate([W.uniform(400, 3, seed=m), np.full((5, 3), 0.4999), np.full((5, 3), -0.5),
                        W.uniform(90, 3, seed=9) * [0.0, 1.0, 1.0] + [0.49, 0, 0]])
    M, NN = x.shape[0], int(np.prod(N))
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=nf.FFTW_ESTIMATE)
    try:
        p.x[:] = x
        p.precompute()
        xr = p.x.astype(np.float64).copy()
        p.f_hat[:] = W.complex_normal(NN, seed=3)
        fh = p.f_hat.astype(np.complex128).copy()
        p.trafo()
        f = p.f.astype(np.complex128).copy()
        p.f[:] = W.complex_normal(M, seed=4)
        y = p.f.astype(np.complex128).copy()
        p.adjoint()
        h = p.f_hat.astype(np.complex128).copy()
    finally:
        p.finalize()
    f0, h0 = O.nfft_trafo(N, n, m, xr, fh), O.nfft_adjoint(N, n, m, xr, y)
    et, ea = np.linalg.norm(f - f0) / np.linalg.norm(f0), np.linalg.norm(h - h0) / np.linalg.norm(h0)
    print("n0=%d m=%d %s: trafo %.2e adjoint %.2e" % (n[0], m, precision, et, ea))
    assert et < TOL[precision] and ea < TOL[precision]
