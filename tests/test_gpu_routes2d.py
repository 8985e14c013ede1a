"""2-D B^T on either side of the rules that pick its bins and kernel, against
the FP64 oracle: grids that no edge near 16 divides (ragged last bins, tiles
kept in scratch and reduced cell by cell), three blocks of 16 cells with short
windows (given bins), and m = 8, which few nodes on large bins leave to the
LDS-tile kernels.

Tolerances as for the other 2-D kernels: FP64 1e-12, FP32 2e-6."""
import numpy as np
import pytest

import nfft_amd as nf
import oracle as O
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT
TOL = {"double": 1e-12, "single": 2e-6}


def errors(N, n, m, x, precision):
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
    return np.linalg.norm(f - f0) / np.linalg.norm(f0), np.linalg.norm(h - h0) / np.linalg.norm(h0)


def some_nodes(M, seed):
    return np.concatenate([W.uniform(M, 2, seed=seed), np.full((3, 2), -0.5), np.full((2, 2), 0.4999),
                           np.random.default_rng(seed).uniform(0.0, 0.05, (M // 3, 2))])


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n", [(58, 62), (74, 46), (86, 31)], ids=["58x62", "74x46", "86x31"])
def test_ragged_last_bins(n, m, precision):
    e = errors([n[0] // 2, n[1] // 2], list(n), m, some_nodes(900, m), precision)
    print("%s m=%d %s: %.2e %.2e" % (n, m, precision, *e))
    assert max(e) < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 3, 4, 6, 7])
@pytest.mark.parametrize("bins", ["24,20", "30,32", "33,16"])
def test_three_blocks(bins, m, precision, monkeypatch):
    """Bins that divide neither, one or both of 120 x 160 cells; E = bin + 2m + 1
    of up to 48 cells takes three blocks, beyond that other kernels."""
    monkeypatch.setenv("NFFT_HIP_BINS", bins)
    e = errors([60, 80], [120, 160], m, some_nodes(900, m), precision)
    print("bins %s m=%d %s: %.2e %.2e" % (bins, m, precision, *e))
    assert max(e) < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("M", [500, 8000])
def test_widest_window(M, precision):
    """m = 8 on 1024 x 32 cells (bins of 32 x 16): below a sixth of a node per
    cell, and above."""
    e = errors([512, 16], [1024, 32], 8, some_nodes(M, 5), precision)
    print("M=%d %s: %.2e %.2e" % (M, precision, *e))
    assert max(e) < TOL[precision]
