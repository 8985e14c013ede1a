"""B of 3-D plans on either side of the rule that picks its kernel (LDS tiles
over slabs of the ragged bins, or the matrix cores): node sets of one, about
two and several nodes per cell, grids whose bins are ragged or cut into slabs
(a first axis long enough for bins of 16 and 32 cells), windows of all
widths, dimensions of unequal oversampling, both precisions, against the FP64
oracle; plans that time both kernels; batches against single calls; and new
nodes that move a plan from one kernel to the other.

Tolerances as for the other 3-D kernels: FP64 1e-12, FP32 2e-6."""
import numpy as np
import pytest

import nfft_amd as nf
import oracle as O
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT
TOL = {"double": 1e-12, "single": 2e-6}

GRIDS = [([8, 8, 8], [16, 16, 16]), ([10, 9, 12], [20, 18, 24]), ([16, 14, 11], [40, 32, 33]),
         ([24, 12, 20], [90, 17, 50])]
IDS = ["16", "20x18x24", "40x32x33", "90x17x50"]


def trafo_error(p, N, n, m, x):
    p.x[:] = x
    p.precompute()
    xr = p.x.astype(np.float64).copy()
    p.f_hat[:] = W.complex_normal(int(np.prod(N)), seed=3)
    fh = p.f_hat.astype(np.complex128).copy()
    p.trafo()
    ref = O.nfft_trafo(N, n, m, xr, fh)
    return float(np.linalg.norm(p.f.astype(np.complex128) - ref) / np.linalg.norm(ref))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("N,n", GRIDS, ids=IDS)
def test_dense_sets(N, n, m, precision):
    """Several nodes per cell in one corner, where the rule picks LDS tiles up
    to m = 4, and (the tuner) whichever is faster."""
    x = np.concatenate([W.uniform(6000, 3, seed=m) * 0.2 + 0.1, np.full((3, 3), -0.5), np.full((5, 3), 0.4999)])
    for fftw in (nf.FFTW_ESTIMATE, nf.FFTW_MEASURE):
        p = nf.Plan(N, len(x), n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=fftw)
        try:
            e = trafo_error(p, N, n, m, x)
        finally:
            p.finalize()
        print("%s m=%d %s: %.2e" % (n, m, precision, e))
        assert e < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 3, 4])
def test_slabs_of_long_bins(m, monkeypatch):
    """256 x 150 x 150 cells: bins of 16 and 32 cells, cut into slabs.  Against
    an FP64 plan on the LDS-tile kernels' own bins (the oracle takes minutes)."""
    N, n = [20, 16, 18], [256, 150, 150]
    x = np.concatenate([W.uniform(4000, 3, seed=1), np.random.default_rng(2).uniform(-0.02, 0.03, (19000, 3)),
                        np.full((5, 3), 0.4999)]).astype(np.float32)
    fh = W.complex_normal(int(np.prod(N)), seed=3).astype(np.complex64)
    out = {}
    for key, precision in (("bins", "double"), ("double", "double"), ("single", "single")):
        if key == "bins":
            monkeypatch.setenv("NFFT_HIP_INTERP", "lane")
        p = nf.Plan(N, len(x), n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=nf.FFTW_ESTIMATE)
        monkeypatch.delenv("NFFT_HIP_INTERP", raising=False)
        try:
            p.x[:] = x
            p.precompute()
            p.f_hat[:] = fh
            p.trafo()
            out[key] = p.f.astype(np.complex128).copy()
        finally:
            p.finalize()
    for precision in TOL:
        e = np.linalg.norm(out[precision] - out["bins"]) / np.linalg.norm(out["bins"])
        print("m=%d %s: %.2e" % (m, precision, e))
        assert e < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 3, 4])
def test_new_nodes_change_the_kernel(m, precision):
    N, n = [10, 9, 12], [20, 18, 24]
    x1, x2 = W.uniform(9000, 3, seed=1), W.uniform(9000, 3, seed=2) * 0.15
    p = nf.Plan(N, 9000, n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=nf.FFTW_ESTIMATE)
    try:
        for x in (x1, x2, np.linspace(-0.5, 0.4999, 27000).reshape(9000, 3), x2):
            assert trafo_error(p, N, n, m, x) < TOL[precision]
    finally:
        p.finalize()


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 4])
def test_batches(m):
    torch = pytest.importorskip("torch")
    N, n, R, M = [12, 10, 14], [24, 20, 30], 3, 60000
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision="single")
    try:
        p.x[:] = W.uniform(M, 3, seed=9)
        p.precompute()
        NN = int(np.prod(N))
        fh = torch.from_numpy(W.complex_normal(R * NN, seed=1)).to(torch.complex64).cuda()
        t = torch.empty(R * M, dtype=torch.complex64, device="cuda")
        t1 = torch.empty(M, dtype=torch.complex64, device="cuda")
        torch.cuda.synchronize()
        p.trafo_batch_device(fh.data_ptr(), t.data_ptr(), R)
        p.synchronize()
        for r in range(R):
            p.trafo_device(fh[r * NN:].data_ptr(), t1.data_ptr())
            p.synchronize()
            assert torch.equal(t1, t[r * M:(r + 1) * M])
    finally:
        p.finalize()
