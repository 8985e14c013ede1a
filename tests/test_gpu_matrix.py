"""The matrix-core B and B^T of 3-D plans (ragged bins of at most 17 - W cells
along the two last dimensions, columns along the first) against the FP64
oracle, where their geometry can go wrong: grids of 16 cells (one tile row
per period), bins of one cell up, odd and unequal lengths, windows from 4 to
14 taps, dimensions of different oversampling (per-dimension window tables),
dense sets (the split FP32 interpolation), bins of several items (their tiles
summed first), lone nodes and nodes on the wrap.

Tolerances: FP64 1e-12, as for the other kernels.  FP32: each result sums
about (2m+2)^3 products and, for dense cells, up to some thousand node
contributions in FP32 (unit rounding 6e-8, errors growing with the square
root of the count): 2e-6.
"""
import numpy as np
import pytest

import nfft_amd as nf
import oracle as O
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT
TOL = {"double": 1e-12, "single": 2e-6}


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.complex128) - b) / np.linalg.norm(b))


def run(N, n, m, x, precision, fftw_flags=nf.FFTW_ESTIMATE):
    M = x.shape[0]
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=fftw_flags)
    try:
        p.x[:] = x
        p.precompute()
        xr = p.x.astype(np.float64).copy()
        p.f_hat[:] = W.complex_normal(int(np.prod(N)), seed=3)
        fh = p.f_hat.astype(np.complex128).copy()
        p.trafo()
        f = p.f.astype(np.complex128).copy()
        p.f[:] = W.complex_normal(M, seed=4)
        fin = p.f.astype(np.complex128).copy()
        p.adjoint()
        h = p.f_hat.astype(np.complex128).copy()
    finally:
        p.finalize()
    return (rel(f, O.nfft_trafo(N, n, m, xr, fh)), rel(h, O.nfft_adjoint(N, n, m, xr, fin)))


GRIDS = [
    ([8, 8, 8], [16, 16, 16]),      # a tile row is the whole period
    ([10, 9, 12], [20, 18, 24]),    # odd bandwidth, few bins
    ([16, 14, 11], [40, 32, 33]),   # unequal oversampling, ragged bins
    ([24, 12, 20], [90, 17, 50]),   # long first axis, 17 cells: a bin of one cell more
]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("N,n", GRIDS, ids=["16", "20x18x24", "40x32x33", "90x17x50"])
def test_windows_and_grids(N, n, m, precision):
    """Sparse uniform nodes, some on the wrap and one alone in its bin."""
    x = np.concatenate([W.uniform(701, 3, seed=m), np.full((3, 3), -0.5),
                        np.full((1, 3), 0.4999), np.zeros((2, 3))])
    et, ea = run(N, n, m, x, precision)
    print("%s m=%d %s: trafo %.2e adjoint %.2e" % (n, m, precision, et, ea))
    assert et < TOL[precision] and ea < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [2, 4, 6])
def test_dense_cells_and_many_items(m, precision):
    """9001 nodes in one cell and a dense cloud over a few cells of the first
    dimension: the FP32 plan takes the split interpolation, B^T cuts the bins
    into items of 512 nodes and sums their tiles."""
    rng = np.random.default_rng(5)
    x = np.concatenate([np.full((9001, 3), 0.01), rng.uniform(-0.1, 0.02, (9000, 3)) * [1, 0.1, 0.1],
                        np.full((1, 3), 0.31)])
    et, ea = run([12, 16, 10], [32, 32, 20], m, x, precision)
    print("dense m=%d %s: trafo %.2e adjoint %.2e" % (m, precision, et, ea))
    assert et < TOL[precision] and ea < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("dense", [False, True])
def test_batches_and_measured_plans(dense):
    """Batched FP32 calls equal single calls bit for bit, and FFTW_MEASURE
    plans (which time their FFT lines only) meet the same tolerance."""
    torch = pytest.importorskip("torch")
    N, n, m, R = [12, 10, 14], [24, 20, 30], 4, 3
    x = W.uniform(60000 if dense else 900, 3, seed=9)
    M, NN = x.shape[0], int(np.prod(N))
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision="single")
    try:
        p.x[:] = x
        p.precompute()
        fh = torch.from_numpy(W.complex_normal(R * NN, seed=1)).to(torch.complex64).cuda()
        fi = torch.from_numpy(W.complex_normal(R * M, seed=2)).to(torch.complex64).cuda()
        t = torch.empty(R * M, dtype=torch.complex64, device="cuda")
        a = torch.empty(R * NN, dtype=torch.complex64, device="cuda")
        torch.cuda.synchronize()
        p.trafo_batch_device(fh.data_ptr(), t.data_ptr(), R)
        p.adjoint_batch_device(fi.data_ptr(), a.data_ptr(), R)
        p.synchronize()
        for r in range(R):
            t1, a1 = torch.empty_like(t[:M]), torch.empty_like(a[:NN])
            p.trafo_device(fh[r * NN:].data_ptr(), t1.data_ptr())
            p.adjoint_device(fi[r * M:].data_ptr(), a1.data_ptr())
            p.synchronize()
            assert torch.equal(t1, t[r * M:(r + 1) * M]) and torch.equal(a1, a[r * NN:(r + 1) * NN])
    finally:
        p.finalize()
    et, ea = run(N, n, m, x, "single", fftw_flags=nf.FFTW_MEASURE)
    assert et < TOL["single"] and ea < TOL["single"]
