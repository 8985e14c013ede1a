"""The matrix-core B^T of 2-D plans (tiles of up to 32 or 48 cells per edge in
16 x 16 blocks, several wavefronts per item, skipped blocks) against the FP64
oracle, where its geometry can go wrong: tiles of both block counts and wider
ones (which other kernels take), bins that divide the grid and ragged ones,
windows from 4 to 20 taps, dimensions of different oversampling, items of one
to some thousand nodes, lone nodes and nodes on the wrap; and batches, whose
workgroups take two right-hand sides, against single calls.

Tolerances: FP64 1e-12 and FP32 2e-6, as for the 3-D kernels: sums of about
(2m+2)^2 products and, in dense cells, some thousand contributions.
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


def adjoint_error(N, n, m, x, precision):
    p = nf.Plan(N, x.shape[0], n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=nf.FFTW_ESTIMATE)
    try:
        p.x[:] = x
        p.precompute()
        xr = p.x.astype(np.float64).copy()
        p.f[:] = W.complex_normal(x.shape[0], seed=4)
        fin = p.f.astype(np.complex128).copy()
        p.adjoint()
        h = p.f_hat.astype(np.complex128).copy()
    finally:
        p.finalize()
    return rel(h, O.nfft_adjoint(N, n, m, xr, fin))


GRIDS = [
    ([20, 20], [40, 40]),       # ragged bins of 16 cells, 33-cell tiles from m = 8 on
    ([32, 64], [64, 128]),      # bins that divide the grid
    ([40, 30], [100, 64]),      # unequal oversampling
    ([256, 20], [1024, 48]),    # a 32-cell bin edge: three blocks
    ([16, 800], [32, 2048]),    # a 64-cell bin edge: other kernels
]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("N,n", GRIDS, ids=["40", "64x128", "100x64", "1024x48", "32x2048"])
def test_windows_and_grids(N, n, m, precision):
    x = np.concatenate([W.uniform(701, 2, seed=m), np.full((3, 2), -0.5), np.full((1, 2), 0.4999),
                        np.zeros((2, 2))])
    e = adjoint_error(N, n, m, x, precision)
    print("%s m=%d %s: %.2e" % (n, m, precision, e))
    assert e < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["double", "single"])
@pytest.mark.parametrize("M", [1, 2, 5, 63, 64, 65, 257])
def test_item_sizes(M, precision):
    """All nodes in one bin: wavefronts without a node, no
    whole group of four, a chunk and a node."""
    x = np.random.default_rng(M).uniform(0.0, 0.1, (M, 2))
    e = adjoint_error([32, 32], [64, 64], 4, x, precision)
    assert e < TOL[precision]


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 4, 7])
def test_dense_cells_and_batches(m):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(6)
    x = np.concatenate([np.full((5001, 2), 0.01), rng.uniform(-0.1, 0.02, (3000, 2)), np.full((1, 2), 0.31)])
    assert adjoint_error([32, 40], [64, 80], m, x, "double") < TOL["double"]
    assert adjoint_error([32, 40], [64, 80], m, x, "single") < TOL["single"]
    N, n, R = [32, 32], [64, 64], 5
    M, NN = x.shape[0], int(np.prod(N))
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision="single")
    try:
        p.x[:] = x
        p.precompute()
        fi = torch.from_numpy(W.complex_normal(R * M, seed=2)).to(torch.complex64).cuda()
        a = torch.empty(R * NN, dtype=torch.complex64, device="cuda")
        torch.cuda.synchronize()
        p.adjoint_batch_device(fi.data_ptr(), a.data_ptr(), R)
        p.synchronize()
        for r in range(R):
            a1 = torch.empty_like(a[:NN])
            p.adjoint_device(fi[r * M:].data_ptr(), a1.data_ptr())
            p.synchronize()
            assert torch.equal(a1, a[r * NN:(r + 1) * NN])
    finally:
        p.finalize()
