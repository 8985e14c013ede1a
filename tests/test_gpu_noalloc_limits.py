"""Which plans the allocation-free batched adjoint takes, and what it computes
for them: its limit counts the LDS-tile kernels' scratch whichever kernels
run, by bounds where they settle it.  Results against single adjoints, bit for
bit (FP32 kernels in a fixed order)."""
import ctypes

import numpy as np
import pytest

import nfft_amd as nf
from nfft_amd import workloads as W

torch = pytest.importorskip("torch")

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT


def run(N, n, x, nrhs=2, m=4):
    """Return code of the call; with 0, its results are checked."""
    M, NN = x.shape[0], int(np.prod(N))
    fn = nf.lib().nfftf_adjoint_batch_device_noalloc
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    fn.restype = ctypes.c_int
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision="single")
    try:
        p.x[:] = x
        p.precompute()
        g = torch.Generator(device="cuda").manual_seed(3)
        f = torch.randn(nrhs * M, generator=g, device="cuda", dtype=torch.complex64)
        out = torch.full((nrhs * NN,), 7.0, device="cuda", dtype=torch.complex64)
        one = torch.empty(NN, device="cuda", dtype=torch.complex64)
        torch.cuda.synchronize()
        rc = fn(ctypes.addressof(p.p), f.data_ptr(), out.data_ptr(), nrhs)
        p.synchronize()
        if rc:
            assert bool(torch.all(out == 7.0))
            return rc
        for r in range(nrhs):
            p.adjoint_device(f[r * M:].data_ptr(), one.data_ptr())
            p.synchronize()
            assert torch.equal(one, out[r * NN:(r + 1) * NN]), r
        return 0
    finally:
        p.finalize()


@pytest.mark.gpu
def test_grid_beyond_the_array():
    """216^3 cells are 77 MiB: refused, by the lower bound alone."""
    assert run([108] * 3, [216] * 3, W.uniform(3000, 3, seed=1)) == -4


@pytest.mark.gpu
def test_matrix_core_tiles_beyond_the_array():
    """88^3 cells: 1331 LDS tiles and the grid are 55 MiB, the matrix-core tiles
    67 MiB: taken, one right-hand side at a time."""
    assert run([44] * 3, [88] * 3, W.uniform(200000, 3, seed=2), nrhs=3) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M,rc", [(4000000, 0), (4180000, -4)])
def test_counted_limit(M, rc):
    """1024^2 cells in 1024 bins, items of up to 1024 nodes and 13 KB, of which
    the array holds 4366 beside the grid; the bounds (M / 1024 items, 1024 more)
    leave both sets open.  4 * 10^6 uniform nodes: 4 items a bin.  4.18 * 10^6:
    4082 nodes a bin, more than 4096 in two of five: about 4500 items."""
    assert run([512] * 2, [1024] * 2, W.uniform(M, 2, seed=3)) == rc
