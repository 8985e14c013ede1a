"""Batched adjoints cut into chunks of right-hand sides (the static scratch
array of the allocation-free entry point holds only so many; batch_chunk
bounds the plan's own): every chunk, and one of a single right-hand side above
all, must reduce the tiles that it spread, not those of the plan's last single
adjoint.  Each result against the single call with the same input, bit for bit
(FP32 kernels in a fixed order), after a single adjoint of another input that
fills the plan's own tiles.
"""
import ctypes

import numpy as np
import pytest

import nfft_amd as nf
from nfft_amd import workloads as W

torch = pytest.importorskip("torch")

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT


def noalloc(p, f, out, nrhs):
    fn = nf.lib().nfftf_adjoint_batch_device_noalloc
    fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    fn.restype = ctypes.c_int
    return fn(ctypes.addressof(p.p), f.data_ptr(), out.data_ptr(), nrhs)


def check(N, n, m, x, counts):
    M, NN, R = x.shape[0], int(np.prod(N)), max(counts)
    p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision="single")
    try:
        p.x[:] = x
        p.precompute()
        g = torch.Generator(device="cuda").manual_seed(11)
        f = torch.randn(R * M, generator=g, device="cuda", dtype=torch.complex64)
        other = torch.randn(M, generator=g, device="cuda", dtype=torch.complex64)
        ref = torch.empty(R * NN, device="cuda", dtype=torch.complex64)
        out = torch.empty_like(ref)
        scrap = torch.empty(NN, device="cuda", dtype=torch.complex64)
        torch.cuda.synchronize()
        for r in range(R):
            p.adjoint_device(f[r * M:].data_ptr(), ref[r * NN:].data_ptr())
        p.adjoint_device(other.data_ptr(), scrap.data_ptr())
        p.synchronize()
        for nrhs in counts:
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            assert noalloc(p, f, out, nrhs) == 0
            p.synchronize()
            bad = [r for r in range(nrhs) if not torch.equal(out[r * NN:(r + 1) * NN], ref[r * NN:(r + 1) * NN])]
            assert not bad, (nrhs, bad)
    finally:
        p.finalize()


@pytest.mark.gpu
@pytest.mark.parametrize("N,n,M,counts", [
    ([256, 256], [512, 512], 206336, range(2, 14)),   # every remainder of some chunk size
    ([512, 512], [1024, 1024], 1 << 17, range(2, 6)),
    ([600, 600], [1280, 1280], 1 << 20, [2, 3]),      # chunks of one
    ([100, 90], [210, 198], 40000, range(2, 6)),
], ids=["512", "1024", "1280", "210x198"])
def test_two_dimensions(N, n, M, counts):
    check(N, n, 4, W.uniform(M, 2, seed=4), counts)


@pytest.mark.gpu
def test_three_dimensions():
    """Matrix-core plans; 9000 nodes in a few cells give bins of several items."""
    x = np.concatenate([W.uniform(6000, 3, seed=5), np.random.default_rng(6).uniform(0.0, 0.02, (9000, 3))])
    check([24, 20, 28], [48, 40, 56], 4, x, range(2, 14))


@pytest.mark.gpu
def test_three_dimensions_lds_tiles(monkeypatch):
    """3-D plans on the LDS-tile kernels (the variable names their B^T)."""
    monkeypatch.setenv("NFFT_HIP_SPREAD", "runs2sbc")
    check([32, 32, 32], [64, 64, 64], 4, W.uniform(6000, 3, seed=7), range(2, 10))
