"""How far FP32 transforms are from FP64 ones on the same (FP32) nodes and data,
beyond the tolerances of the parity tests.

* The mean factor by which results are too large or small, Re <exact, result -
  exact> / |exact|^2, stays below half of FP32's unit roundoff, 2^-25: rounded
  window polynomials and roots of unity alone make up to 1.4e-7.
* An adjoint of several nodes per cell stays below 1.05 times the error that
  kernels summing runs of a cell's nodes in registers had: 2.07e-7 (256^2 cells,
  2^18 radial nodes, m = 6), 1.32e-7 (m = 2), 3.28e-7 (64^3 cells, 2^20 uniform
  nodes, m = 6).
"""
import numpy as np
import pytest

import nfft_amd as nf

torch = pytest.importorskip("torch")

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT


def nodes(kind, M, d, g):
    kw = {"generator": g, "device": "cuda", "dtype": torch.float64}
    if kind == "uniform":
        x = torch.rand((M, d), **kw) - 0.5
    else:
        a = torch.randn((M // 256, d), **kw)
        r = torch.arange(256, device="cuda", dtype=torch.float64) / 256 - 0.5
        x = ((a / a.norm(dim=1, keepdim=True))[:, None, :] * r[None, :, None]).reshape(-1, d)
    x = (x - torch.round(x)).float()
    return torch.where(x >= 0.5, x - 1, x).cpu().numpy()


def pairs(N, n, m, kind, M):
    """(exact, result) of the trafo and of the adjoint."""
    g = torch.Generator(device="cuda").manual_seed(m)
    x = nodes(kind, M, len(N), g)
    M, NN = x.shape[0], int(np.prod(N))
    fh = torch.randn(NN, generator=g, device="cuda", dtype=torch.complex64)
    f = torch.randn(M, generator=g, device="cuda", dtype=torch.complex64)
    out = []
    for precision, ct in (("double", torch.complex128), ("single", torch.complex64)):
        p = nf.Plan(N, M, n=n, m=m, flags=FLAGS, precision=precision, fftw_flags=nf.FFTW_ESTIMATE)
        try:
            p.x[:] = x
            p.precompute()
            a, b, t, h = fh.to(ct), f.to(ct), torch.empty(M, dtype=ct, device="cuda"), torch.empty(NN, dtype=ct, device="cuda")
            torch.cuda.synchronize()
            p.trafo_device(a.data_ptr(), t.data_ptr())
            p.adjoint_device(b.data_ptr(), h.data_ptr())
            p.synchronize()
            out.append((t.to(torch.complex128), h.to(torch.complex128)))
        finally:
            p.finalize()
    return list(zip(*out))


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("N,n", [([75] * 3, [150] * 3), ([64] * 3, [128] * 3), ([90, 75, 60], [180, 150, 120]),
                                 ([128] * 2, [256] * 2), ([300, 250], [600, 500]), ([2100], [4200])],
                         ids=["150^3", "128^3", "180x150x120", "256^2", "600x500", "4200"])
def test_mean_factor(N, n, m):
    if len(N) == 1:  # (its adjoint's fixed-point tiles have an error of their own)
        cases = pairs(N, n, m, "uniform", 100000)[:1]
    else:
        cases = pairs(N, n, m, "uniform", 100000)
    for exact, y in cases:
        g = float(torch.vdot(exact, y - exact).real / exact.norm() ** 2)
        print("%s m=%d: %+.2e" % (n, m, g))
        assert abs(g) < 2.0 ** -25


@pytest.mark.gpu
@pytest.mark.parametrize("N,n,m,kind,M,before", [
    ([128] * 2, [256] * 2, 6, "radial", 1 << 18, 2.07e-7),
    ([128] * 2, [256] * 2, 2, "radial", 1 << 18, 1.32e-7),
    ([32] * 3, [64] * 3, 6, "uniform", 1 << 20, 3.28e-7)], ids=["256^2-6", "256^2-2", "64^3-6"])
def test_dense_adjoints(N, n, m, kind, M, before):
    exact, y = pairs(N, n, m, kind, M)[1]
    e = float((y - exact).norm() / exact.norm())
    print("%s m=%d: %.3e" % (n, m, e))
    assert e < 1.05 * before
