"""A solver whose plan gets new nodes between solves: the captured step of the
first nodes must not be replayed for the second ones (item counts, several
items per bin, list addresses).  Steps as graph replays against eager steps
(NFFT_HIP_CGNR_GRAPH=0) of a solver on the same plan, bit for bit."""
import numpy as np
import pytest

import nfft_amd as nf
from nfft_amd import workloads as W

FLAGS = nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT


def solve(s, y, steps=4):
    s.y[:] = y
    s.f_hat_iter[:] = 0
    s.before_loop()
    for _ in range(steps):
        s.loop_one_step()
    return s.f_hat_iter.copy(), s.r_iter.copy(), float(s.s.dot_z_hat_iter)


@pytest.mark.gpu
@pytest.mark.parametrize("N,n", [([40, 48], [80, 96]), ([12, 14, 10], [24, 28, 20])], ids=["2d", "3d"])
def test_new_nodes_between_solves(N, n, monkeypatch):
    d, M = len(N), 20000
    rng = np.random.default_rng(3)
    few = W.uniform(M, d, seed=1)                 # spread over all bins
    dense = rng.uniform(0.0, 0.03, (M, d))        # a few cells: bins of several items
    y = W.complex_normal(M, seed=2)
    p = nf.Plan(N, M, n=n, m=4, flags=FLAGS, precision="single")
    try:
        p.x[:] = dense
        p.precompute()
        monkeypatch.setenv("NFFT_HIP_CGNR_GRAPH", "1")
        s = nf.Solver(p, nf.CGNR)
        monkeypatch.setenv("NFFT_HIP_CGNR_GRAPH", "0")
        e = nf.Solver(p, nf.CGNR)
        try:
            for x in (dense, few, dense):
                p.x[:] = x
                p.precompute()
                a, b = solve(s, y), solve(e, y)
                assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]
                assert np.linalg.norm(a[1]) < np.linalg.norm(y)
        finally:
            s.finalize()
            e.finalize()
    finally:
        p.finalize()
