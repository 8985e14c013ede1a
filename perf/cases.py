"""The transforms that the performance of this library is judged by.

Each case is work a program using the plan API has it do: a plan and its node
data exist (``prepare``), and one pass runs transforms through the public
entry points of ``nfft_amd`` (``run``).  Sizes are those of the benchmark
(``bench.py``), of the tests, and of the reference's own benchmark program
(examples/nfft/nfft_benchomp.c), plus ragged ones.  Plans use FFTW_ESTIMATE, the
default of the initialisers.

Keys of a case:
  op         trafo, adjoint, pair (both), host (both through the plan's host
             arrays), batch (both, ``nrhs`` vectors sharing the nodes),
             cgnr (weighted CGNR steps), weights (Pipe-Menon density weights)
  dim, N0..  dimension and bandwidths
  n0..       oversampled grid lengths
  m          window cut-off (2m + 2 taps per dimension)
  prec       single or double
  nodes      uniform, clustered (half uniform, half a narrow Gaussian at the
             centre), radial (spokes through the centre)
  M          node count (spokes x samples for radial sets)
  spokes     radial sets: number of spokes
  nrhs       right-hand sides (batch)
  steps      iterations (cgnr, weights)
"""
import math

import numpy as np
import torch

import nfft_amd as nf
from nfft_amd import density

FLAGS = (nf.PRE_PHI_HUT | nf.PRE_PSI | nf.MALLOC_X | nf.MALLOC_F_HAT | nf.MALLOC_F | nf.FFTW_INIT
         | nf.NFFT_SORT_NODES)


def _case(op, N, n, m, prec, nodes, M, **more):
    c = {"op": op, "dim": len(N), "m": m, "prec": prec, "nodes": nodes, "M": M, "spokes": 0,
         "nrhs": 1, "steps": 0}
    for t in range(len(N)):
        c["N%d" % t] = int(N[t])
        c["n%d" % t] = int(n[t])
    c.update(more)
    return c


def _named(name, *a, **more):
    return dict(_case(*a, **more), name=name)


def listed():
    return [
        # the smallest real call: one short 1-D transform pair; launches and
        # latency count
        _named("1d_small_f64", "pair", [1024], [2048], 6, "double", "uniform", 4096),
        # the reference benchmark's 1-D size: long axis, few taps per node
        _named("1d_2pow21_f32", "pair", [1 << 21], [1 << 22], 4, "single", "uniform", 1 << 21),
        # a program written for the reference: default plan (m = 8, grid of the
        # next power of two doubled), odd bandwidth, host arrays
        _named("2d_host_default_f64", "host", [151, 94], [512, 256], 8, "double", "uniform", 20011),
        # 2-D with a dense cluster, both precisions
        _named("2d_512_f32", "pair", [512, 512], [1024, 1024], 4, "single", "clustered", 1 << 20),
        _named("2d_512_m6_f64", "pair", [512, 512], [1024, 1024], 6, "double", "clustered", 1 << 20),
        # multi-coil imaging: 32 right-hand sides on one radial trajectory
        _named("2d_coils32_f32", "batch", [256, 256], [512, 512], 4, "single", "radial", 403 * 512,
               spokes=403, nrhs=32),
        # iterative reconstruction of one image: ten weighted CGNR steps
        _named("2d_cgnr_f32", "cgnr", [256, 256], [512, 512], 4, "single", "radial", 251 * 512,
               spokes=251, steps=10),
        # density weights of a new trajectory: twenty B B^T products
        _named("2d_weights_f32", "weights", [256, 256], [512, 512], 4, "single", "radial", 251 * 512,
               spokes=251, steps=20),
        # the headline workload, each direction: 3-D radial ("kooshball") set
        _named("3d_kooshball_trafo_f32", "trafo", [128] * 3, [256] * 3, 4, "single", "radial",
               16384 * 1024, spokes=16384),
        _named("3d_kooshball_adjoint_f32", "adjoint", [128] * 3, [256] * 3, 4, "single", "radial",
               16384 * 1024, spokes=16384),
        # the reference benchmark's 3-D size in double precision
        _named("3d_128_f64", "pair", [128] * 3, [256] * 3, 4, "double", "uniform", 1 << 21),
        # ragged 3-D sizes on a grid that is no power of two, short window
        _named("3d_ragged_f32", "pair", [90, 75, 60], [180, 150, 120], 3, "single", "uniform", 300007),
    ]


def _smooth(v):
    """The next even length at or above v whose prime factors are 2, 3, 5."""
    v = int(v) + int(v) % 2
    while True:
        r = v
        for p in (2, 3, 5):
            while r % p == 0:
                r //= p
        if r == 1:
            return v
        v += 2


def draw(rng):
    op = rng.choice(["pair", "pair", "pair", "trafo", "adjoint", "host", "batch", "cgnr", "weights"])
    prec = rng.choice(["single", "single", "double"])

    def log_uniform(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    if op in ("cgnr", "weights"):
        dim, prec = 2, "single"
    elif op == "batch":
        dim, prec = rng.choice([2, 2, 3]), "single"
    else:
        dim = rng.choice([1, 2, 2, 3, 3])
    m = rng.choice([2, 3, 4, 4, 4, 5, 6]) if prec == "single" else rng.choice([3, 4, 4, 5, 6, 8])
    lo, hi = {1: (512, 1 << 20), 2: (48, 640), 3: (24, 128)}[dim]
    if op in ("cgnr", "weights"):
        lo, hi = 64, 300
    if op == "batch" and dim == 3:
        hi = 64
    N = [log_uniform(lo, hi) for _ in range(dim)]
    if rng.random() < 0.5:
        N = [N[0]] * dim  # isotropic, as most programs have it
    if rng.random() < 0.5:  # the default grid: the next power of two, doubled
        n = [2 << (t - 1).bit_length() for t in N]
    else:
        n = [_smooth(2 * t) for t in N]
    nrhs = rng.choice([2, 3, 8, 16, 33]) if op == "batch" else 1
    # taps of one direction stay far below the largest listed case's
    top = min(1 << 21, int(2.0e9 / (2 * m + 2) ** dim / nrhs / (2 if prec == "double" else 1)))
    M = log_uniform(1000, max(2000, top))
    steps = rng.choice([3, 5, 8]) if op == "cgnr" else rng.choice([5, 10, 20]) if op == "weights" else 0
    if op in ("cgnr", "weights"):
        M = max(M // 4, 4 * N[0] * N[1])
    nodes = rng.choice(["uniform", "clustered", "radial"]) if dim > 1 else "uniform"
    if op in ("cgnr", "weights"):
        nodes = "radial"
    spokes = 0
    if nodes == "radial":
        samples = 2 * max(N)
        spokes = max(8, M // samples)
        M = spokes * samples
    return _case(op, N, n, m, prec, nodes, M, spokes=spokes, nrhs=nrhs, steps=steps)


def _sizes(case):
    d = case["dim"]
    return [case["N%d" % t] for t in range(d)], [case["n%d" % t] for t in range(d)]


def _nodes(case, g):
    """Node coordinates (M, d) on the GPU in the plan's precision, in [-1/2, 1/2)."""
    d, M = case["dim"], case["M"]
    kw = {"generator": g, "device": "cuda", "dtype": torch.float64}
    if case["nodes"] == "uniform":
        x = torch.rand((M, d), **kw) - 0.5
    elif case["nodes"] == "clustered":
        h = M // 2
        x = torch.cat([torch.rand((h, d), **kw) - 0.5, 0.05 * torch.randn((M - h, d), **kw)])
    else:
        S = case["spokes"]
        if d == 2:  # golden-angle spokes from a random first angle
            a = torch.rand(1, **kw) * math.pi
            th = a + torch.arange(S, device="cuda", dtype=torch.float64) * (math.pi * 2 / (1 + 5 ** 0.5))
            dirs = torch.stack([torch.cos(th), torch.sin(th)], 1)
        else:
            dirs = torch.randn((S, d), **kw)
            dirs = dirs / dirs.norm(dim=1, keepdim=True)
        K = M // S
        rad = torch.arange(K, device="cuda", dtype=torch.float64) / K - 0.5
        x = (dirs[:, None, :] * rad[None, :, None]).reshape(M, d)
    x = x - torch.round(x)
    x = x.to(torch.float32 if case["prec"] == "single" else torch.float64)
    return torch.where(x >= 0.5, x - 1, x)


def _inputs(case, seed):
    """Everything a pass reads, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    ct = torch.complex64 if case["prec"] == "single" else torch.complex128
    N, _ = _sizes(case)
    NN, R = int(np.prod(N)), case["nrhs"]
    s = {"x": _nodes(case, g)}
    if case["op"] in ("pair", "host", "batch", "trafo"):
        s["fh"] = torch.randn(R * NN, generator=g, device="cuda", dtype=ct)
    if case["op"] in ("pair", "host", "batch", "adjoint", "cgnr"):
        s["f"] = torch.randn(R * case["M"], generator=g, device="cuda", dtype=ct)
    if case["op"] == "cgnr":
        # density weights as a program reads them from a file: the ramp |x|
        w = s["x"].double().norm(dim=1)
        s["w"] = (w + 0.5 / max(N)).float()
    return s


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    N, n = _sizes(case)
    NN, R, M = int(np.prod(N)), case["nrhs"], case["M"]
    p = nf.Plan(N, M, n=n, m=case["m"], flags=FLAGS, precision=case["prec"])
    p.x[:] = s.pop("x").cpu().numpy()
    p.precompute()
    s["plan"] = p
    ct = torch.complex64 if case["prec"] == "single" else torch.complex128
    op = case["op"]
    if op in ("pair", "batch", "trafo"):
        s["f_out"] = torch.empty(R * M, dtype=ct, device="cuda")
    if op in ("pair", "batch", "adjoint"):
        s["fh_out"] = torch.empty(R * NN, dtype=ct, device="cuda")
    if op == "host":
        s["fh"], s["f"] = s["fh"].cpu().numpy(), s["f"].cpu().numpy()
    if op == "cgnr":
        sv = nf.Solver(p, nf.CGNR | nf.PRECOMPUTE_WEIGHT)
        sv.set_sync(0)
        sv.y[:] = s.pop("f").cpu().numpy()
        sv.w[:] = s.pop("w").cpu().numpy()
        s["solver"] = sv
    if op == "weights":
        s["w"] = torch.empty(M, dtype=torch.float32, device="cuda")
    p.synchronize()
    return s


def run(s):
    case, p = s["case"], s["plan"]
    op = case["op"]
    if op == "host":
        p.f_hat[:] = s["fh"]
        p.trafo()
        f = p.f.copy()
        p.f[:] = s["f"]
        p.adjoint()
        return {"f": f, "f_hat": p.f_hat.copy()}
    if op == "cgnr":
        sv = s["solver"]
        sv.f_hat_iter[:] = 0
        sv.before_loop()
        for _ in range(case["steps"]):
            sv.loop_one_step()
        sv.set_sync(1)
        sv.sync()
        sv.set_sync(0)
        return {"f_hat": sv.f_hat_iter.copy()}
    if op == "weights":
        s["w"].fill_(1.0)
        return {"w": density.pipe_menon_device(p, s["w"], case["steps"])}
    out = {}
    if op == "batch":
        p.trafo_batch_device(s["fh"].data_ptr(), s["f_out"].data_ptr(), case["nrhs"])
        p.adjoint_batch_device(s["f"].data_ptr(), s["fh_out"].data_ptr(), case["nrhs"])
        return {"f": s["f_out"], "f_hat": s["fh_out"]}
    if op in ("pair", "trafo"):
        p.trafo_device(s["fh"].data_ptr(), s["f_out"].data_ptr())
        out["f"] = s["f_out"]
    if op in ("pair", "adjoint"):
        p.adjoint_device(s["f"].data_ptr(), s["fh_out"].data_ptr())
        out["f_hat"] = s["fh_out"]
    return out


def work(case):
    """Inputs read once and outputs written once per transform; the taps of B
    / B^T (a complex value times a real weight, two FMAs) and 5 n log2 n of
    the oversampled FFT."""
    N, n = _sizes(case)
    c = 8 if case["prec"] == "single" else 16
    NN, nn, M, d, R = int(np.prod(N)), int(np.prod(n)), case["M"], case["dim"], case["nrhs"]
    b_flops = 4.0 * M * (2 * case["m"] + 2) ** d
    f_flops = 5.0 * nn * math.log2(nn)
    one = {"bytes": float(R * (NN + M) * c + M * d * (c // 2)), "flops": R * (b_flops + f_flops)}
    if case["op"] == "weights":
        return {"bytes": case["steps"] * 2.0 * M * (4 + d * 4), "flops": case["steps"] * 2 * b_flops}
    times = {"trafo": 1, "adjoint": 1, "cgnr": 2 * case["steps"] + 2}.get(case["op"], 2)
    return {"bytes": times * one["bytes"], "flops": times * one["flops"]}


# ---------------------------------------------------------------- 64-bit results
class _Ndft:
    """The nonequispaced DFT in complex128: separable products for short
    axes, an oversampled FFT with a wide Kaiser-Bessel window for a long 1-D
    axis."""

    def __init__(self, x, N):
        self.x, self.N = x.double(), N
        self.wide = len(N) == 1 and N[0] * x.shape[0] > 1 << 31
        self.chunk = max(1, min(x.shape[0], (1 << 27) // max(1, int(np.prod(N[:-1])))))
        if self.wide:
            self._window(14)

    def _phase(self, t, a, b, sign):
        k = torch.arange(self.N[t], device="cuda", dtype=torch.float64) - self.N[t] // 2
        y = self.x[a:b, t, None] * k[None, :]
        y = (y - torch.round(y)) * (sign * 2 * math.pi)
        return torch.complex(torch.cos(y), torch.sin(y))

    def _window(self, m):
        N, self.n, self.mw = self.N[0], 2 * self.N[0], m
        b = math.pi * 1.5
        y = self.x[:, 0] * self.n
        c = torch.floor(y)
        w = torch.arange(2 * m + 2, device="cuda", dtype=torch.float64) - m
        u = (y - c)[:, None] - w[None, :]
        r = m * m - u * u
        z = torch.sqrt(r.abs())
        small = z < 1e-7
        v = torch.where(r > 0, torch.sinh(b * z), torch.sin(b * z)) / torch.where(small, torch.ones_like(z), z)
        self.psi = torch.where(small, torch.full_like(v, b), v) / math.pi
        self.idx = (c[:, None] + w[None, :]).long() % self.n
        k = torch.arange(N, device="cuda", dtype=torch.float64) - N // 2
        self.kpos = k.long() % self.n
        self.hat = torch.special.i0(m * torch.sqrt(b * b - (2 * math.pi * k / self.n) ** 2))

    def trafo(self, fh):
        M, N = self.x.shape[0], self.N
        if self.wide:
            g = torch.zeros(self.n, dtype=torch.complex128, device="cuda")
            g[self.kpos] = fh / self.hat
            g = torch.fft.fft(g)
            return torch.cat([(g[self.idx[a:a + (1 << 20)]] * self.psi[a:a + (1 << 20)]).sum(1)
                              for a in range(0, M, 1 << 20)])
        F = fh.reshape(-1, N[-1])
        out = torch.empty(M, dtype=torch.complex128, device="cuda")
        for a in range(0, M, self.chunk):
            b = min(M, a + self.chunk)
            z = self._phase(len(N) - 1, a, b, -1.0) @ F.t()
            for t in range(len(N) - 2, -1, -1):
                z = (z.reshape(b - a, -1, N[t]) * self._phase(t, a, b, -1.0)[:, None, :]).sum(2)
            out[a:b] = z.reshape(-1)
        return out

    def adjoint(self, f):
        M, N = self.x.shape[0], self.N
        if self.wide:
            g = torch.zeros(self.n, 2, dtype=torch.float64, device="cuda")
            for a in range(0, M, 1 << 20):
                v = torch.view_as_real(f[a:a + (1 << 20), None] * self.psi[a:a + (1 << 20)])
                g.index_add_(0, self.idx[a:a + (1 << 20)].reshape(-1), v.reshape(-1, 2))
            g = torch.fft.ifft(torch.view_as_complex(g), norm="forward")
            return g[self.kpos] / self.hat
        out = torch.zeros(int(np.prod(N[:-1])), N[-1], dtype=torch.complex128, device="cuda")
        for a in range(0, M, self.chunk):
            b = min(M, a + self.chunk)
            z = f[a:b, None]
            for t in range(len(N) - 1):
                z = (z[:, :, None] * self._phase(t, a, b, 1.0)[:, None, :]).reshape(b - a, -1)
            out += z.t().contiguous() @ self._phase(len(N) - 1, a, b, 1.0)
        return out.reshape(-1)


def _pipe_menon(case, x):
    """w <- w / (B B^T w) with the plan's window scaled to peak 1, in FP64."""
    N, n = _sizes(case)
    m = case["m"]
    idx, psi = None, None
    for t in range(2):
        b = math.pi * (2.0 - N[t] / n[t])
        y = x[:, t].double() * n[t]
        c = torch.floor(y)
        w = torch.arange(2 * m + 2, device="cuda", dtype=torch.float64) - m
        u = (y - c)[:, None] - w[None, :]
        r = m * m - u * u
        z = torch.sqrt(r.abs())
        small = z < 1e-7
        v = torch.where(r > 0, torch.sinh(b * z), torch.sin(b * z)) / torch.where(small, torch.ones_like(z), z)
        v = torch.where(small, torch.full_like(v, b), v) / (math.sinh(b * m) / m)
        i = (c[:, None] + w[None, :]).long() % n[t]
        if idx is None:
            idx, psi = i, v
        else:
            idx = (idx[:, :, None] * n[1] + i[:, None, :]).reshape(x.shape[0], -1)
            psi = (psi[:, :, None] * v[:, None, :]).reshape(x.shape[0], -1)
    w = torch.ones(x.shape[0], dtype=torch.float64, device="cuda")
    for _ in range(case["steps"]):
        g = torch.zeros(n[0] * n[1], dtype=torch.float64, device="cuda")
        g.index_add_(0, idx.reshape(-1), (psi * w[:, None]).reshape(-1))
        w = w / (g[idx] * psi).sum(1)
    return w


def exact(case, seed):
    """The same outputs from the definition, in 64 bits.  None for products
    of bandwidths and nodes that would take too long (the 2^24-node sets)."""
    N, _ = _sizes(case)
    R, M, NN = case["nrhs"], case["M"], int(np.prod(N))
    if case["dim"] == 3 and float(NN) * M > 1.0e13:
        return None
    s = _inputs(case, seed)
    if case["op"] == "weights":
        return {"w": _pipe_menon(case, s["x"])}
    A = _Ndft(s["x"], N)
    if case["op"] == "cgnr":
        # weighted CGNR (minimise the weighted residual), from zero
        y, w = s["f"].to(torch.complex128), s["w"].double()
        fh = torch.zeros(NN, dtype=torch.complex128, device="cuda")
        r = y.clone()
        z = A.adjoint(w * r)
        p, zz = z.clone(), torch.vdot(z, z).real
        for _ in range(case["steps"]):
            v = A.trafo(p)
            alpha = zz / (w * v.abs() ** 2).sum()
            fh = fh + alpha * p
            r = r - alpha * v
            z = A.adjoint(w * r)
            old, zz = zz, torch.vdot(z, z).real
            p = z + (zz / old) * p
        return {"f_hat": fh}
    out = {}
    if "fh" in s:
        out["f"] = torch.cat([A.trafo(s["fh"][r * NN:(r + 1) * NN].to(torch.complex128))
                              for r in range(R)])
    if "f" in s:
        out["f_hat"] = torch.cat([A.adjoint(s["f"][r * M:(r + 1) * M].to(torch.complex128))
                                  for r in range(R)])
    if case["op"] == "host":
        return {k: v.cpu().numpy() for k, v in out.items()}
    return out
