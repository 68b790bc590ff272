"""Performance cases of the NFFT library: what programs call, at the sizes they use.

A case is a dict of plain values.  ``path`` names the way a program uses the
library, the other keys give the problem:

* ``plan``      coefficients and samples on the GPU, nodes fixed (an iterative
                reconstruction, a particle mesh at one time step): the plan and its
                nodes are in hand, a pass is transform_dev and / or adjoint_dev;
* ``nodes``     the nodes move before every pass (time stepping, trajectory sweeps):
                set_nodes_dev, transform_dev, adjoint_dev;
* ``host``      the call sequence of the original library on its host arrays: copy in,
                transform, copy out, copy in, adjoint, copy out;
* ``autograd``  cunfft_amd.autograd.nfft and its backward, gradients with respect to the
                coefficients and the nodes;
* ``batch``     many uneven 2D problems with several right-hand sides in one launch,
                autotuned once at set-up as bench.py does;
* ``solve``     the inverse NFFT by conjugate gradients, a fixed number of iterations.

``exact`` evaluates the same sums (roll-off, oversampled FFT, window taps) with
torch in 64 bits, without the library.
"""
import math

import numpy as np
import torch

import cunfft_amd as cu
from cunfft_amd.autograd import NFFTOperator, nfft
from cunfft_amd.batch import Batch

GRIDS = [v for a in range(1, 25) for b in range(0, 3) if 32 <= (v := 2 ** a * 3 ** b)]


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # The smallest call: a 1D transform of a signal of 1024 samples, default cut-off.
        dict(name="1d_1024_m6_f64_forward", path="plan", d=1, N0=1024, n0=2048, M=4096, m=6,
             double=True, window="gauss", nodes="uniform", dirs="forward"),
        # The other end of 1D: long series (the largest 1D size of the original's
        # runtime tables), whose axis takes two FFT passes.
        dict(name="1d_4m_m4_f64", path="plan", d=1, N0=1 << 22, n0=1 << 23, M=1 << 22, m=4,
             double=True, window="gauss", nodes="uniform", dirs="both"),
        # Radial imaging slice, forward and adjoint per iteration, FP32.
        dict(name="2d_radial512_m4_f32", path="plan", d=2, N0=512, N1=512, n0=1024, n1=1024,
             M=512 * 512, m=4, double=False, window="gauss", nodes="radial", dirs="both"),
        # The drop-in use: the original's own call sequence with its default cut-off.
        dict(name="2d_host512_m6_f64", path="host", d=2, N0=512, N1=512, n0=1024, n1=1024,
             M=512 * 512, m=6, double=True, window="gauss", nodes="uniform"),
        # A learned sampling pattern: value and gradients, nodes new in every step.
        dict(name="2d_autograd256_m4_f64", path="autograd", d=2, N0=256, N1=256, n0=512, n1=512,
             M=65536, m=4, double=True, window="gauss", nodes="uniform"),
        # Unequal sizes that are no powers of two, an odd node count, the Kaiser-Bessel
        # window, moving nodes.
        dict(name="2d_nodes192x144_m3_f32_kb", path="nodes", d=2, N0=192, N1=144, n0=384, n1=288,
             M=50021, m=3, double=False, window="kb", nodes="uniform"),
        # The headline benchmark: 3D, half of the nodes in a cluster, FP32 ...
        dict(name="3d_128_m4_f32", path="plan", d=3, N0=128, N1=128, N2=128, n0=256, n1=256,
             n2=256, M=1 << 21, m=4, double=False, window="gauss", nodes="cluster", dirs="both"),
        # ... and FP64.
        dict(name="3d_128_m4_f64", path="plan", d=3, N0=128, N1=128, N2=128, n0=256, n1=256,
             n2=256, M=1 << 21, m=4, double=True, window="gauss", nodes="cluster", dirs="both"),
        # 3D with the default cut-off (the original's 64^3 row), the adjoint alone.
        dict(name="3d_64_m6_f64_adjoint", path="plan", d=3, N0=64, N1=64, N2=64, n0=128, n1=128,
             n2=128, M=1 << 18, m=6, double=True, window="gauss", nodes="uniform", dirs="adjoint"),
        # Gradients in 3D on an uneven box, FP32.
        dict(name="3d_autograd96x64x128_m4_f32", path="autograd", d=3, N0=96, N1=64, N2=128,
             n0=192, n1=128, n2=256, M=400009, m=4, double=False, window="gauss", nodes="cluster"),
        # Slices and coils of a study: uneven 2D problems, 8 right-hand sides, FP32.
        dict(name="2d_batch24x8_m4_f32", path="batch", d=2, P=24, R=8, M=65536, m=4, double=False),
        # Inverse NFFT of a density-weighted radial acquisition.
        dict(name="2d_solve256_m4_f64", path="solve", d=2, N0=256, N1=256, n0=512, n1=512,
             M=100800, m=4, double=True, window="gauss", nodes="radial", iters=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _next_pow2(v):
    return 1 << (v - 1).bit_length()


def draw(rng):
    path = rng.choice(["plan", "plan", "plan", "nodes", "host", "autograd", "batch", "solve"])
    if path == "batch":
        return dict(path="batch", d=2, P=rng.randint(4, 24), R=rng.randint(1, 8),
                    M=_log_int(rng, 8192, 65536), m=rng.randint(2, 6), double=rng.random() < 0.25)
    d = 2 if path == "solve" else rng.choice([1, 2, 2, 3, 3])
    double = path == "solve" or rng.random() < 0.5
    c = dict(path=path, d=d)
    top = {1: 1 << 20, 2: 512, 3: 128}[d]
    if path in ("host", "solve"):
        top = {1: 1 << 18, 2: 256 if path == "solve" else 512, 3: 64}[d]
    for t in range(d):
        N = 2 * _log_int(rng, {1: 256, 2: 16, 3: 8}[d], top // 2)
        if d > 1 and rng.random() < 0.5:
            N = max(32, N // 16 * 16)   # sizes that an exact twofold grid suits
        n = 2 * N if 2 * N in GRIDS and rng.random() < 0.5 else 2 * _next_pow2(N)
        c["N%d" % t], c["n%d" % t] = N, n
    cells = math.prod(c["N%d" % t] for t in range(d))
    c["m"] = rng.choice([2, 3, 4, 4, 4, 5, 6, 6]) if d < 3 else rng.choice([3, 4, 4, 5, 6])
    # about one node per coefficient, at most what the largest listed case costs
    most = {1: 1 << 21, 2: 1 << 19, 3: (1 << 21) * 1000 // (2 * c["m"] + 2) ** 3}[d]
    most //= {"solve": 8, "host": 4, "autograd": 4}.get(path, 1)
    M = int(cells * math.exp(rng.uniform(math.log(0.3), math.log(3.0))))
    c["M"] = max(1000, min(most, M)) | 1
    c["double"] = double
    c["window"] = rng.choice(["gauss", "gauss", "gauss", "kb"])
    c["nodes"] = rng.choice(["uniform", "cluster"] if d != 2 else ["uniform", "cluster", "radial"])
    if path == "plan":
        c["dirs"] = rng.choice(["forward", "adjoint", "both", "both"])
    if path == "solve":
        c["iters"] = rng.randint(5, 12)
    return c


# ----------------------------------------------------------------- inputs --
def _sizes(case):
    d = case["d"]
    return [case["N%d" % t] for t in range(d)], [case["n%d" % t] for t in range(d)]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _nodes(case, g):
    """(M, d) nodes in [-1/2, 1/2), float64 on the GPU."""
    M, d = case["M"], case["d"]
    if case["nodes"] == "radial":
        # spokes through the centre from a random first angle
        spokes = max(1, math.isqrt(M))
        per = -(-M // spokes)
        j = torch.arange(M, device="cuda")
        first = torch.rand(1, generator=g, device="cuda", dtype=torch.float64) * math.pi
        th = first + (j // per).double() * (math.pi / spokes)
        r = -0.5 + (j % per).double() / per
        return torch.stack([r * torch.cos(th), r * torch.sin(th)], 1).contiguous()
    x = torch.rand(M, d, generator=g, device="cuda", dtype=torch.float64) - 0.5
    if case["nodes"] == "cluster":
        # half of them around the centre, wrapped onto the torus
        k = M // 2
        c = 0.1 * torch.randn(M - k, d, generator=g, device="cuda", dtype=torch.float64)
        x[k:] = c - torch.floor(c + 0.5)
    return x


def _complex(n, double, g):
    re = torch.randn(n, 2, generator=g, device="cuda",
                     dtype=torch.float64 if double else torch.float32)
    return torch.view_as_complex(re)


def _inputs(case, seed):
    """The arrays of a single-problem case: x, fhat, f (weights for a solve)."""
    g = _gen(seed)
    N, _ = _sizes(case)
    x = _nodes(case, g)
    fhat = _complex(math.prod(N), case["double"], g)
    f = _complex(case["M"], case["double"], g)
    return x, fhat, f


def _radius_weights(case, x):
    """Density weights of a radial acquisition (|x|, floored at the centre)."""
    w = x.norm(dim=1).clamp_min(0.25 / case["N0"])
    return w.to(torch.float64 if case["double"] else torch.float32).contiguous()


def _batch_inputs(case, seed):
    """N (P, 2), M (P,), and per problem x, fhat (R, N_total), f (R, M).  The sizes
    belong to the case, the values to the seed."""
    r = np.random.default_rng([case["P"], case["R"], case["M"]])
    side = r.choice([64, 96, 128, 192, 256], case["P"])
    M = r.integers(4096, case["M"], case["P"], endpoint=True)
    g = _gen(seed)
    probs = []
    for i in range(case["P"]):
        x = torch.rand(int(M[i]), 2, generator=g, device="cuda", dtype=torch.float64) - 0.5
        Nt = int(side[i]) ** 2
        fhat = _complex(case["R"] * Nt, case["double"], g).view(case["R"], Nt)
        f = _complex(case["R"] * int(M[i]), case["double"], g).view(case["R"], int(M[i]))
        probs.append((x, fhat, f))
    return np.stack([side, side], 1), M, probs


def _flags(case):
    return cu.KAISER_BESSEL if case["window"] == "kb" else 0


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ------------------------------------------------------- prepare and run --
def prepare(case, seed):
    path = case["path"]
    precision = "double" if case["double"] else "single"
    s = {"case": case}
    if path == "batch":
        N, M, probs = _batch_inputs(case, seed)
        b = Batch(N, M, m=case["m"], n_rhs=case["R"], n=2 * N, precision=precision)
        out = []
        for i, (x, fhat, f) in enumerate(probs):
            b.set_nodes_dev(i, x.data_ptr(), _stream())
            fhat_in, f_out, f_in, fhat_out = b.tensors(i)
            fhat_in.copy_(fhat)
            f_in.copy_(f)
            # the views do not own the batch's buffers: each keeps its batch alive
            f_out.batch = fhat_out.batch = b
            out.append((f_out, fhat_out))
        torch.cuda.synchronize()
        b.autotune(reps=2, stream=_stream())
        torch.cuda.synchronize()
        s.update(batch=b, out=out)
        return s
    N, n = _sizes(case)
    x, fhat, f = _inputs(case, seed)
    if path == "autograd":
        s["op"] = NFFTOperator(N, case["M"], n=n, m=case["m"], precision=precision,
                               flags=_flags(case))
        s.update(x=x, fhat=fhat, f=f)
        return s
    flags = cu.CUFFT_INIT | cu.CUFFT_BOTH | _flags(case)
    if path == "host":
        p = cu.Plan(N, case["M"], n=n, m=case["m"], precision=precision, flags=flags)
        p.x[:] = x.cpu().numpy()
        p.f_hat[:] = fhat.cpu().numpy()
        p.f[:] = f.cpu().numpy()
        s.update(plan=p, f_hat=p.f_hat.copy(), f=p.f.copy())
        return s
    p = cu.Plan(N, case["M"], n=n, m=case["m"], precision=precision,
                flags=flags | cu.NO_HOST_BUFFERS)
    p.set_nodes_dev(x.data_ptr(), _stream())
    s.update(plan=p, x=x, fhat=fhat, f=f, f_out=torch.empty_like(f), h_out=torch.empty_like(fhat))
    if path == "solve":
        s["w"] = _radius_weights(case, x)
    return s


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "batch":
        s["batch"].execute(stream=_stream())
        return s["out"]
    if path == "autograd":
        fhat = s["fhat"].detach().requires_grad_(True)
        x = s["x"].detach().requires_grad_(True)
        f = nfft(fhat, x, s["op"])
        f.backward(s["f"])
        return f.detach(), fhat.grad, x.grad
    p = s["plan"]
    if path == "host":
        p.f_hat[:] = s["f_hat"]
        p.copyDataToDevice()
        p.transform()
        p.copyDataToHost()
        f = p.f.copy()
        p.f[:] = s["f"]
        p.copyDataToDeviceAd()
        p.adjoint()
        p.copyDataToHostAd()
        return f, p.f_hat.copy()
    st = _stream()
    if path == "solve":
        s["h_out"].zero_()
        _, hist = p.solve_dev(s["f"].data_ptr(), s["h_out"].data_ptr(), s["w"].data_ptr(),
                              max_iter=case["iters"], tol=0.0, stream=st)
        return s["h_out"], np.array(hist)
    if path == "nodes":
        p.set_nodes_dev(s["x"].data_ptr(), st)
    dirs = case.get("dirs", "both")
    out = []
    if dirs != "adjoint":
        p.transform_dev(s["fhat"].data_ptr(), s["f_out"].data_ptr(), st)
        out.append(s["f_out"])
    if dirs != "forward":
        p.adjoint_dev(s["f"].data_ptr(), s["h_out"].data_ptr(), st)
        out.append(s["h_out"])
    return out


# ------------------------------------------------------------------- work --
def _transform_work(N, n, M, m, real):
    """Bytes (nodes, input, output) and flops (roll-off, FFT, taps) of one transform."""
    d = len(N)
    cells, grid = math.prod(N), math.prod(n)
    taps = (2 * m + 2) ** d
    flops = 5.0 * grid * math.log2(grid) + 2.0 * cells + 4.0 * M * taps
    return 8.0 * d * M + 2.0 * real * (cells + M), flops


def work(case):
    real = 8 if case["double"] else 4
    if case["path"] == "batch":
        r = np.random.default_rng([case["P"], case["R"], case["M"]])
        side = r.choice([64, 96, 128, 192, 256], case["P"])
        M = r.integers(4096, case["M"], case["P"], endpoint=True)
        nb = nf = 0.0
        for a, b in zip(side, M):
            a, b = int(a), int(b)
            _, fl = _transform_work([a, a], [2 * a, 2 * a], b, case["m"], real)
            nb += 16.0 * b + case["R"] * 4.0 * real * (a * a + b)
            nf += 2 * case["R"] * fl
        return {"bytes": nb, "flops": nf}
    N, n = _sizes(case)
    by, fl = _transform_work(N, n, case["M"], case["m"], real)
    d, M = case["d"], case["M"]
    inout = by - 8.0 * d * M
    dirs = case.get("dirs", "both")
    if dirs != "both":
        return {"bytes": by, "flops": fl}
    if case["path"] == "autograd":
        # forward, adjoint and the d derivative sums; the node gradient is written
        taps = (2 * case["m"] + 2) ** d
        return {"bytes": 8.0 * d * M + 2 * inout + 8.0 * d * M,
                "flops": 3 * fl + 4.0 * d * M * taps}
    if case["path"] == "solve":
        return {"bytes": 8.0 * d * M + real * M + inout, "flops": 2.0 * fl * (case["iters"] + 1)}
    return {"bytes": 8.0 * d * M + 2 * inout, "flops": 2 * fl}


# ------------------------------------------------------------------ exact --
class _Sums:
    """Forward, adjoint and node gradient of one geometry in 64 bits."""

    def __init__(self, N, n, m, window, x):
        self.N, self.n, self.m, self.d = N, n, m, len(N)
        self.idx, self.w, self.dw, roll = [], [], [], []
        l = torch.arange(2 * m + 2, device="cuda")
        for t in range(self.d):
            sigma = n[t] / N[t]
            nx = n[t] * x[:, t]
            u = torch.round(nx) - torch.signbit(x[:, t]).double() - m
            s = (nx - u)[:, None] - l.double()[None, :]
            k = torch.arange(N[t], device="cuda", dtype=torch.float64) - N[t] // 2
            if window == "kb":
                b = math.pi * (2 - 1 / sigma)
                q = m * m - s * s
                r = q.abs().sqrt()
                z, safe = b * r, r.clamp_min(1e-300)
                w = torch.where(q > 0, torch.sinh(z), torch.sin(z)) / (math.pi * safe)
                dw = torch.where(q > 0, -s * (z * torch.cosh(z) - torch.sinh(z)),
                                 s * (z * torch.cos(z) - torch.sin(z))) / (math.pi * safe ** 3)
                # near |s| = m by the power series of sinh(b r) / r in q
                near = q.abs() < 1e-3
                b2 = b * b
                w = torch.where(near, (b / math.pi) * (1 + b2 * q / 6 + (b2 * q) ** 2 / 120
                                                      + (b2 * q) ** 3 / 5040), w)
                dw = torch.where(near, -2 * s * (b * b2 / math.pi) * (
                    1 / 6 + b2 * q / 60 + (b2 * q) ** 2 / 1680 + (b2 * q) ** 3 / 90720), dw)
                arg = m * torch.sqrt(b * b - (2 * math.pi * k / n[t]) ** 2)
                roll.append(1 / torch.special.i0(arg))
            else:
                b = 2 * sigma / (2 * sigma - 1) * m / math.pi
                w = torch.exp(-s * s / b) / math.sqrt(math.pi * b)
                dw = -2 * s / b * w
                roll.append(torch.exp(math.pi ** 2 * b / n[t] ** 2 * k * k))
            self.idx.append((u.long()[:, None] + l[None, :]) % n[t])
            self.w.append(w)
            self.dw.append(n[t] * dw)
        self.roll = roll[0]
        for v in roll[1:]:
            self.roll = self.roll[..., None] * v
        self.pos = [(torch.arange(N[t], device="cuda") - N[t] // 2) % n[t] for t in range(self.d)]

    def _taps(self, w):
        """(flat grid index (M, W), weight (M, W)) over the last axis, tap by tap of
        the axes before it."""
        W, d = 2 * self.m + 2, self.d
        last = self.idx[d - 1]
        for q in range(W ** (d - 1)):
            at, wt, rem = 0, 1.0, q
            for t in range(d - 2, -1, -1):
                stride = math.prod(self.n[t + 1:])
                at = at + self.idx[t][:, rem % W] * stride
                wt = wt * w[t][:, rem % W]
                rem //= W
            if d == 1:
                yield last, w[0]
            else:
                yield at[:, None] + last, wt[:, None] * w[d - 1]

    def _grid(self, fhat):
        g = torch.zeros(self.n, dtype=torch.complex128, device="cuda")
        v = fhat.to(torch.complex128).view(self.N) * self.roll
        g[torch.meshgrid(*self.pos, indexing="ij")] = v
        return torch.fft.fftn(g).reshape(-1)

    def _gather(self, g, w):
        f = 0
        for at, wt in self._taps(w):
            f = f + (g[at] * wt).sum(1)
        return f

    def forward(self, fhat):
        return self._gather(self._grid(fhat), self.w)

    def node_gradient(self, fhat, v):
        g, out = self._grid(fhat), []
        for t in range(self.d):
            w = [self.dw[k] if k == t else self.w[k] for k in range(self.d)]
            out.append((v.to(torch.complex128).conj() * self._gather(g, w)).real)
        return torch.stack(out, 1)

    def adjoint(self, f):
        f = f.to(torch.complex128)
        re = torch.zeros(math.prod(self.n), dtype=torch.float64, device="cuda")
        im = torch.zeros_like(re)
        for at, wt in self._taps(self.w):
            at = at.reshape(-1)
            re.index_add_(0, at, (f.real[:, None] * wt).reshape(-1))
            im.index_add_(0, at, (f.imag[:, None] * wt).reshape(-1))
        g = torch.complex(re, im).view(self.n)
        h = torch.fft.ifftn(g, norm="forward")
        return (h[torch.meshgrid(*self.pos, indexing="ij")] * self.roll).reshape(-1)


def _solve(sums, y, w, iters):
    """CGNR from zero: the iterate and the weighted relative residuals."""
    y, w = y.to(torch.complex128), w.double()
    wn = lambda v: float((w * (v.real ** 2 + v.imag ** 2)).sum())   # noqa: E731
    r = y
    z = sums.adjoint(w * r)
    f, p, zz = torch.zeros_like(z), z, float(z.abs().square().sum())
    hist = [math.sqrt(wn(r) / wn(y))]
    for _ in range(iters):
        v = sums.forward(p)
        a = zz / wn(v)
        f, r = f + a * p, r - a * v
        z = sums.adjoint(w * r)
        zn = float(z.abs().square().sum())
        p, zz = z + (zn / zz) * p, zn
        hist.append(math.sqrt(wn(r) / wn(y)))
    return f, np.array(hist)


def exact(case, seed):
    m = case["m"]
    if case["path"] == "batch":
        N, _, probs = _batch_inputs(case, seed)
        out = []
        for side, (x, fhat, f) in zip(N.tolist(), probs):
            sums = _Sums(side, [2 * v for v in side], m, "gauss", x)
            out.append((torch.stack([sums.forward(v) for v in fhat]),
                        torch.stack([sums.adjoint(v) for v in f])))
        return out
    N, n = _sizes(case)
    x, fhat, f = _inputs(case, seed)
    sums = _Sums(N, n, m, case["window"], x)
    if case["path"] == "solve":
        h, hist = _solve(sums, f, _radius_weights(case, x), case["iters"])
        return h, hist
    if case["path"] == "autograd":
        return sums.forward(fhat), sums.adjoint(f), sums.node_gradient(fhat, f)
    dirs = case.get("dirs", "both")
    out = []
    if dirs != "adjoint":
        out.append(sums.forward(fhat))
    if dirs != "forward":
        out.append(sums.adjoint(f))
    return tuple(out) if case["path"] == "host" else out
