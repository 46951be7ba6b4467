"""Work that users of this package have it do, as timed cases.

A case is a dict of plain values. ``listed()`` gives the standing ones, ``draw(rng)`` another of
the same ranges, ``prepare`` what a program holds before the call (inputs, operators and their
sample plans), ``run`` one pass through the public entry points, ``work`` the bytes and operations
a pass cannot do without and ``exact`` the pass's results in 64 bits, by plain torch.

Trajectories are radial, spiral (2D) and kooshball (3D), rotated by the seed; coil maps are smooth,
images and k-space complex Gaussian. Density compensation is the sample's share of k-space area
(volume), so that A^H D A is near the identity and CG-SENSE is well conditioned.
"""

from __future__ import annotations

import math
import random

import torch

from mr_recon_amd import diff
from mr_recon_amd.algs import density_compensation
from mr_recon_amd.batched import BatchedSense, Problem
from mr_recon_amd.fourier import hip_nufft
from mr_recon_amd.linops import sense_linop
from mr_recon_amd.recons import CG_SENSE_recon

MAX_EIGEN = 1.2   # bound on the eigenvalues of A^H D A used to scale the CG systems
LAMDA = 0.05      # regularisation of the CG systems


def listed():
    return [
        # one small 2D image forward and adjoint (a preview, a calibration region, a unit test):
        # launches and host work
        dict(name="nufft2d_64", kind="nufft", im="64x64", coils=1, traj="radial", lines=32, read=128, width=6.0, os=2.0),
        # 2D spiral SENSE, a slice of an ordinary study, each direction
        dict(name="sense2d_fwd", kind="forward", im="256x256", coils=16, traj="spiral", lines=32, read=4096, width=4.0,
             os=1.25),
        dict(name="sense2d_adj", kind="adjoint", im="256x256", coils=16, traj="spiral", lines=32, read=4096, width=4.0,
             os=1.25),
        # odd image and coil counts, wide kernel: the normal operator inside an iterative solver
        dict(name="sense2d_odd", kind="normal", im="230x187", coils=11, traj="radial", lines=233, read=461, width=6.0,
             os=1.25),
        # 3D kooshball SENSE at the benchmark's size, each direction
        dict(name="sense3d_fwd", kind="forward", im="128x128x128", coils=32, traj="kooshball", lines=20000, read=256,
             width=4.0, os=1.25),
        dict(name="sense3d_adj", kind="adjoint", im="128x128x128", coils=32, traj="kooshball", lines=20000, read=256,
             width=4.0, os=1.25),
        # 3D volume with ragged extents, few coils (after coil compression), wide kernel
        dict(name="sense3d_odd", kind="normal", im="90x104x77", coils=7, traj="kooshball", lines=4001, read=190, width=6.0,
             os=1.25),
        # Toeplitz normal operator of a 3D volume
        dict(name="toep3d", kind="toeplitz", im="96x96x96", coils=16, traj="kooshball", lines=6000, read=192, width=4.0,
             os=1.25),
        # a whole CG-SENSE reconstruction of a slice (Toeplitz normal operator)
        dict(name="cg2d", kind="cg", im="256x256", coils=16, traj="spiral", lines=32, read=4096, width=4.0, os=1.25,
             iters=15),
        # many uneven slices reconstructed at once from one captured graph
        dict(name="batched2d", kind="batched", problems=24, mix=2024, width=4.0, os=1.25, iters=8),
        # trajectory optimisation: loss, image and trajectory gradients through an unrolled CG
        dict(name="grad2d", kind="grad", im="256x256", coils=16, traj="spiral", lines=64, read=2048, width=6.0, os=1.25,
             iters=4),
        # density compensation of a new 3D trajectory (the sample plan is part of the call)
        dict(name="dcf3d", kind="dcf", im="96x96x96", coils=1, traj="kooshball", lines=8000, read=192, width=4.0, os=1.0,
             iters=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: image edges 48..320 (2D) and 32..128 (3D), 1..32 coils, kernel widths 4 and 6,
    oversampling 1.25 and 2, sample counts from a tenth to a few times the pixels."""
    kind = rng.choice(["nufft", "forward", "adjoint", "normal", "forward", "adjoint", "normal", "toeplitz", "cg", "batched",
                       "grad", "dcf"])
    width = rng.choice([4.0, 4.0, 6.0])
    os_ = rng.choice([1.25, 1.25, 2.0])
    if kind == "batched":
        return dict(kind=kind, problems=rng.randint(4, 24), mix=rng.randint(0, 10 ** 6), width=width, os=1.25,
                    iters=rng.randint(4, 10))
    three_d = kind == "dcf" or (kind in ("nufft", "forward", "adjoint", "normal", "toeplitz") and rng.random() < 0.5)
    if three_d:
        n = [_log(rng, 32, 112) for _ in range(3)]
        n = [n[0]] * 3 if rng.random() < 0.4 else n
        coils = _log(rng, 1, 16)
        read = 2 * max(n)
        lines = _log(rng, 500, 8000)
        traj = "kooshball"
    else:
        n = [_log(rng, 48, 320) for _ in range(2)]
        n = [n[0]] * 2 if rng.random() < 0.4 else n
        coils = _log(rng, 1, 32)
        traj = rng.choice(["radial", "spiral"])
        read = 2 * max(n) if traj == "radial" else rng.randint(1000, 4096)
        lines = rng.randint(max(16, max(n) // 2), 2 * max(n)) if traj == "radial" else rng.randint(8, 48)
    if kind == "toeplitz":
        n = [v + v % 2 for v in n]
    c = dict(kind=kind, im="x".join(map(str, n)), coils=1 if kind == "dcf" else coils, traj=traj, lines=lines, read=read,
             width=4.0 if kind == "dcf" else width, os=1.0 if kind == "dcf" else os_)
    if kind in ("cg", "grad", "dcf"):
        c["iters"] = {"cg": rng.randint(8, 20), "grad": rng.randint(2, 4), "dcf": rng.randint(10, 30)}[kind]
    if kind == "cg":
        c["im"] = "x".join(str(v + v % 2) for v in n)
    return c


# ---------------------------------------------------------------------------------------------
# inputs

def _im(case):
    return tuple(int(v) for v in case["im"].split("x"))


def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1009 + salt)
    return g


def _randn(shape, g):
    """Complex Gaussian, unit variance."""
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.complex64)


def _trajectory(traj, im, lines, read, seed):
    """(trj (lines, read, d) float32 in cycles per FOV, dcf (lines, read) float32): rotated by the seed."""
    r0 = random.Random(int(seed) * 7919 + 13)
    f = dict(dtype=torch.float64, device="cuda")
    d = len(im)
    if traj == "spiral":
        tau = torch.arange(read, **f) / read
        r = 0.5 * tau ** 1.5
        dr = 0.75 * tau ** 0.5 / read
        turns = max(im) / (2.0 * lines)
        ph = 2 * math.pi * (turns * tau[None] + (torch.arange(lines, **f) / lines)[:, None] + r0.random())
        k = torch.stack([r * torch.cos(ph), r * torch.sin(ph)], -1)
        share = 2 * math.pi * r * dr / lines
        share[0] = share[1] * 0.1
        share = share[None].expand(lines, read)
    else:
        r = (torch.arange(read, **f) - read // 2) / read
        if traj == "radial":
            th = math.radians(111.246) * torch.arange(lines, **f) + 2 * math.pi * r0.random()
            u = torch.stack([torch.cos(th), torch.sin(th)], -1)
        else:
            i = torch.arange(lines, **f) + 0.5
            z = 1 - 2 * i / lines
            ph = math.pi * (3 - math.sqrt(5)) * i + 2 * math.pi * r0.random()
            s = torch.sqrt(1 - z * z)
            u = torch.stack([s * torch.cos(ph), s * torch.sin(ph), z], -1)
        k = u[:, None] * r[None, :, None]
        ra = torch.clamp(r.abs(), min=0.25 / read)
        share = math.pi * ra / (lines * read) if d == 2 else 2 * math.pi * ra * ra / (lines * read)
        share = share[None].expand(lines, read)
    n = torch.tensor(im, **f)
    return (k * n).float().contiguous(), (share * float(math.prod(im))).float().contiguous()


def _maps(coils, im, seed):
    """Smooth coil maps (coils, *im), root sum of squares 1."""
    r0 = random.Random(int(seed) * 104729 + 7)
    ax = [(torch.arange(n, device="cuda") - n // 2) / n for n in im]
    m = []
    for c in range(coils):
        e = 0
        cen = [r0.gauss(0, 1) for _ in im]
        nrm = math.sqrt(sum(v * v for v in cen)) or 1.0
        for a, v in zip(torch.meshgrid(*ax, indexing="ij"), cen):
            e = e + (a - 0.4 * v / nrm) ** 2
        ph = 2 * math.pi * r0.random()
        m.append(torch.exp(-e / 0.3) * complex(math.cos(ph), math.sin(ph)))
    m = torch.stack(m)
    return (m / m.abs().square().sum(0, keepdim=True).sqrt()).to(torch.complex64).contiguous()


def _mix(case):
    """Sizes of the batched problems: (edge, coils, trajectory, lines, readout)."""
    r = random.Random(int(case["mix"]))
    out = []
    for _ in range(case["problems"]):
        n, c, m = r.choice([128, 192, 256]), r.choice([8, 16, 32]), r.randint(20000, 130000)
        out.append((n, c, "radial", -(-m // (2 * n)), 2 * n) if r.random() < 0.5 else (n, c, "spiral", 16, -(-m // 16)))
    return out


def _nufft(case):
    return hip_nufft(_im(case), oversamp=case["os"], width=case["width"])


def _inputs(case, seed):
    """Trajectory, density compensation, maps, image and k-space of a single-problem case."""
    im, C = _im(case), case["coils"]
    trj, dcf = _trajectory(case["traj"], im, case["lines"], case["read"], seed)
    g = _gen(seed)
    mps = _maps(C, im, seed)
    x = _randn(im, g)
    y = _randn((C, case["lines"], case["read"]), g)
    return trj, dcf, mps, x, y


def _batched_inputs(case, seed):
    out = []
    for i, (n, c, traj, lines, read) in enumerate(_mix(case)):
        trj, dcf = _trajectory(traj, (n, n), lines, read, seed * 131 + i)
        out.append((trj.reshape(-1, 2), dcf.reshape(-1), _maps(c, (n, n), seed * 131 + i),
                    _randn((c, lines * read), _gen(seed, 1 + i))))
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, kind=kind)
    if kind == "batched":
        ps = _batched_inputs(case, seed)
        B = BatchedSense([Problem(t, m, d) for t, d, m, _ in ps], oversamp=case["os"], width=case["width"])
        B.capture(num_iters=case["iters"], lamda_l2=LAMDA, max_eigen=MAX_EIGEN)
        s.update(B=B, ksp=[y for *_, y in ps])
        return s
    if kind == "dcf":
        s.update(trj=_trajectory(case["traj"], _im(case), case["lines"], case["read"], seed)[0])
        return s
    trj, dcf, mps, x, y = _inputs(case, seed)
    nf = _nufft(case)
    if kind == "nufft":
        g = _gen(seed, 3)
        s.update(nf=nf, trj=trj[None], img=_randn((1, case["coils"], *_im(case)), g), ksp=y[None])
        nf.plan(s["trj"][0])
        return s
    if kind == "grad":
        s.update(nf=nf, trj=trj, mps=mps, dcf=dcf, x=x, y=y, x0=_randn(_im(case), _gen(seed, 5)))
        return s
    s.update(A=sense_linop(trj, mps, dcf=dcf, nufft=nf, use_toeplitz=kind in ("toeplitz", "cg")), x=x, y=y)
    return s


def run(s):
    kind = s["kind"]
    if kind == "nufft":
        return s["nf"].forward(s["img"], s["trj"]), s["nf"].adjoint(s["ksp"], s["trj"])
    if kind == "forward":
        return s["A"].forward(s["x"])
    if kind == "adjoint":
        return s["A"].adjoint(s["y"])
    if kind in ("normal", "toeplitz"):
        return s["A"].normal(s["x"])
    if kind == "cg":
        return CG_SENSE_recon(s["A"], s["y"], max_iter=s["case"]["iters"], lamda_l2=LAMDA, max_eigen=MAX_EIGEN,
                              tolerance=0.0, clear_gpu_mem=False, verbose=False)
    if kind == "batched":
        return s["B"].replay(s["ksp"])
    if kind == "grad":
        # the trajectory of a training step is a new tensor: its plan is built in the step
        x = s["x"].clone().requires_grad_(True)
        k = s["trj"].clone().requires_grad_(True)
        fit = torch.sum(torch.abs(diff.sense_forward(x, k, s["mps"], s["nf"]) - s["y"]) ** 2)
        rec = diff.unrolled_cg_sense(s["y"], k, s["mps"], s["nf"], num_iters=s["case"]["iters"], lamda_l2=LAMDA,
                                     max_eigen=MAX_EIGEN, dcf=s["dcf"])
        loss = fit + torch.sum(torch.abs(rec - s["x0"]) ** 2)
        loss.backward()
        return loss.detach(), x.grad, k.grad
    return density_compensation(s["trj"], _im(s["case"]), s["case"]["iters"])


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without

def _work(kind, im, C, M, width, os_, iters):
    d = len(im)
    npx = math.prod(im)
    G = math.prod(math.ceil(os_ * n) for n in im)
    pts = math.floor(width) ** d
    one = C * (8.0 * M * pts / 2 + 5.0 * G * math.log2(G))          # interpolation or gridding, and one transform
    toep = C * (2 * 5.0 * 2 ** d * npx * math.log2(2 ** d * npx))   # two transforms of the doubled grid
    maps = 8.0 * C * npx
    ksp = 8.0 * C * M
    crd = 4.0 * d * M
    if kind == "nufft":
        return dict(bytes=2 * (8.0 * C * npx + ksp + crd), flops=2 * one)
    if kind in ("forward", "adjoint"):
        return dict(bytes=8.0 * npx + maps + ksp + crd + (4.0 * M if kind == "adjoint" else 0), flops=one)
    if kind == "normal":
        return dict(bytes=16.0 * npx + maps + crd + 4.0 * M, flops=2 * one)
    if kind == "toeplitz":
        return dict(bytes=16.0 * npx + maps + 8.0 * 2 ** d * npx, flops=toep)
    if kind == "cg":
        return dict(bytes=8.0 * npx + maps + ksp + crd + 4.0 * M + (iters + 1) * (56.0 * npx + maps + 8.0 * 2 ** d * npx),
                    flops=one + (iters + 1) * toep)
    if kind == "batched":
        return dict(bytes=8.0 * npx + maps + ksp + crd + (iters + 1) * (56.0 * npx + maps + crd),
                    flops=one + 2 * (iters + 1) * one)
    if kind == "grad":
        n = 2 + (iters + 1)  # transforms pairs forward; backward repeats them with the trajectory terms
        return dict(bytes=3 * n * (16.0 * npx + maps + crd) + 2 * ksp + crd, flops=2 * 2 * n * one)
    return dict(bytes=iters * (2 * 8.0 * npx + crd + 8.0 * M), flops=iters * 2 * 8.0 * M * pts / 2)


def work(case):
    if case["kind"] == "batched":
        b = f = 0.0
        for n, c, _, lines, read in _mix(case):
            w = _work("batched", (n, n), c, lines * read, case["width"], case["os"], case["iters"])
            b, f = b + w["bytes"], f + w["flops"]
        return dict(bytes=b, flops=f)
    return _work(case["kind"], _im(case), case["coils"], case["lines"] * case["read"], case["width"], case["os"],
                 case.get("iters", 0))


# ---------------------------------------------------------------------------------------------
# the same results in 64 bits

class _Exact:
    """Kaiser-Bessel NUFFT in 64 bits at the 32-bit sample coordinates that define the transform
    (t = fl(fl(k G/N) + G//2) mod G): apodize, zero-pad, transform, interpolate / width^d; adjoint
    its conjugate transpose. Grids are (points, coils). ``k64``: gradients go to it."""

    def __init__(self, im, trj, width, os_, beta=None, scaled=True, k64=None):
        self.im, self.d, self.w = im, len(im), width
        d, dev = self.d, trj.device
        self.G = tuple(math.ceil(os_ * n) for n in im) if scaled else im
        if beta is None:
            beta = math.pi * (((width / os_) * (os_ - 0.5)) ** 2 - 0.8) ** 0.5
        t = trj.reshape(-1, d).float()
        if scaled:
            sc = torch.tensor([G / n for G, n in zip(self.G, im)], dtype=torch.float32, device=dev)
            t = t * sc + torch.tensor([float(G // 2) for G in self.G], device=dev)
        t = torch.remainder(t, torch.tensor(self.G, dtype=torch.float32, device=dev))
        r = width / 2
        P = int(math.floor(width)) + 1
        low = torch.ceil(t - r)
        td = t.double()
        if k64 is not None:
            kk = k64.reshape(-1, d)
            td = td + (kk - kk.detach()) * sc.double()
        self.idx, self.wt = [], []   # per dimension and patch point: grid index and weight
        for a in range(d):
            ii, ww = [], []
            for j in range(P):
                u = (low[:, a].double() + j - td[:, a]) / r
                inside = (u.detach().abs() * r) <= r
                z = (1 - u * u).clamp(min=1e-30).sqrt()
                ww.append(torch.where(inside, torch.special.i0(beta * z), torch.zeros_like(z)))
                g = low[:, a].long() + j - (self.G[a] // 2 if scaled else 0)
                ii.append(torch.remainder(g, self.G[a]))
            self.idx.append(ii)
            self.wt.append(ww)
        self.P, self.M = P, t.shape[0]
        self.npts = math.prod(self.G)
        self.scale = 1.0 / (width ** d * math.sqrt(math.prod(im))) if scaled else 1.0
        apod = torch.ones(im, dtype=torch.float64, device=dev)
        if scaled:
            for a, n in enumerate(im):
                x = (torch.arange(n, dtype=torch.float64, device=dev) - n // 2) / self.G[a]
                q = (beta ** 2 - (math.pi * width * x) ** 2).sqrt()
                shape = [1] * d
                shape[a] = n
                apod = apod * (q / torch.sinh(q)).reshape(shape)
        self.apod = apod
        self.order = None

    def points(self):
        """Flat grid index and weight of every patch point of every sample."""
        for m in range(self.P ** self.d):
            lin, w = 0, 1.0
            for a in range(self.d):
                j = (m // self.P ** (self.d - 1 - a)) % self.P
                lin = lin * self.G[a] + self.idx[a][j]
                w = w * self.wt[a][j]
            yield lin, w

    def _pad(self, x):
        """(*im) pixels of each coil -> spectrum of the padded grid, (points, coils)."""
        C, d = x.shape[0], self.d
        pad = torch.zeros((C, *self.G), dtype=torch.complex128, device=x.device)
        lo = [(G // 2) - n // 2 for G, n in zip(self.G, self.im)]
        sl = tuple([slice(None)] + [slice(a, a + n) for a, n in zip(lo, self.im)])
        pad[sl] = x * self.apod
        dims = tuple(range(1, d + 1))
        pad = torch.roll(pad, [-(G // 2) for G in self.G], dims)
        return torch.fft.fftn(pad, dim=dims).reshape(C, -1).t().contiguous()

    def _crop(self, g):
        """(points, coils) -> (coils, *im): the adjoint of _pad."""
        C, d = g.shape[1], self.d
        dims = tuple(range(1, d + 1))
        x = torch.fft.ifftn(g.t().reshape(C, *self.G), dim=dims, norm="forward")
        x = torch.roll(x, [G // 2 for G in self.G], dims)
        lo = [(G // 2) - n // 2 for G, n in zip(self.G, self.im)]
        return x[tuple([slice(None)] + [slice(a, a + n) for a, n in zip(lo, self.im)])] * self.apod

    def interp(self, g):
        out = torch.zeros((self.M, g.shape[1]), dtype=g.dtype, device=g.device)
        for lin, w in self.points():
            out = out + w[:, None] * g[lin]
        return out

    def grid(self, y):
        """Adjoint of interp: samples sharing a patch corner are summed first, then added at
        distinct points, so that no atomic additions are needed."""
        if self.order is None:
            key = 0
            for a in range(self.d):
                key = key * self.G[a] + self.idx[a][0]
            self.order = torch.argsort(key)
            ks = key[self.order]
            new = torch.ones_like(ks, dtype=torch.bool)
            new[1:] = ks[1:] != ks[:-1]
            self.first = torch.nonzero(new).reshape(-1)
            self.lengths = torch.diff(torch.cat([self.first, self.first.new_tensor([self.M])]))
        ys = torch.view_as_real(y[self.order]).reshape(self.M, -1)
        g = torch.zeros((self.npts, ys.shape[1]), dtype=torch.float64, device=y.device)
        for lin, w in self.points():
            v = torch.segment_reduce(ys * w[self.order][:, None], "sum", lengths=self.lengths, axis=0, unsafe=True)
            at = lin[self.order][self.first]
            g[at] = g[at] + v
        return torch.view_as_complex(g.reshape(self.npts, -1, 2))

    def forward(self, x):
        """x (C, *im) -> (C, M)."""
        return torch.cat([self.interp(self._pad(v)).t() for v in x.to(torch.complex128).split(8)]) * self.scale

    def adjoint(self, y):
        """y (C, M) -> (C, *im)."""
        return torch.cat([self._crop(self.grid(v.t().contiguous())) for v in y.to(torch.complex128).split(8)]) * self.scale


def _exact_cg(normal, b, iters):
    b = b / math.sqrt(MAX_EIGEN)
    A = lambda v: normal(v) / MAX_EIGEN + LAMDA * v  # noqa: E731
    x = b
    r = b - A(x)
    p = r
    rz = torch.sum(r.abs() ** 2)
    for _ in range(iters):
        ap = A(p)
        al = rz / torch.sum((p.conj() * ap).real)
        x = x + al * p
        r = r - al * ap
        rn = torch.sum(r.abs() ** 2)
        p = r + (rn / rz) * p
        rz = rn
    return x


def _exact_toeplitz(im, trj, dcf, width, os_):
    """x -> A^H D A x for one coil by the point spread function on the doubled grid (at 32-bit
    coordinates of the doubled image, as the kernels are built)."""
    d = len(im)
    im2 = tuple(2 * n for n in im)
    E = _Exact(im2, trj * 2.0, width, os_)
    psf = E.adjoint(dcf.reshape(1, -1).to(torch.complex128))[0] * 2.0 ** d
    dims = tuple(range(d))
    # centred orthonormal transform of the kernel, applied between centred orthonormal transforms
    K = torch.fft.fftn(torch.fft.ifftshift(psf, dim=dims), dim=dims, norm="ortho")
    ddims = tuple(range(1, d + 1))
    lo = [(a - n) // 2 for a, n in zip(im2, im)]
    sl = tuple([slice(None)] + [slice(a, a + n) for a, n in zip(lo, im)])

    def apply(v):  # (C, *im)
        p = torch.zeros((v.shape[0], *im2), dtype=torch.complex128, device=v.device)
        p[sl] = v
        f = torch.fft.fftn(p, dim=ddims) * K
        return torch.fft.ifftn(f, dim=ddims)[sl]

    return apply


def _exact_grad(case, seed):
    im = _im(case)
    trj, dcf, mps, x, y = _inputs(case, seed)
    x0 = _randn(im, _gen(seed, 5)).to(torch.complex128)
    m = mps.to(torch.complex128)
    y = y.reshape(y.shape[0], -1).to(torch.complex128)
    D = dcf.reshape(-1).double()
    x = x.to(torch.complex128).requires_grad_(True)
    k = trj.double().requires_grad_(True)
    E = _Exact(im, trj, case["width"], case["os"], k64=k)
    pts = list(E.points())

    class Pad(torch.autograd.Function):
        @staticmethod
        def forward(ctx, v):
            return E._pad(v)

        @staticmethod
        def backward(ctx, g):
            return E._crop(g)

    class Crop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, g):
            return E._crop(g)

        @staticmethod
        def backward(ctx, v):
            return E._pad(v)

    class Interp(torch.autograd.Function):
        """(grid, weights) -> samples; the gradient of the weights by recomputation."""

        @staticmethod
        def forward(ctx, g, *w):
            ctx.save_for_backward(g, *w)
            return sum(wi[:, None] * g[l] for (l, _), wi in zip(pts, w))

        @staticmethod
        def backward(ctx, gy):
            g, *w = ctx.saved_tensors
            gw = [(gy.conj() * g[l]).real.sum(1) for l, _ in pts]
            return (E.grid(gy), *gw)

    class Grid(torch.autograd.Function):
        @staticmethod
        def forward(ctx, v, *w):
            ctx.save_for_backward(v, *w)
            return E.grid(v)

        @staticmethod
        def backward(ctx, gg):
            v, *w = ctx.saved_tensors
            gv = sum(wi[:, None] * gg[l] for (l, _), wi in zip(pts, w))
            return (gv, *[(gg[l].conj() * v).real.sum(1) for l, _ in pts])

    W = [w for _, w in pts]
    for a in range(E.d):
        E.wt[a] = [w.detach() for w in E.wt[a]]

    def fwd(v):
        return Interp.apply(Pad.apply(m * v), *W).t() * E.scale

    def adj(v):
        return (m.conj() * Crop.apply(Grid.apply((v * D).t().contiguous(), *W))).sum(0) * E.scale

    fit = torch.sum(torch.abs(fwd(x) - y) ** 2)
    rec = _exact_cg(lambda v: adj(fwd(v)), adj(y), case["iters"])
    loss = fit + torch.sum(torch.abs(rec - x0) ** 2)
    loss.backward()
    return loss.detach(), x.grad, k.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched":
        out = []
        for (trj, dcf, mps, y), (n, *_) in zip(_batched_inputs(case, seed), _mix(case)):
            E = _Exact((n, n), trj, case["width"], case["os"])
            m = mps.to(torch.complex128)

            def adj(v):
                return (m.conj() * E.adjoint(v * dcf.double())).sum(0)

            out.append(_exact_cg(lambda v: adj(E.forward(m * v)), adj(y), case["iters"]))
        return out
    im = _im(case)
    if kind == "dcf":
        trj = _trajectory(case["traj"], im, case["lines"], case["read"], seed)[0]
        E = _Exact(im, trj, 4.0, 1.0, beta=8.0, scaled=False)
        w = torch.ones(E.M, dtype=torch.float64, device="cuda")
        for _ in range(case["iters"]):
            w = w / E.interp(E.grid(w.to(torch.complex128)[:, None]))[:, 0].abs()
        return (w / w.max()).reshape(trj.shape[:-1])
    if kind == "grad":
        return _exact_grad(case, seed)
    trj, dcf, mps, x, y = _inputs(case, seed)
    C = case["coils"]
    if kind == "nufft":
        img = _randn((1, C, *im), _gen(seed, 3))
        E = _Exact(im, trj, case["width"], case["os"])
        return E.forward(img[0]).reshape(1, *y.shape), E.adjoint(y.reshape(C, -1))[None]
    m = mps.to(torch.complex128)
    D = dcf.reshape(-1).double()
    if kind == "toeplitz":
        T = _exact_toeplitz(im, trj, dcf, case["width"], case["os"])
        return sum((c.conj() * T(c * x)).sum(0) for c in m.split(4))
    E = _Exact(im, trj, case["width"], case["os"])
    if kind == "forward":
        return torch.cat([E.forward(c * x) for c in m.split(8)]).reshape(y.shape)

    def adj(v):
        return sum((c.conj() * E.adjoint(q * D)).sum(0) for c, q in zip(m.split(8), v.reshape(C, -1).split(8)))

    if kind == "adjoint":
        return adj(y)
    if kind == "normal":
        return sum((c.conj() * E.adjoint(E.forward(c * x) * D)).sum(0) for c in m.split(8))
    T = _exact_toeplitz(im, trj, dcf, case["width"], case["os"])
    return _exact_cg(lambda v: (m.conj() * T(m * v)).sum(0), adj(y), case["iters"])
