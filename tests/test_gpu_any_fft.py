"""GPU parity of the fused pad+FFT / iFFT+crop / Toeplitz transforms on grid lengths without a
compiled radix plan, against a plain torch fp64 restatement (place pixel n at grid index
(n - c) mod G, torch.fft, the mirror crop and coil reduction).

Tolerance: an fp32 transform of length L by passes of radix up to 16 rounds a few times per
pass, under 1e-6 relative L2; the chirp-z form is two such transforms of 2 L with three more
products. 5e-6 leaves a factor of several over three dimensions."""

import math

import pytest
import torch

from helpers import rel_l2

pytestmark = pytest.mark.gpu

TOL = 5e-6

# smooth lengths of each radix, primes (chirp-z) and their squares, mixtures with compiled
# lengths, the shortest and longest, lengths at the launch-shape limits, images at both ends of N <= G
CASES = [
    ((77,), (97,), 3), ((2,), (2,), 1), ((500,), (640 - 9,), 2), ((300,), (599,), 1),
    ((20, 31), (26, 49), 5), ((230, 187), (288, 234), 3), ((64, 50), (64, 63), 1), ((33, 47), (320, 59), 2),
    ((90, 100), (121, 169), 17), ((400, 20), (630, 22), 2), ((2, 3), (3, 5), 1), ((50, 512), (61, 637), 4),
    ((9, 10, 11), (12, 13, 14), 33), ((30, 26, 24), (37, 33, 31), 7), ((20, 16, 24), (25, 64, 40), 2),
    ((7, 5, 64), (11, 10, 160), 9), ((60, 40), (136, 95), 3), ((11, 70), (17, 323), 2), ((64, 5, 7), (128, 7, 11), 1),
]


def _rand(shape, seed, dev):
    return torch.randn(shape, dtype=torch.complex64, generator=torch.Generator().manual_seed(seed)).to(dev)


def _place(N, G, center):
    return [(torch.arange(n) - c) % g for n, g, c in zip(N, G, center)]


def _ref_pad(x, N, G, center, smaps, apod, scale):
    """x (nx, *N), smaps (ns, *N) -> (nx, ns, *G) complex128."""
    D = len(N)
    a = 1.0
    for d, t in enumerate(apod.double().split(list(N))):
        a = a * t.reshape([-1 if e == d else 1 for e in range(D)])
    v = x.to(torch.complex128)[:, None] * smaps.to(torch.complex128)[None] * a * scale
    g = torch.zeros((*v.shape[:2], *G), dtype=torch.complex128, device=v.device)
    ix = torch.meshgrid(*[i.to(v.device) for i in _place(N, G, center)], indexing="ij")
    g[(slice(None), slice(None), *ix)] = v
    return torch.fft.fftn(g, dim=tuple(range(-D, 0)))


def _ref_crop(grid, N, G, center, smaps, apod, scale, conj):
    D = len(N)
    a = 1.0
    for d, t in enumerate(apod.double().split(list(N))):
        a = a * t.reshape([-1 if e == d else 1 for e in range(D)])
    v = torch.fft.ifftn(grid.to(torch.complex128), dim=tuple(range(-D, 0)), norm="forward")
    ix = torch.meshgrid(*[i.to(v.device) for i in _place(N, G, center)], indexing="ij")
    v = v[(slice(None), slice(None), *ix)]
    s = smaps.to(torch.complex128)
    return (v * (s.conj() if conj else s)[None]).sum(1) * a * scale


@pytest.mark.parametrize("N,G,ns", CASES)
def test_any_lengths(dev, N, G, ns):
    from mr_recon_amd import ops

    assert ops.fused_any_supported(G) and not ops.fused_supported(G)
    seed = sum(N) + sum(G) + ns
    for nx, center, conj in ((1, tuple(n // 2 for n in N), True), (2, tuple(0 for _ in N), False)):
        x = _rand((nx, *N), seed, dev)
        smaps = _rand((ns, *N), seed + 1, dev)
        apod = (torch.rand(sum(N), generator=torch.Generator().manual_seed(seed + 2)) + 0.5).to(dev)
        got = ops.pad_fft(x, N, G, smaps=smaps, apod=apod, scale=0.3, center=center)
        assert rel_l2(got, _ref_pad(x, N, G, center, smaps, apod, 0.3).to(got.dtype)) < TOL
        grid = _rand((nx, ns, *G), seed + 3, dev)
        prev = _rand((nx, *N), seed + 4, dev)
        want = _ref_crop(grid, N, G, center, smaps, apod, 0.3, conj)
        got = ops.ifft_crop(grid.clone(), N, G, nx, smaps=smaps, apod=apod, scale=0.3, center=center, conj_maps=conj)
        assert rel_l2(got, want.to(got.dtype)) < TOL
        got = ops.ifft_crop(grid.clone(), N, G, nx, smaps=smaps, apod=apod, scale=0.3, center=center, conj_maps=conj,
                            out=prev.clone(), accumulate=True)
        assert rel_l2(got, (want + prev).to(got.dtype)) < TOL


@pytest.mark.parametrize("N,G,ns", [c for c in CASES if len(c[0]) > 1])
def test_any_toeplitz(dev, N, G, ns):
    from mr_recon_amd import ops

    seed = sum(N) + 7 * ns
    x = _rand(N, seed, dev)
    smaps = _rand((ns, *N), seed + 1, dev)
    kern = _rand(G, seed + 2, dev) / math.prod(G)
    one = torch.ones(sum(N), device=dev)
    cen = tuple(n // 2 for n in N)
    spec = _ref_pad(x[None], N, G, cen, smaps, one, 1.0) * kern.to(torch.complex128)
    want = _ref_crop(spec, N, G, cen, smaps, one, 1.0, True)
    got = ops.toeplitz_normal(x, N, G, smaps, kern)
    assert rel_l2(got, want.to(got.dtype)) < TOL


def test_without_maps(dev):
    from mr_recon_amd import ops

    N, G = (41, 29), (53, 37)
    x = _rand((5, *N), 3, dev)
    ones = torch.ones((1, *N), dtype=torch.complex64, device=dev)
    one = torch.ones(sum(N), device=dev)
    cen = tuple(n // 2 for n in N)
    want = _ref_pad(x, N, G, cen, ones, one, 1.0)[:, 0]
    got = ops.pad_fft(x, N, G)
    assert got.shape == (5, *G) and rel_l2(got, want.to(got.dtype)) < TOL
    back = ops.ifft_crop(got.clone(), N, G, 5, scale=1.0 / math.prod(G))
    assert rel_l2(back, x) < TOL
