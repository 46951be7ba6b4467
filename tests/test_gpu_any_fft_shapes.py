"""GPU parity of the run-time-length transforms for every launch shape that lengths 2..640 reach
(threads and transforms of a block, direct / chirp-z / radix 17 and 19): each shape along the
contiguous axis, along a strided axis and inside a Toeplitz transform, with partly filled blocks of
rows and columns. tests/test_host_any_plan.py checks that no shape is left out.

Tolerance as in test_gpu_any_fft.py: transforms of up to 2 L points in fp32, three dimensions."""

import math

import pytest
import torch

from helpers import rel_l2
from test_gpu_any_fft import TOL, _rand, _ref_crop, _ref_pad

pytestmark = pytest.mark.gpu

# direct 256 / 512 / 1024 threads and 8 transforms; chirp-z likewise; radix 17 / 19 likewise
LENGTHS = [88, 169, 289, 352, 377, 630, 637, 97, 129, 211, 293, 353, 631, 34, 152, 266, 340, 608, 578]


def _cases():
    for i, L in enumerate(LENGTHS):
        n = max(2, int(0.8 * L))
        yield (18, n), (22, L), (3, 17, 8)[i % 3]
        yield (n, 19), (L, 26), (2, 16, 5)[i % 3]
        yield (4, n, 6), (5, L, 9), 3


@pytest.mark.parametrize("N,G,ns", list(_cases()))
def test_launch_shapes(dev, N, G, ns):
    from mr_recon_amd import ops

    assert ops.fused_any_supported(G) and not ops.fused_supported(G)
    seed = sum(N) + ns
    x, smaps = _rand((1, *N), seed, dev), _rand((ns, *N), seed + 1, dev)
    one, cen = torch.ones(sum(N), device=dev), tuple(n // 2 for n in N)
    got = ops.pad_fft(x, N, G, smaps=smaps)
    assert rel_l2(got, _ref_pad(x, N, G, cen, smaps, one, 1.0).to(got.dtype)) < TOL
    grid = _rand((1, ns, *G), seed + 2, dev)
    want = _ref_crop(grid, N, G, cen, smaps, one, 1.0, True)
    got = ops.ifft_crop(grid.clone(), N, G, 1, smaps=smaps)
    assert rel_l2(got, want.to(got.dtype)) < TOL
    kern = _rand(G, seed + 3, dev) / math.prod(G)
    spec = _ref_pad(x, N, G, cen, smaps, one, 1.0) * kern.to(torch.complex128)
    want = _ref_crop(spec, N, G, cen, smaps, one, 1.0, True)
    got = ops.toeplitz_normal(x[0], N, G, smaps, kern)
    assert rel_l2(got, want.to(got.dtype)) < TOL


@pytest.mark.parametrize("L,tol", [(88, 1.2e-7), (90, 1.2e-7), (136, 1.2e-7), (152, 1.2e-7), (340, 1.2e-7),
                                   (97, 3e-7), (211, 3e-7), (467, 3e-7)])
def test_rows_against_64_bits(dev, L, tol):
    """Relative L2 error of rows of random values. A rounding to 32 bits adds about 0.3e-7; a direct
    transform of two or three passes rounds a value some ten times, in its twiddle products and
    sums (radix 17 and 19 sum in 64 bits); the chirp-z form is two transforms of 2 L points and three
    products."""
    from mr_recon_amd import ops

    x = _rand((512, L), L, dev)
    got = ops.pad_fft(x, (L,), (L,), center=(0,)).to(torch.complex128)
    want = torch.fft.fft(x.to(torch.complex128), dim=-1)
    assert float((got - want).norm() / want.norm()) < tol
