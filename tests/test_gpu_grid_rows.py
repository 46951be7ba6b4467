"""GPU parity of the matrix-core gridding kernels that accumulate in registers, where they can go
wrong: 2D rows of corners in 8-corner windows (tile edges 8, 16, 32; kernel points P = 2..8; coil
counts around a wave's), rows that an item never reaches, samples on the lattice (the fifth row
of P = 5 takes a ring of 8 slots), items cut at arbitrary places, and k-space values that are not
finite, which must stay inside their own patch. Against the oracle and the per-lane kernel."""

import numpy as np
import pytest
import torch

from helpers import edge_coords, rel_l2
from oracle import interp_ref
from test_gpu_grid_mfma import grid_kernel

pytestmark = pytest.mark.gpu

TOL = 1e-5  # fp32 sums of a few thousand terms: ~sqrt(terms) x 6e-8


def _both(dev, k, y, G, width, beta, S=None, tile=None, dcf=None):
    from mr_recon_amd import ops
    from mr_recon_amd.plan import SamplePlan

    plan = SamplePlan(k.to(dev), G, width, beta, samples_per_item=S, tile=tile)
    outs = []
    for mode in (1, 0):
        out = torch.empty((y.shape[0], *G), dtype=torch.complex64, device=dev)
        with grid_kernel(mode):
            ops.gridding(y.to(dev), plan, out, dcf=None if dcf is None else dcf.to(dev))
        outs.append(out)
    return outs


def _coords2(G, width, seed, lattice=0.0):
    rng = np.random.default_rng(seed)
    parts = [edge_coords(G, 1200, seed=seed, width=width),
             (5 + rng.random((900, 2)) * 3).astype(np.float32),                        # a hot corner row
             np.repeat((rng.random((6, 2)) * min(G)).astype(np.float32), [1, 3, 4, 5, 64, 131], axis=0)]
    k = np.concatenate(parts).astype(np.float64)
    on = rng.random(len(k)) < lattice
    k[on] = np.floor(k[on]) + (width / 2 - np.floor(width / 2))
    return torch.from_numpy(k[rng.permutation(len(k))].astype(np.float32))


@pytest.mark.parametrize("width", [1.5, 2.0, 3.5, 4.0, 5.0, 6.0, 7.0])
@pytest.mark.parametrize("tile", [8, 16, 32])
def test_rows_vs_oracle_and_lane_kernel(dev, width, tile):
    G = (44, 37)  # odd extents: partial tiles, the generic reduce
    for C in (1, 2, 4, 5, 9):
        k = _coords2(G, width, seed=int(10 * width) + C)
        g = torch.Generator().manual_seed(C)
        y = torch.randn((C, k.shape[0]), dtype=torch.complex64, generator=g)
        dcf = torch.rand(k.shape[0], generator=g) + 0.5
        a, b = _both(dev, k, y, G, width, 2.3 * width, tile=tile, dcf=dcf)
        assert rel_l2(a, b) < TOL
        if width >= 2:  # the oracle's kernel has the narrower support of the reference's CPU path below
            assert rel_l2(a, interp_ref.grid(y * dcf, k, G, width, beta=2.3 * width)) < TOL


@pytest.mark.parametrize("frac", [0.0, 0.01, 1.0])
@pytest.mark.parametrize("S", [1, 63, 64, 65, 300])
def test_rows_lattice_and_item_boundaries(dev, frac, S):
    G = (40, 48)
    k = _coords2(G, 4.0, seed=S, lattice=frac)
    y = torch.randn((6, k.shape[0]), dtype=torch.complex64, generator=torch.Generator().manual_seed(S))
    a, b = _both(dev, k, y, G, 4.0, 9.0, S=S)
    ref = interp_ref.grid(y, k, G, 4.0, beta=9.0)
    assert rel_l2(a, ref) < TOL and rel_l2(a, b) < TOL


@pytest.mark.parametrize("D,width", [(2, 4.0), (2, 6.0), (3, 4.0), (3, 6.0)])
def test_non_finite_samples_stay_in_their_patch(dev, D, width):
    G = (32,) * D
    rng = np.random.default_rng(7)
    k = torch.from_numpy((rng.random((700, D)) * 32).astype(np.float32))
    y = torch.randn((3, 700), dtype=torch.complex64, generator=torch.Generator().manual_seed(1))
    y[0, 5] = complex(float("inf"), 0.0)
    y[1, 77] = complex(0.0, float("nan"))
    y[2, 300] = complex(3e38, -3e38)
    a, b = _both(dev, k, y, G, width, 2.3 * width, S=128)
    fa, fb = torch.isfinite(torch.view_as_real(a)), torch.isfinite(torch.view_as_real(b))
    assert torch.equal(fa, fb) and not fa.all() and fa.float().mean() > 0.9
    ok = fa.all(-1) & (b.abs() < 1e25)  # outside the patches of the three samples
    assert rel_l2(a[ok], b[ok]) < TOL
