"""Phase-1 gridding writes the subgrids of its own (item, coil) slots and nothing else: coil counts
that leave a matrix block partly or wholly without coils (2D blocks of 2 coils with 4 ring slots, 4
single coils with 8; 3D blocks of 2), samples on the lattice (8 ring slots for P = 5), and a guard
behind the last slot. Slot by slot against the per-lane kernel, so that a store past a coil's
subgrid shows in its neighbour."""

import numpy as np
import pytest
import torch

from test_gpu_grid_mfma import grid_kernel

pytestmark = pytest.mark.gpu

TOL = 1e-5  # fp32 sums of a few thousand terms: ~sqrt(terms) x 6e-8
GUARD = 1 << 16


def _scratch(plan, y, mode):
    from mr_recon_amd import ops

    need = ops.gridding_scratch_elems(plan, y.shape[0])
    buf = torch.full((need + GUARD,), complex(7.0, -3.0), dtype=torch.complex64, device=y.device)
    with grid_kernel(mode):
        ops.gridding_partial(y, plan, y.shape[0], scratch=buf)
    assert bool((buf[need:] == complex(7.0, -3.0)).all())
    return buf[:need].view(plan.nitems * y.shape[0], plan.subgrid)


@pytest.mark.parametrize("D,width,tile", [(2, 2.0, 16), (2, 4.0, 8), (2, 4.0, 16), (2, 4.0, 32), (2, 6.0, 8),
                                          (2, 6.0, 16), (2, 6.0, 32), (2, 7.0, 16), (3, 2.0, 8), (3, 4.0, 8),
                                          (3, 6.0, 8)])
@pytest.mark.parametrize("lattice", [0.0, 0.05])
def test_slots_and_guard(dev, D, width, tile, lattice):
    from mr_recon_amd.plan import SamplePlan

    G = (45, 50) if D == 2 else (17, 20, 19)
    rng = np.random.default_rng(int(10 * width) + tile)
    k = rng.random((900, D)) * np.array(G)
    on = rng.random(len(k)) < lattice
    k[on] = np.floor(k[on]) + (width / 2 - np.floor(width / 2))
    plan = SamplePlan(torch.from_numpy(k.astype(np.float32)).to(dev), G, width, 2.3 * width, tile=tile,
                      samples_per_item=64)
    for C in (1, 2, 3, 5, 6, 7, 9):
        y = torch.randn((C, 900), dtype=torch.complex64, generator=torch.Generator().manual_seed(C)).to(dev)
        a, b = _scratch(plan, y, 1).to(torch.complex128), _scratch(plan, y, 0).to(torch.complex128)
        off = torch.linalg.vector_norm(a - b, dim=1)
        assert bool((off <= TOL * torch.linalg.vector_norm(b, dim=1)).all())
