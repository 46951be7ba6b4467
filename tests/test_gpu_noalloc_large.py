"""No-allocation gridding of large 3D plans on small grids: what the static scratch holds with items
of the uncapped length goes through, and equals gridding with a caller's scratch bit for bit."""

import pytest
import torch

from mr_recon_amd import ops
from mr_recon_amd.plan import SamplePlan, item_lengths

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,npts,batch", [(80, 14_000_000, 1), (64, 8_000_000, 2)])
def test_large_plan_fits(dev, G, npts, batch):
    g = torch.Generator(device=dev).manual_seed(npts)
    k = torch.rand((npts, 3), generator=g, device=dev) * G
    plan = SamplePlan(k, (G,) * 3, 4.0, 9.0)
    assert plan.S == item_lengths(npts, 3)[-1]
    y = torch.randn((batch, npts), dtype=torch.complex64, generator=g, device=dev)
    ref = torch.empty((batch, G, G, G), dtype=torch.complex64, device=dev)
    ops.gridding(y, plan, ref)
    got = torch.full_like(ref, float("nan"))
    ops.gridding_noalloc(y, plan, got)
    assert torch.equal(got, ref)


def test_short_items_where_nothing_is_lost(dev):
    """More tiles than the scratch has subgrids for: no batch fits with either length."""
    G, npts = 160, 3_000_000
    k = torch.rand((npts, 3), generator=torch.Generator(device=dev).manual_seed(1), device=dev) * G
    plan = SamplePlan(k, (G,) * 3, 4.0, 9.0)
    assert plan.S == 2560 and plan.nitems == int(plan.tile_items[-1])
    with pytest.raises(RuntimeError, match="scratch"):
        ops.gridding_noalloc(torch.zeros((1, npts), dtype=torch.complex64, device=dev), plan,
                             torch.empty((1, G, G, G), dtype=torch.complex64, device=dev))
