"""GPU parity of the 3D gridding reduction by point pairs with the oracle: odd and even last
extents, extents that leave a one-point tile past the wrap (three covering tiles per dim), even
and odd subgrid edges, batch counts around a thread's (1 has a kernel of its own), tiles cut into
many items, and accumulation into a grid."""

import numpy as np
import pytest
import torch

from helpers import rel_l2
from oracle import interp_ref

pytestmark = pytest.mark.gpu

TOL = 1e-5  # fp32 sums of a few thousand terms: ~sqrt(terms) x 6e-8


@pytest.mark.parametrize("G", [(20, 17, 33), (16, 24, 25), (33, 19, 16), (25, 16, 31), (17, 18, 22)])
@pytest.mark.parametrize("width", [4.0, 5.0, 6.0])
def test_pairs_vs_oracle(dev, G, width):
    from mr_recon_amd import ops
    from mr_recon_amd.plan import SamplePlan

    rng = np.random.default_rng(int(width) + sum(G))
    k = np.concatenate([rng.random((1500, 3)) * np.array(G), rng.random((900, 3)) * 3.0])  # the origin tile is hot
    k = torch.from_numpy(k[rng.permutation(len(k))].astype(np.float32))
    for C, S in ((1, 16), (3, 32), (4, 256), (5, 16)):
        y = torch.randn((C, k.shape[0]), dtype=torch.complex64, generator=torch.Generator().manual_seed(C))
        plan = SamplePlan(k.to(dev), G, width, 2.3 * width, samples_per_item=S)
        out = torch.empty((C, *G), dtype=torch.complex64, device=dev)
        ops.gridding(y.to(dev), plan, out)
        ref = interp_ref.grid(y, k, G, width, beta=2.3 * width)
        assert rel_l2(out, ref) < TOL
        prev = torch.randn((C, *G), dtype=torch.complex64, generator=torch.Generator().manual_seed(9)).to(dev)
        both = prev.clone()
        ops.gridding(y.to(dev), plan, both, accumulate=True)
        assert rel_l2(both - prev, out) < TOL
