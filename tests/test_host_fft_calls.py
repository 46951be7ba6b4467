"""Host side of the fused FFT calls (no GPU): what is refused before anything is launched, and the
tables they read."""

import pytest
import torch

from mr_recon_amd import ops

# grids with compiled radix plans, with run-time plans, and beyond both
GRIDS = [((50, 48), (64, 64)), ((50, 41), (61, 52)), ((600, 30), (700, 40))]


@pytest.mark.parametrize("N,G", GRIDS)
@pytest.mark.parametrize("trailing", [lambda N: (N[0], N[1] - 1), lambda N: (N[0] - 3, N[1]), lambda N: N[::-1]])
def test_toeplitz_refuses_maps_of_another_shape(N, G, trailing):
    """Maps smaller than the image would be read past their end."""
    x, kern = torch.zeros(N, dtype=torch.complex64), torch.zeros(G, dtype=torch.complex64)
    with pytest.raises(ValueError, match="image shape"):
        ops.toeplitz_normal(x, N, G, torch.zeros((3, *trailing(N)), dtype=torch.complex64), kern)
