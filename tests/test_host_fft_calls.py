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


@pytest.mark.parametrize("N,G", GRIDS[1:])
@pytest.mark.parametrize("n", [lambda g: g + 1, lambda g: 2 * g - 1])
def test_ifft_crop_refuses_parts_of_a_grid(N, G, n):
    """Values behind the last whole grid are a mistake of the caller's, not to be dropped."""
    grid = torch.zeros(n(G[0] * G[1]), dtype=torch.complex64)
    with pytest.raises(ValueError, match="whole grids"):
        ops.ifft_crop(grid, N, G, 1)


@pytest.mark.parametrize("tables,L,values", [("_any_fft", 76, 76), ("_any_fft", 97, 97 + 2 * 195), ("_lds_fft", 64, 64)])
def test_tables_under_another_default_device(tables, L, values):
    """The library fills the tables through a host address, whatever device new tensors go to by
    default; the first L values are the length's roots (chirp tables start with those of their M)."""
    from mr_recon_amd import gridfft

    own = type(getattr(gridfft, tables))()
    with torch.device("meta"):
        own.tables(torch.device("cpu"), (L,))
    tab = (own._arr if tables == "_any_fft" else own._tw)[(None, (L,))][0][0]
    assert tab.device.type == "cpu" and tab.numel() == 2 * values
    M = 195 if values > L else L
    got = torch.view_as_complex(tab.view(-1, 2))[:M].to(torch.complex128)
    m = torch.arange(M, dtype=torch.float64)
    want = torch.polar(torch.ones(M, dtype=torch.float64), -2 * torch.pi * m / M)
    assert float((got - want).abs().max()) < 1e-7
