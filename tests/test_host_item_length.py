"""The rules for the length of a work item (no GPU)."""

import pytest

from mr_recon_amd import plan


@pytest.mark.parametrize("npts,ndim,want", [(1, 2, (256,)), (262144, 3, (256,)), (262145, 3, (512,)),
                                            (2_621_440, 3, (2560,)), (2_621_441, 3, (2560, 2816)),
                                            (5_120_000, 3, (2560, 5120)), (20_000_000, 3, (2560, 8192)),
                                            (20_000_000, 2, (8192,)), (5_120_000, 1, (5120,))])
def test_lengths(npts, ndim, want):
    assert plan.item_lengths(npts, ndim) == want
    assert plan.default_samples_per_item(npts, ndim) == want[0]


@pytest.mark.parametrize("nitems", [(5898, 2144), (3700, 1500), (5755, 5297), (4800, 4700), (1000, 400), (9000, 4000)])
@pytest.mark.parametrize("P", [4, 5, 7])
def test_no_batch_that_fitted_is_refused(nitems, P):
    """The no-allocation scratch holds as many batch entries as with the longest items."""
    limit, sub = (64 << 20) - 256, (7 + P) ** 3
    i = plan.choose_item_length(nitems, sub, limit)
    for batch in range(1, 70):
        if nitems[-1] * batch * sub * 8 <= limit:
            assert nitems[i] * batch * sub * 8 <= limit
    if limit // (nitems[0] * sub * 8) == limit // (nitems[1] * sub * 8):
        assert i == 0  # the preferred size where it refuses nothing


@pytest.mark.parametrize("npts,ndim,want", [(1000, 2, 256), (262144, 3, 256), (288_000, 3, 512), (409_600, 2, 512),
                                            (640_000, 3, 512), (960_000, 3, 512), (1_536_000, 3, 768),
                                            (5_120_000, 3, 1280), (8_192_000, 2, 4096)])
def test_dcf_length(npts, ndim, want):
    """Half the usual length, but items of 512 samples are not halved."""
    assert plan.dcf_samples_per_item(npts, ndim) == want


@pytest.mark.parametrize("n,npts,coils,want", [
    (64, 7680, 4, 256), (24, 25_600, 8, 256), (24, 51_200, 4, 256), (12, 49_920, 8, 256), (4, 102_400, 8, 256),
    (24, 25_600, 16, 512), (24, 40_960, 8, 512), (12, 102_400, 8, 512), (2, 512_000, 8, 512), (12, 49_920, 32, 512),
    (32, 51_200, 8, 768), (24, 76_800, 12, 1024), (16, 131_072, 16, 1024), (24, 409_600, 8, 1024), (0, 1, 1, 256)])
def test_batch_length(n, npts, coils, want):
    """Longer items only where enough waves are left to fill the device."""
    assert plan.batch_samples_per_item([(npts, coils)] * n) == want
