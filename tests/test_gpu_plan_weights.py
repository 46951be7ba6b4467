"""Kaiser-Bessel weights of sample plans against I0 in 64 bits, at the widths and oversampling that
the error figure in common.h is given for, and the entry points with 32-bit shapes.

Tolerance, relative L2 over the weights: the two-float argument with correctly rounded functions
gives 0.6e-7 .. 0.9e-7 (evaluated in numpy); hardware square root, reciprocal root and exponential
(1 ulp each) add in squares up to 3 x (0.35e-7)^2, 1.1e-7 in all. One weight: 9.8.2 of Abramowitz &
Stegun is good to 1.9e-7 / 0.399 and the rounding of eight products to 8 x 0.6e-7."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL, TOL_ONE = 1.5e-7, 1e-6


def _errors(plan, w, betas):
    t, P = plan.tsort.view(-1, 3).double(), plan.P
    low = torch.ceil(plan.tsort.view(-1, 3) - plan.width / 2).double()
    d = (low[..., None] + torch.arange(P, device=t.device) - t[..., None]).abs()
    b = torch.tensor(betas, dtype=torch.float64, device=t.device)[None, :, None]
    z = b * (1 - (d / (plan.width / 2)) ** 2).clamp(min=0).sqrt()
    exact = torch.where(d <= plan.width / 2, torch.special.i0(z), torch.zeros_like(z))
    e = w.view(-1, 3, P).double() - exact
    return float(e.norm() / exact.norm()), float((e.abs() / exact.clamp(min=1)).max())


def _beta(width, oversamp):
    return math.pi * math.sqrt((width / oversamp * (oversamp - 0.5)) ** 2 - 0.8)


@pytest.mark.parametrize("width", [4.0, 6.0])
@pytest.mark.parametrize("oversamp", [1.25, 2.0])
def test_plan_weights(dev, width, oversamp):
    from mr_recon_amd import _lib
    from mr_recon_amd.plan import SamplePlan

    beta = _beta(width, oversamp)
    k = (torch.rand((200_000, 3), generator=torch.Generator().manual_seed(1)) * 100 + 10).to(dev)
    for betas in ((beta,) * 3, (beta, 0.8 * beta, 1.1 * beta)):
        plan = SamplePlan(k, (128,) * 3, width, betas)
        l2, one = _errors(plan, plan.wsort, betas)
        assert l2 < TOL and one < TOL_ONE
        # shapes in 32 bits: the same kernel, exact for the rounded shape
        b32 = [float(torch.tensor(b, dtype=torch.float32)) for b in betas]
        w, base = torch.empty_like(plan.wsort), torch.empty_like(plan.lbase)
        st = torch.cuda.current_stream(dev).cuda_stream
        args = (3, plan.P, plan.tsort.data_ptr(), plan.npts, _lib.ints((128,) * 3), _lib.ints((0,) * 3), width)
        _lib.check(_lib.lib().mra_plan_weights_dims(*args, _lib.floats(b32), w.data_ptr(), base.data_ptr(), st))
        l2, one = _errors(plan, w, b32)
        assert l2 < TOL and one < TOL_ONE and torch.equal(base, plan.lbase)
        if len(set(betas)) == 1:
            w2 = torch.empty_like(w)
            _lib.check(_lib.lib().mra_plan_weights(*args, b32[0], w2.data_ptr(), base.data_ptr(), st))
            assert torch.equal(w2, w)
