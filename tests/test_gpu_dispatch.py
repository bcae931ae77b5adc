"""Which kernels and launch shapes a plan takes, and the calls that depend on it (rel-L2 1e-5, the parity bar,
where outputs of different kernels are compared)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm())


def _plan(kind, shape, batch, dev, channels=None, **kw):
    from torchfsm_amd.engine import SpectralPlan

    c = channels or (len(shape) if kind in ("conv", "nsp", "cons") else 1)
    lin = [("lap", -1.0), ("biharm", -1.0)] if (kind or "").startswith("ks") else [("lap", 0.01)]
    length = 20.0 if (kind or "").startswith("ks") else 1.0
    return SpectralPlan([(0, length, n) for n in shape], batch, c, nonlinear=kind,
                        nonlinear_coef=1.0 if kind == "nsp" else -1.0, linear=lin, device=dev, **kw)


def _smooth(plan, dev, seed):
    """A field of a few modes and a little of every other."""
    g = torch.Generator(device=dev).manual_seed(seed)
    grid = torch.meshgrid(*[torch.arange(n, device=dev) / n for n in plan.n], indexing="ij")
    a = torch.randn(2, plan.batch, plan.channels, *([1] * plan.ndim), generator=g, device=dev)
    u = sum(a[i] * torch.sin(2 * math.pi * sum((i + 1) * x for x in grid) + i) for i in range(2))
    return (0.3 * u + 0.002 * torch.randn(u.shape, generator=g, device=dev)).contiguous()


@pytest.mark.parametrize("n", [6144, 65536])
def test_autotune_leaves_long_1d_plans_alone(dev, n):
    """The kernels of long 1D meshes have no launch shape: autotune() returns the plan's own, tries nothing, and
    the plan steps as before."""
    from torchfsm_amd.autotune import autotune

    plan = _plan("conv", (n,), 2, dev)
    plan.set_scheme("SETDRK2", 1e-5)
    u = _smooth(plan, dev, n)
    a, b = plan.forward(u), plan.forward(u)
    plan.step(a, 3)
    before = plan.tuning
    assert autotune(plan, b) == (before, {}) and plan.tuning == before
    plan.step(b, 3)
    assert torch.equal(a, b)
    with pytest.raises(ValueError, match="launch shape"):
        plan.set_tuning(*before)
