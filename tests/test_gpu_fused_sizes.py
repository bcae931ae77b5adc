"""Sizes and shapes of the fused kernels beyond the workloads' own, against the unfused path of the
same plan and the oracle (rel-L2 1e-5, the parity bar: float32 rounding of a few evaluations is below
1e-6)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _rel(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm())


@pytest.mark.parametrize("kind", ["burgers", "nsp", "kshd"])
@pytest.mark.parametrize("shape,batch", [((256, 16, 32), 2), ((32, 256, 64), 1), ((16, 32, 256), 3)])
def test_3d_axes_of_256_points(dev, kind, shape, batch):
    """A 256-point x, y or z axis of a 3D mesh steps on the fused kernels."""
    import torchfsm_amd as tfa
    from oracle import refpath
    from torchfsm_amd import pde
    from torchfsm_amd.workloads import fourier_modes_field

    c = 1 if kind == "kshd" else 3
    length = 20 * math.pi if kind == "kshd" else 1.0
    dt = 0.02 if kind == "kshd" else 5e-4
    mi = [(0, length, n) for n in shape]
    op, terms = {"burgers": (pde.Burgers(0.01), refpath.burgers_terms(0.01)),
                 "nsp": (pde.NavierStokes(100.0), refpath.ns_velocity_terms(100.0)),
                 "kshd": (pde.KuramotoSivashinskyHighDim(), refpath.ks_highdim_terms())}[kind]
    u = 0.5 * fourier_modes_field(shape, 3, c, batch, seed=7).to(dev)
    op.register_mesh(tfa.MeshGrid(mi, device=dev), c)
    plan = op._prepare(batch, dev, dt)
    assert not plan.general
    uh = plan.forward(u)
    plan.step(uh, 3)
    fused = plan.inverse(uh)
    plan.set_general(True)
    uh = plan.forward(u)
    plan.step(uh, 3)
    unfused = plan.inverse(uh)
    ref = refpath.integrate(terms, mi, u, dt, 3, scheme="SETDRK4")
    assert _rel(fused, ref) <= TOL and _rel(fused, unfused) <= TOL


def test_3d_256_sub_batches(dev):
    """256^3 with two samples steps one sample per stream, as each sample alone (bit for bit)."""
    import torchfsm_amd as tfa
    from torchfsm_amd import pde

    n = 256
    op = pde.Burgers(0.01)
    mesh = tfa.MeshGrid([(0, 1, n)] * 3, device=dev)
    g = torch.Generator(device=dev).manual_seed(3)
    u = 0.1 * torch.randn(2, 3, n, n, n, generator=g, device=dev)
    op.register_mesh(mesh, 3)
    plan = op._prepare(2, dev, 1e-4)
    assert plan.streams == 2 and plan.tuning[4] == 1
    both = op.integrate(u, dt=1e-4, step=2)
    for b in range(2):
        assert torch.equal(op.integrate(u[b:b + 1].contiguous(), dt=1e-4, step=2), both[b:b + 1])
