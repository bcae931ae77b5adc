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


@pytest.mark.parametrize("n,batch,scheme", [(6144, 2, "SETDRK3"), (8192, 3, "SETDRK4"), (10000, 1, "SETDRK2"), (12544, 2, "ETDRK1"),
                                            (65536, 5, "SETDRK4"), (307200, 1, "SETDRK2"), (1048576, 1, "SETDRK4")])
def test_long_1d_meshes(dev, n, batch, scheme):
    """N = L1 L2 beyond 4096 points: Burgers with Convection and with ConservativeConvection, per-sample
    coefficients and a source, against the unfused path and the oracle; a single evaluation too.  (SETDRK
    schemes and ETDRK1: ETDRK2's float32 c2 is off by 1e6 at the lowest modes of such long boxes, where the
    oracle's own float32 and float64 runs differ by 5e-3.)"""
    from oracle import refpath
    from torchfsm_amd.engine import SpectralPlan

    length = n / 512.0
    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.arange(n, device=dev, dtype=torch.float64) / n
    u = sum(torch.randn(batch, 1, 1, generator=g, device=dev, dtype=torch.float64)
            * torch.cos(2 * math.pi * (int(n / 512 * f) * x + f)) for f in (0.3, 1.0, 2.2)).float().contiguous()
    u = u + 0.1 * torch.randn(batch, 1, n, generator=g, device=dev)  # content at every frequency, N/2 too
    src = torch.randn(1, 1, n, generator=g, device=dev)
    for kind in ("conv", "cons"):
        nus = [0.01 + 0.01 * b for b in range(batch)]
        plan = SpectralPlan([(0, length, n)], batch, 1, nonlinear=kind, nonlinear_coef=-1.0,
                            linear=[("lap", nus if batch > 1 else nus[0])], device=dev)
        assert not plan.general
        plan.add_source(src, 0.2)
        plan.set_scheme(scheme, 2e-4)
        uh = plan.forward(u)
        ev = plan.apply(uh)
        plan.step(uh, 4)
        fused = plan.inverse(uh)
        plan.set_general(True)
        uh = plan.forward(u)
        ev_g = plan.apply(uh)
        plan.step(uh, 4)
        h = n // 2 + 1
        assert _rel(torch.view_as_real(ev[..., :h]), torch.view_as_real(ev_g[..., :h])) <= TOL
        assert _rel(fused, plan.inverse(uh)) <= TOL
        for b in range(0, batch, 2):
            terms = [(nus[b], "lap", None), (-1, kind, None), (0.2, "src", src)]
            ref = refpath.integrate(terms, [(0, length, n)], u[b:b + 1], 2e-4, 4, scheme=scheme)
            assert _rel(fused[b:b + 1], ref) <= TOL


def test_long_1d_recorder_and_gradient(dev):
    """A recorded long 1D trajectory ends in the unrecorded result; the adjoint's evaluations agree with
    the unfused path's."""
    import torchfsm_amd as tfa
    from torchfsm_amd import pde
    from torchfsm_amd.integrator import SETDRKIntegrator
    from torchfsm_amd.traj_recorder import AutoRecorder

    n = 8192
    g = torch.Generator(device=dev).manual_seed(1)
    u = torch.randn(2, 1, n, generator=g, device=dev)
    mesh = tfa.MeshGrid([(0, 16.0, n)], device=dev)
    op = pde.Burgers(0.02)
    op.set_integrator(SETDRKIntegrator.SETDRK2)
    op.register_mesh(mesh, 1)
    end = op.integrate(u, dt=2e-4, step=5)
    traj = op.integrate(u, dt=2e-4, step=5, trajectory_recorder=AutoRecorder())
    assert traj.shape == (2, 6, 1, n) and torch.equal(traj[:, -1], end)
    grads = []
    for general in (False, True):
        x = u.clone().requires_grad_(True)
        op._prepare(2, dev, 2e-4).set_general(general)
        op.integrate(x, dt=2e-4, step=5).square().sum().backward()
        grads.append(x.grad)
    assert _rel(grads[0], grads[1]) <= TOL


@pytest.mark.parametrize("n,batch", [(32, 1), (64, 5), (96, 9), (100, 13), (112, 3), (128, 3), (256, 2), (512, 2), (768, 1), (800, 2),
                                     (1024, 2), (2048, 3), (4096, 1)])
def test_1d_stepper_lengths_and_batches(dev, n, batch):
    """The persistent 1D stepper at every kind of radix plan and at batches that leave part of a workgroup
    idle: Convection (SETDRK3) and ConservativeConvection (SETDRK4) with per-sample coefficients and a
    source, per-sample step counts, and a complex L, against the oracle."""
    from oracle import refpath
    from torchfsm_amd.engine import SpectralPlan

    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.arange(n, device=dev) / n
    amp = torch.rand(batch, 1, 1, generator=g, device=dev)
    u = (amp * torch.sin(2 * math.pi * x) + 0.3 + 0.02 * torch.randn(batch, 1, n, generator=g, device=dev)).contiguous()
    src = torch.randn(1, 1, n, generator=g, device=dev)
    dt, mi = 0.1 / n, [(0, 1.0, n)]
    nus = [0.02 + 0.01 * b for b in range(batch)]
    for kind, scheme in (("conv", "SETDRK3"), ("cons", "SETDRK4")):
        plan = SpectralPlan(mi, batch, 1, nonlinear=kind, nonlinear_coef=-1.0,
                            linear=[("lap", nus if batch > 1 else nus[0])], device=dev)
        plan.add_source(src, 0.2)
        plan.set_scheme(scheme, dt)
        uh = plan.forward(u)
        plan.step(uh, 6)
        out = plan.inverse(uh)
        counts = torch.arange(batch, device=dev, dtype=torch.int32)
        uv = plan.forward(u)
        plan.step_varying(uv, counts, 6)
        part = plan.inverse(uv)
        for b in range(0, batch, 2):
            terms = [(nus[b], "lap", None), (-1, kind, None), (0.2, "src", src)]
            assert _rel(out[b:b + 1], refpath.integrate(terms, mi, u[b:b + 1], dt, 6, scheme=scheme)) <= TOL
            if 0 < b <= 6:
                assert _rel(part[b:b + 1], refpath.integrate(terms, mi, u[b:b + 1], dt, b, scheme=scheme)) <= TOL
        assert _rel(part[:1], u[:1]) <= TOL
    plan = SpectralPlan(mi, batch, 1, nonlinear="conv", nonlinear_coef=-1.0, linear=[(("deriv", 0, 3), -1e-4), ("lap", 0.02)],
                        device=dev)
    plan.set_scheme("SETDRK4", dt)
    uh = plan.forward(u)
    plan.step(uh, 5)
    terms = [(-1e-4, "deriv", (0, 3)), (0.02, "lap", None), (-1, "conv", None)]
    assert _rel(plan.inverse(uh), refpath.integrate(terms, mi, u, dt, 5, scheme="SETDRK4")) <= TOL


@pytest.mark.parametrize("kind", ["vc", "conv", "nsp", "ks", "ks_keep_mean"])
@pytest.mark.parametrize("n0,n1,batch", [(30, 42, 3), (225, 301, 2), (67, 64, 5), (64, 67, 2), (17, 512, 2), (16, 18, 1), (128, 6, 2),
                                         (9, 8, 4), (384, 50, 1), (143, 169, 1), (1024, 131, 1), (600, 601, 1), (5, 1031, 1)])
def test_2d_run_time_lengths(dev, kind, n0, n1, batch):
    """2D meshes where an axis has no fixed-size kernel (composite, prime and mixed with fixed-size axes):
    every SETDRK4 stage with a source, per-sample step counts and a single evaluation, against the oracle."""
    from oracle import refpath
    from torchfsm_amd.engine import SpectralPlan
    from torchfsm_amd.workloads import fourier_modes_field

    c = 2 if kind in ("conv", "nsp") else 1
    ks = kind.startswith("ks")
    length = 20.0 if ks else 1.0
    mi = [(0, length, n0), (0, length, n1)]
    u = 0.5 * fourier_modes_field((n0, n1), 2, c, batch, seed=n0 + n1, kabs=2).to(dev)
    g = torch.Generator(device=dev).manual_seed(n0)
    u = u + 0.02 * torch.randn(u.shape, generator=g, device=dev)
    src = torch.randn(1, 1, n0, n1, generator=g, device=dev)
    dt = 0.01 if ks else 0.2 / max(n0, n1)
    lin = [("lap", -1.0), ("biharm", -1.0)] if ks else [("lap", 0.01)]
    coef = 1.0 if kind == "nsp" else -1.0
    plan = SpectralPlan(mi, batch, c, nonlinear=kind, nonlinear_coef=coef, linear=lin, device=dev)
    assert plan.general
    plan.add_source(src, 0.3)
    terms = [(v, k, None) for k, v in lin] + [(coef, kind, None), (0.3, "src", src)]
    for scheme in ("SETDRK4", "SETDRK3"):
        plan.set_scheme(scheme, dt)
        uh = plan.forward(u)
        plan.step(uh, 4)
        ref = refpath.integrate(terms, mi, u, dt, 4, scheme=scheme)
        assert _rel(plan.inverse(uh), ref) <= TOL
    if not plan._plan or kind == "ks":
        return
    counts = torch.tensor([b % 3 for b in range(batch)], dtype=torch.int32, device=dev)
    plan.set_scheme("SETDRK2", dt)
    uh = plan.forward(u)
    plan.step_varying(uh, counts, 2)
    out = plan.inverse(uh)
    for b in range(batch):
        k = int(counts[b])
        ref = u[b:b + 1] if k == 0 else refpath.integrate(terms, mi, u[b:b + 1], dt, k, scheme="SETDRK2")
        assert _rel(out[b:b + 1], ref) <= TOL


@pytest.mark.parametrize("n,batch", [(2, 1), (3, 2), (7, 3), (30, 2), (97, 1), (143, 5), (360, 2), (767, 1), (1000, 3), (1021, 2), (2039, 1),
                                     (2187, 1), (4000, 2)])
def test_1d_run_time_lengths(dev, n, batch):
    """The persistent 1D stepper at run-time lengths: Convection and ConservativeConvection with a source,
    per-sample coefficients, a recorded trajectory and a single evaluation, against the oracle."""
    from oracle import refpath
    from torchfsm_amd.engine import SpectralPlan

    g = torch.Generator(device=dev).manual_seed(n)
    x = torch.arange(n, device=dev) / n
    amp = torch.rand(batch, 1, 1, generator=g, device=dev)
    u = (amp * torch.sin(2 * math.pi * x) + 0.3 + 0.02 * torch.randn(batch, 1, n, generator=g, device=dev)).contiguous()
    src = torch.randn(1, 1, n, generator=g, device=dev)
    dt, mi = 0.1 / n, [(0, 1.0, n)]
    nus = [0.02 + 0.01 * b for b in range(batch)]
    for kind, scheme in (("conv", "SETDRK4"), ("cons", "SETDRK3")):
        plan = SpectralPlan(mi, batch, 1, nonlinear=kind, nonlinear_coef=-1.0,
                            linear=[("lap", nus if batch > 1 else nus[0])], device=dev)
        assert plan.general
        plan.add_source(src, 0.2)
        plan.set_scheme(scheme, dt)
        uh = plan.forward(u)
        rec = torch.tensor([0, -1, 1, -1, 2], dtype=torch.int32, device=dev)
        traj = torch.zeros((batch, 3) + tuple(plan.spec_shape[1:]), dtype=torch.complex64, device=dev)
        plan.step(uh, 4, rec, traj)
        for b in range(batch):
            terms = [(nus[b], "lap", None), (-1, kind, None), (0.2, "src", src)]
            for t, k in ((1, 2), (2, 4)):
                ref = refpath.integrate(terms, mi, u[b:b + 1], dt, k, scheme=scheme)
                assert _rel(plan.inverse(traj[b:b + 1, t].contiguous()), ref) <= TOL
            assert _rel(plan.inverse(uh[b:b + 1].contiguous()), ref) <= TOL


@pytest.mark.parametrize("shape,batch,c", [((32,), 3, 1), ((100,), 1, 2), ((4096,), 2, 1), ((97,), 2, 1), ((16, 16), 2, 1), ((512, 48), 3, 2),
                                           ((30, 42), 1, 1), ((64, 50), 2, 1), ((1024, 32), 1, 1), ((16, 32, 64), 2, 1), ((20, 16, 16), 1, 2)])
def test_linear_integrate_from_field_to_field(dev, shape, batch, c):
    """ETDRK0 from field to field (per-sample diffusion; a complex L with one channel) against the separate
    transforms and steps of the same plan and against the oracle."""
    from oracle import refpath
    from torchfsm_amd.engine import SpectralPlan

    g = torch.Generator(device=dev).manual_seed(sum(shape))
    u = torch.randn(batch, c, *shape, generator=g, device=dev)
    mi = [(0, 1.0, n) for n in shape]
    nus = [1e-3 * (b + 1) for b in range(batch)]
    lins = [[("lap", nus if batch > 1 else nus[0])]]
    if c == 1:
        # along the last axis: on another axis' Nyquist plane the half spectrum holds the Hermitian part
        lins.append([(("deriv", len(shape) - 1, 1), -0.3), ("lap", 1e-3)])
    for lin in lins:
        plan = SpectralPlan(mi, batch, c, linear=lin, device=dev)
        plan.set_scheme("ETDRK0", 0.1)
        for steps in (0, 1, 3):
            out = plan.integrate_linear(u, steps)
            uh = plan.forward(u)
            plan.step(uh, steps)
            assert _rel(out, plan.inverse(uh)) <= 1e-6  # the same products, transforms of the same lengths
            if steps == 0:
                continue
            for b in range(batch):
                t = [(nus[b], "lap", None)] if len(lin) == 1 else [(-0.3, "deriv", (len(shape) - 1, 1)),
                                                                              (1e-3, "lap", None)]
                ref = refpath.integrate(t, mi, u[b:b + 1], 0.1, steps, scheme="ETDRK0")
                assert _rel(out[b:b + 1], ref) <= TOL


@pytest.mark.parametrize("shape", [(16,), (17,), (100,), (64, 48), (30, 34), (16, 16, 16), (6, 5, 4), (8, 8, 2)])
def test_forward_leaves_zero_padding(dev, shape):
    """The padded columns of a spectrum that forward() allocates are zero."""
    from torchfsm_amd.engine import SpectralPlan

    plan = SpectralPlan([(0, 1.0, n) for n in shape], 2, 1, device=dev)
    junk = torch.full((2, 1) + shape[:-1] + (plan.pitch,), float("nan"), dtype=torch.complex64, device=dev)
    del junk  # the allocator hands the same block out again
    uh = plan.forward(torch.ones(2, 1, *shape, device=dev))
    assert bool((uh[..., shape[-1] // 2 + 1:] == 0).all()) and bool(torch.isfinite(torch.view_as_real(uh)).all())


@pytest.mark.parametrize("kind", ["burgers", "nsp"])
@pytest.mark.parametrize("shape,batch", [((32, 32, 32), 3), ((64, 64, 64), 2), ((64, 32, 16), 1), ((16, 64, 32), 2)])
@pytest.mark.parametrize("scheme", ["SETDRK2", "SETDRK4"])
def test_3d_small_mesh_defaults(dev, kind, shape, batch, scheme):
    """The default plans of small 3D meshes, with content at every frequency and a source, against the
    unfused path and the oracle."""
    from oracle import refpath
    from torchfsm_amd.engine import SpectralPlan

    g = torch.Generator(device=dev).manual_seed(sum(shape))
    u = 0.3 * torch.randn(batch, 3, *shape, generator=g, device=dev)
    src = torch.randn(1, 3, *shape, generator=g, device=dev)
    mi = [(0, 1.0, n) for n in shape]
    name, coef = {"burgers": ("conv", -1.0), "nsp": ("nsp", 1.0)}[kind]
    plan = SpectralPlan(mi, batch, 3, nonlinear=name, nonlinear_coef=coef, linear=[("lap", 0.01)], device=dev)
    plan.add_source(src, 0.2)
    plan.set_scheme(scheme, 1e-3)
    uh = plan.forward(u)
    plan.step(uh, 3)
    out = plan.inverse(uh)
    plan.set_general(True)
    uh = plan.forward(u)
    plan.step(uh, 3)
    terms = [(0.01, "lap", None), (coef, name, None), (0.2, "src", src)]
    ref = refpath.integrate(terms, mi, u, 1e-3, 3, scheme=scheme)
    assert _rel(out, plan.inverse(uh)) <= TOL and _rel(out, ref) <= TOL


@pytest.mark.parametrize("term,shape,B,sb,ns", [("vc", (128, 128), 129, 65, 2), ("conv", (200, 200), 53, 27, 2),
                                                ("nsp", (256, 256), 33, 17, 2), ("nsp", (512, 512), 9, 5, 2),
                                                ("conv", (48, 48, 48), 9, 5, 2), ("nsp", (96, 96, 96), 3, 1, 2)])
def test_default_sub_batches_equal_whole_batch(dev, term, shape, B, sb, ns):
    """The default sub-batches on two streams, with a shorter last one, against one launch over the whole
    batch: the same kernels, so equal bit for bit; the last sample against a plan of one sample (other
    launch shapes at most) within the float32 bar."""
    from torchfsm_amd.engine import SpectralPlan

    D = len(shape)
    C = 1 if term == "vc" else D
    g = torch.Generator(device=dev).manual_seed(B)
    u = 0.3 * torch.randn(B, C, *shape, generator=g, device=dev)

    def plan_of(batch):
        p = SpectralPlan([(0, 1.0, n) for n in shape], batch, C, nonlinear=term, nonlinear_coef=-1.0,
                         linear=[("lap", 0.01)], device=dev)
        p.set_scheme("SETDRK4", 1e-3)
        return p

    plan = plan_of(B)
    assert plan.tuning[4] == sb and plan.streams == ns and not plan.general
    uh = plan.forward(u)
    plan.step(uh, 3)
    plan.set_tuning(*plan.tuning[:4], 0)
    plan.set_streams(1)
    uw = plan.forward(u)
    plan.step(uw, 3)
    assert torch.equal(uh, uw)
    one = plan_of(1)
    u1 = one.forward(u[B - 1:].contiguous())
    one.step(u1, 3)
    assert _rel(plan.inverse(uh)[B - 1:], one.inverse(u1)) <= TOL


@pytest.mark.parametrize("n", [32, 64])
@pytest.mark.parametrize("term,C", [("vc", 1), ("conv", 2)])
@pytest.mark.parametrize("rate", [0.5, 2 / 3, 0.9])
def test_persistent_2d_stepper_bands(dev, n, term, C, rate):
    """The persistent 2D stepper with the 2/3 rule's band, a narrower and a wider one, against the tiled kernels
    (the same arithmetic up to fused multiply-adds)."""
    from torchfsm_amd.engine import SpectralPlan

    plan = SpectralPlan([(0, 1.0, n)] * 2, 3, C, nonlinear=term, nonlinear_coef=-1.0, linear=[("lap", 0.01)],
                        dealias_rate=rate, device=dev)
    plan.set_scheme("SETDRK4", 1e-3)
    g = torch.Generator(device=dev).manual_seed(n)
    u = 0.3 * torch.randn(3, C, n, n, generator=g, device=dev)
    assert plan.persistent
    res = []
    for on in (True, False):
        plan.set_persistent(on)
        uh = plan.forward(u)
        plan.step(uh, 4)
        res.append(plan.inverse(uh))
    assert _rel(res[0], res[1]) <= 1e-6
