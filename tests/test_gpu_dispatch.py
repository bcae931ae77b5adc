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


RUNTIME = [("vc", (30, 42), 3), ("conv", (64, 67), 2), ("nsp", (67, 64), 2), ("ks", (48, 60), 2), ("ks_keep_mean", (17, 30), 1),
           ("conv", (1000,), 2), ("cons", (97,), 3)]


@pytest.mark.parametrize("kind,shape,batch", RUNTIME)
def test_run_time_lengths_against_the_unfused_path(dev, kind, shape, batch):
    """set_general(True) takes a plan off the run-time-length kernels and set_general(False) puts it back: steps and
    a single evaluation agree, and the first ones come back bit for bit."""
    plan = _plan(kind, shape, batch, dev)
    assert plan.path == "runtime" and plan.general
    plan.set_scheme("SETDRK4", 1e-3)
    u = _smooth(plan, dev, sum(shape))
    h = shape[-1] // 2 + 1
    res = []
    for on in (False, True, False):
        plan.set_general(on)
        assert plan.path == ("unfused" if on else "runtime") and plan.general
        uh = plan.forward(u)
        ev = torch.view_as_real(plan.apply(uh)[..., :h])
        plan.step(uh, 4)
        res.append((plan.inverse(uh), ev))
    assert _rel(res[0][0], res[1][0]) <= TOL and _rel(res[0][1], res[1][1]) <= TOL
    assert torch.equal(res[0][0], res[2][0]) and torch.equal(res[0][1], res[2][1])


@pytest.mark.parametrize("kind,shape,path", [("conv", (256,), "fixed"), ("conv", (8192,), "long1d"), ("vc", (64, 64), "fixed"),
                                             ("nsp", (32, 32, 32), "fixed"), ("conv", (40, 40, 40), "unfused"),
                                             ("ks", (1000,), "unfused"), (None, (30, 30), "linear")])
def test_plan_path(dev, kind, shape, path):
    """The kernels a plan starts on; a plan with fused ones goes to the unfused path and back."""
    plan = _plan(kind, shape, 2, dev)
    assert plan.path == path and plan.general == (path == "unfused")
    if path == "unfused":
        with pytest.raises(ValueError):
            plan.set_general(False)
    elif path != "linear":
        plan.set_general(True)
        assert plan.path == "unfused" and plan.general
        plan.set_general(False)
        assert plan.path == path and not plan.general


def test_force_takes_a_run_time_length_plan_to_the_unfused_path(dev):
    plan = _plan("nsp", (30, 34), 2, dev)
    assert plan.path == "runtime"
    plan.add_force(torch.ones(1, 2, 30, 34, device=dev), 0.1)
    assert plan.path == "unfused"
    with pytest.raises(ValueError):
        plan.set_general(False)


@pytest.mark.parametrize("kind,scheme", [("conv", "SETDRK4"), ("cons", "SETDRK3")])
@pytest.mark.parametrize("n,path", [(2049, "unfused"), (2045, "runtime"), (3745, "unfused"), (3750, "runtime"), (3888, "runtime"),
                                    (4000, "runtime"), (4095, "runtime"), (4097, "unfused")])
def test_1d_stepper_up_to_4096_points(dev, kind, scheme, n, path):
    """The persistent 1D stepper takes every mesh whose FFT length (the mesh's own, or Bluestein's) is at most 4096,
    with its state in global memory where LDS does not hold it: against the unfused path."""
    plan = _plan(kind, (n,), 2, dev)
    assert plan.path == path
    plan.set_scheme(scheme, 0.1 / n)
    u = _smooth(plan, dev, n)
    res = []
    for on in (False, True):
        if path == "runtime":
            plan.set_general(on)
        uh = plan.forward(u)
        ev = plan.apply(uh)[..., : n // 2 + 1]
        plan.step(uh, 4)
        res.append((plan.inverse(uh), torch.view_as_real(ev)))
    assert _rel(res[0][0], res[1][0]) <= TOL and _rel(res[0][1], res[1][1]) <= TOL


@pytest.mark.parametrize("n", [97, 1000, 4000])
def test_integrate_on_the_1d_stepper_takes_no_graph(dev, n):
    """The run-time-length 1D stepper runs every step of integrate() in one launch: no graph of 16 steps is captured
    around it, and the steps are those of one plan.step call."""
    import torchfsm_amd as tfa
    from torchfsm_amd import pde

    op = pde.Burgers(0.01)
    op.register_mesh(tfa.MeshGrid([(0, 1, n)], device=dev), 1)
    plan = op._prepare(2, dev, 0.1 / n)
    assert plan.path == "runtime"
    u = _smooth(plan, dev, n)
    out = op.integrate(u, dt=0.1 / n, step=40)
    assert getattr(plan, "_step_graph", None) is None
    uh = plan.forward(u)
    plan.step(uh, 40)
    assert torch.equal(out, plan.inverse(uh))


@pytest.mark.parametrize("kind,shape,batch,sub,streams", [
    # narrow meshes: a sub-batch holds about 2M points (one channel of 512 and 1024 points 4M), never a few samples
    ("conv", (1024, 16), 64, 0, 1), ("conv", (1024, 48), 64, 32, 2), ("nsp", (1024, 48), 32, 0, 1), ("nsp", (1024, 256), 64, 8, 2),
    ("conv", (512, 48), 64, 0, 1), ("nsp", (512, 64), 128, 64, 2), ("vc", (512, 48), 64, 0, 1), ("vc", (512, 64), 256, 128, 2),
    ("ks_keep_mean", (512, 128), 64, 0, 1), ("vc", (1024, 256), 64, 16, 2),
    # ConservativeConvection has two channels
    ("cons", (512, 48), 64, 0, 1), ("cons", (512, 512), 32, 8, 2), ("cons", (1024, 64), 32, 0, 1), ("cons", (1024, 1024), 8, 2, 2),
    # square ones
    ("conv", (512, 512), 32, 16, 2), ("nsp", (512, 1024), 32, 16, 2), ("vc", (512, 512), 64, 16, 2), ("vc", (512, 512), 16, 0, 1),
    ("conv", (1024, 1024), 8, 4, 2), ("nsp", (1024, 1024), 4, 0, 1), ("vc", (1024, 1024), 8, 0, 1),
    # KSConvection and long columns of ConservativeConvection from 4M points
    ("ks_keep_mean", (256, 256), 32, 0, 1), ("ks_keep_mean", (256, 1024), 16, 8, 2), ("cons", (256, 1024), 8, 0, 1),
    ("cons", (256, 256), 32, 16, 2), ("cons", (128, 1024), 16, 8, 2),
    # nothing to overlap: the batch mean couples the samples, or there is no product term
    ("ks", (512, 512), 64, 0, 1), (None, (256, 256), 64, 0, 1)])
def test_2d_sub_batches(dev, kind, shape, batch, sub, streams):
    """The sub-batches and streams a 2D plan starts with."""
    plan = _plan(kind, shape, batch, dev)
    assert (plan.tuning[4], plan.streams) == (sub, streams)


@pytest.mark.parametrize("kind,shape,batch", [("conv", (1024, 48), 65), ("cons", (512, 64), 257), ("vc", (512, 64), 257)])
def test_narrow_sub_batches_equal_the_whole_batch(dev, kind, shape, batch):
    """The sub-batches of narrow meshes, a shorter last one among them, against one launch over the whole batch: the
    same kernels, so equal bit for bit."""
    plan = _plan(kind, shape, batch, dev)
    assert 0 < plan.tuning[4] < batch and batch % plan.tuning[4] and plan.streams == 2
    plan.set_scheme("SETDRK4", 1e-4)
    u = _smooth(plan, dev, batch)
    res = []
    for whole in (False, True):
        if whole:
            plan.set_tuning(*plan.tuning[:4], 0)
            plan.set_streams(1)
        uh = plan.forward(u)
        plan.step(uh, 3)
        res.append(plan.inverse(uh))
    assert torch.equal(res[0], res[1])


@pytest.mark.parametrize("kind", ["ks", "ks_keep_mean", "cons", "vc", "conv", "nsp"])
@pytest.mark.parametrize("shape,batch", [((64, 16), 3), ((128, 48), 2), ((256, 64), 2), ((256, 256), 1)])
def test_stage_kernels_of_four_values_per_thread(dev, kind, shape, batch):
    """The column kernels compiled per stage, of 4 values per thread, with a source: every evaluation of every
    scheme, the field pass and a single evaluation, against the unfused path."""
    plan = _plan(kind, shape, batch, dev)
    assert plan.path == "fixed" and plan.tuning[1] == 1
    u = _smooth(plan, dev, sum(shape))
    plan.add_source(u[:1].roll(3, -1).contiguous(), 0.2)
    h = shape[-1] // 2 + 1
    for scheme in ("ETDRK1", "SETDRK1", "SETDRK2", "ETDRK2", "SETDRK3", "SETDRK4"):
        plan.set_scheme(scheme, 1e-3)
        res = []
        for on in (False, True):
            plan.set_general(on)
            uh = plan.forward(u)
            ev = torch.view_as_real(plan.apply(uh)[..., :h])
            plan.step(uh, 3)
            res.append((plan.inverse(uh), ev))
        assert _rel(res[0][0], res[1][0]) <= TOL and _rel(res[0][1], res[1][1]) <= TOL


def test_precision_of_transforms_of_any_length(dev):
    """Lengths with a prime factor above 13 run as circular convolutions, whose rounding errors depend on the
    convolution's length: forward transforms of white noise at 22 lengths against float64, in the rms.  Powers of two
    give 1.44e-7, the chosen lengths 1.54e-7, the shortest smooth lengths 1.61e-7."""
    import numpy as np

    ns = (53, 58, 86, 101, 185, 199, 222, 227, 230, 235, 266, 290, 316, 341, 355, 401, 543, 632, 812, 919, 970, 1017)
    total = 0.0
    for n in ns:
        plan = _plan(None, (n,), 64, dev)
        u = torch.randn(64, 1, n, generator=torch.Generator().manual_seed(n + 1))
        got = plan.forward(u.to(dev))[..., : n // 2 + 1].cpu().to(torch.complex128).numpy()
        ref = np.fft.rfft(u.double().numpy())
        total += float(np.linalg.norm(got - ref) ** 2 / np.linalg.norm(ref) ** 2)
    assert (total / len(ns)) ** 0.5 <= 1.575e-7


@pytest.mark.parametrize("shape,batch", [((23,), 1), ((500,), 64), ((1015,), 300), ((2039,), 1), ((2039,), 300), ((4095,), 1), ((4095,), 300),
                                         ((1017, 9), 2), ((9, 1017), 2), ((17, 1031), 40), ((2050, 34), 1), ((6, 1015, 5), 3)])
def test_general_transforms_by_launch_shape(dev, shape, batch):
    """General-length transforms there and back with few workgroups (more threads, tables in LDS) and many (two
    workgroups per CU), short and long lines, rows and strided columns, against numpy in float64."""
    import numpy as np

    plan = _plan(None, shape, batch, dev)
    u = torch.randn(batch, 1, *shape, generator=torch.Generator().manual_seed(sum(shape) + batch))
    uh = plan.forward(u.to(dev))
    got = uh[..., : shape[-1] // 2 + 1].cpu().to(torch.complex128).numpy()
    ref = np.fft.rfftn(u.double().numpy(), axes=tuple(range(2, 2 + len(shape))))
    assert float(np.linalg.norm(got - ref) / np.linalg.norm(ref)) <= 1e-6
    assert _rel(plan.inverse(uh).cpu(), u) <= 1e-6


@pytest.mark.parametrize("kind,shape,batch,path", [("conv", (509, 64), 1, "runtime"), ("nsp", (993, 40), 1, "runtime"), ("vc", (1000, 48), 2, "runtime"),
                                                   ("ks", (787, 20), 1, "runtime"), ("vc", (2039, 32), 1, "runtime"), ("conv", (2039, 32), 1, "unfused"),
                                                   ("nsp", (2039, 32), 3, "unfused"), ("conv", (2039, 32), 4, "runtime"), ("vc", (112, 37), 2, "runtime"),
                                                   ("nsp", (200, 30), 1, "runtime"), ("conv", (100, 301), 1, "runtime"), ("ks", (100, 37), 60, "runtime"), ("conv", (127, 126), 4, "runtime")])
def test_2d_run_time_lengths_with_few_columns(dev, kind, shape, batch, path):
    """Meshes with fewer than 64 workgroups' worth of columns, one column and several fields per workgroup, and the long
    ones that step unfused: against the unfused path."""
    plan = _plan(kind, shape, batch, dev)
    assert plan.path == path
    plan.set_scheme("SETDRK4", 0.02 / max(shape))
    u = _smooth(plan, dev, sum(shape))
    res = []
    for on in (False, True):
        if path == "runtime":
            plan.set_general(on)
        uh = plan.forward(u)
        plan.step(uh, 3)
        res.append(plan.inverse(uh))
    assert _rel(res[0], res[1]) <= TOL and bool(torch.isfinite(res[0]).all())


@pytest.mark.parametrize("shape", [(16,), (17,), (100,), (4096,), (64, 48), (30, 34), (1024, 32), (16, 16, 16), (6, 5, 4), (8, 8, 2)])
def test_forward_writes_its_padding_into_a_given_spectrum(dev, shape):
    """tfsm_plan_forward_fills: where it says so, forward() overwrites every element of a spectrum full of NaN, the
    padded columns with zeros; elsewhere it leaves the padded columns alone."""
    plan = _plan(None, shape, 2, dev)
    u = torch.randn(2, 1, *shape, generator=torch.Generator().manual_seed(1)).to(dev)
    out = torch.full((2, 1) + shape[:-1] + (plan.pitch,), complex(float("nan"), float("nan")), dtype=torch.complex64, device=dev)
    plan.forward(u, out)
    h = shape[-1] // 2 + 1
    assert bool(torch.isfinite(torch.view_as_real(out[..., :h])).all())
    pad = torch.view_as_real(out[..., h:])
    assert bool((pad == 0).all()) if plan._forward_fills else bool(pad.isnan().all())
