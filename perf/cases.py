"""Performance cases of the framework: what its users have it do, through its public entry points.

A case is a dict of plain values:
  eq       "burgers", "ks" (1D Kuramoto-Sivashinsky), "ns_vorticity" (2D, with Kolmogorov forcing and
           drag), "ns_velocity" (2D / 3D), "heat" (exact diffusion) or "pressure" (one evaluation)
  shape    points per axis, "128x128"
  batch    samples
  length   domain length of every axis
  nu       viscosity
  dt, steps, scheme ("auto" is the operator's own choice)
  record   the whole trajectory is returned
  grad     the gradients of a loss of the final field with respect to the initial field and the
           viscosity are returned too

exact() is the same mathematics in float64 with torch's FFTs on the full complex spectrum.
"""

import math

import torch

from torchfsm_amd import field, pde
from torchfsm_amd.integrator import ETDRKIntegrator, SETDRKIntegrator
from torchfsm_amd.mesh import MeshGrid
from torchfsm_amd.operator import Laplacian, Velocity2Pressure
from torchfsm_amd.traj_recorder import AutoRecorder

TWO_PI = 2 * math.pi
INTEGRATORS = {"ETDRK2": ETDRKIntegrator.ETDRK2, "SETDRK2": SETDRKIntegrator.SETDRK2}


def case(eq, shape, batch, length, nu, dt=1.0, steps=1, scheme="auto", record=False, grad=False):
    return {"eq": eq, "shape": "x".join(str(n) for n in shape), "batch": batch, "length": length, "nu": nu, "dt": dt,
            "steps": steps, "scheme": scheme, "record": record, "grad": grad}


def listed():
    cases = {
        # the first thing a user runs: the 1D Burgers example with its whole trajectory (pure latency)
        "burgers1d_128_trajectory": case("burgers", [128], 1, 1.0, 0.01, 0.01, 200, record=True),
        # a batch of 1D Kuramoto-Sivashinsky solves of the middle of the serving range
        "ks1d_2048_b8": case("ks", [2048], 8, 64 * math.pi, 0.0, 0.1, 50),
        # small 2D flows in batches, as for generating training data: launches and latency count
        "ns2d_64_b16": case("ns_vorticity", [64, 64], 16, TWO_PI, 1e-3, 1e-3, 50),
        # the flagship: a large batch of 512^2 Kolmogorov flows
        "ns2d_512_b64": case("ns_vorticity", [512, 512], 64, TWO_PI, 1e-3, 1e-3, 10),
        # differentiable simulation: gradients through a 2D Burgers roll-out
        "burgers2d_128_b16_gradient": case("burgers", [128, 128], 16, 1.0, 0.01, 0.002, 30, "ETDRK2", grad=True),
        # 3D vector Burgers, the bandwidth-bound 3D shape
        "burgers3d_128_b8": case("burgers", [128, 128, 128], 8, 1.0, 0.01, 1e-3, 5, "ETDRK2"),
        # velocity-form 3D Navier-Stokes of ordinary size with few samples
        "nsvel3d_64_b2": case("ns_velocity", [64, 64, 64], 2, TWO_PI, 0.01, 5e-3, 10),
        # one large 3D simulation
        "burgers3d_256": case("burgers", [256, 256, 256], 1, 1.0, 0.01, 5e-4, 2, "ETDRK2"),
        # a grid given by the user's data: ragged axes, one of them not a product of small primes
        "ns2d_225x301_b4": case("ns_vorticity", [225, 301], 4, TWO_PI, 1e-3, 1e-3, 10),
        # long 1D domains
        "burgers1d_65536_b16": case("burgers", [65536], 16, 128.0, 0.01, 5e-4, 20),
        # exact diffusion in one step, as the initial-condition generator does it: transforms only
        "heat2d_512_b16": case("heat", [512, 512], 16, TWO_PI, 0.01, 1.0, 1),
        # a diagnostic of given fields: the pressure of a velocity field (the smallest calls)
        "pressure2d_256_b8": case("pressure", [256, 256], 8, TWO_PI, 0.0),
    }
    return [dict(c, name=name) for name, c in cases.items()]


# ------------------------------------------------------------------------------ drawn cases
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _axis(rng, lo, hi):
    """A power of two (what most users take), a round mixed-radix size, or any integer."""
    kind = rng.random()
    if kind < 0.45:
        return 2 ** rng.randint(math.ceil(math.log2(lo)), int(math.log2(hi)))
    if kind < 0.7:
        sizes = [n for n in (48, 96, 100, 112, 192, 200, 384, 400, 768, 800) if lo <= n <= hi]
        if sizes:
            return rng.choice(sizes)
    return _log_int(rng, lo, hi)


def _is_pow2(n):
    return n & (n - 1) == 0


def _common(shape):
    """Powers of two and small round sizes; other grids cost several times more a point."""
    return all(_is_pow2(n) or n in (48, 96, 100, 112, 192, 200) for n in shape)


def _steps(rng, point_steps, points, lo, hi):
    return max(1, min(rng.randint(lo, hi), int(point_steps // points)))


def draw(rng):
    kind = rng.randrange(9)
    if kind == 0:  # short 1D Burgers
        n = _axis(rng, 64, 4096)
        steps = rng.randint(20, 200 if _common([n]) else 60)
        return case("burgers", [n], _log_int(rng, 1, 64), 1.0, max(0.01, 1.3 / n), 0.15 / n, steps,
                    rng.choice(["auto", "ETDRK2"]), record=rng.random() < 0.5)
    if kind == 1:  # 1D Kuramoto-Sivashinsky
        n = rng.choice([512, 1024, 2048, 4096, _log_int(rng, 500, 4100)])
        return case("ks", [n], _log_int(rng, 1, 16), rng.uniform(32, 128) * math.pi, 0.0, 0.1, rng.randint(10, 50))
    if kind == 2:  # 2D vorticity, square or not
        n0 = _axis(rng, 48, 1024)
        n1 = n0 if rng.random() < 0.6 else _axis(rng, 48, 1024)
        points = n0 * n1
        batch = _log_int(rng, 1, max(1, min(64, 2 ** 24 // points)))
        budget = 1.6e8 if _common([n0, n1]) else 8e6
        batch = max(1, min(batch, int(budget // points)))
        return case("ns_vorticity", [n0, n1], batch, TWO_PI, 1e-3, 0.1 * TWO_PI / max(n0, n1) / 4,
                    _steps(rng, budget, points * batch, 5, 50))
    if kind == 3:  # 2D velocity
        n0 = _axis(rng, 48, 512)
        n1 = n0 if rng.random() < 0.6 else _axis(rng, 48, 512)
        points = n0 * n1
        budget = 4e7 if _common([n0, n1]) else 6e6
        batch = max(1, min(_log_int(rng, 1, 32), int(budget // points)))
        return case("ns_velocity", [n0, n1], batch, TWO_PI, 5e-3, 0.1 * TWO_PI / max(n0, n1),
                    _steps(rng, budget, points * batch, 5, 30))
    if kind == 4:  # gradients
        dims = rng.choice([1, 2, 2])
        shape = [_axis(rng, 64, 1024)] if dims == 1 else [_axis(rng, 48, 256)] * 2
        points = math.prod(shape)
        batch = max(1, min(_log_int(rng, 1, 16), int(2.6e5 // points)))
        return case("burgers", shape, batch, 1.0, max(0.01, 1.3 / min(shape)), 0.15 / max(shape),
                    _steps(rng, 7.8e6, points * batch, 10, 30), rng.choice(["auto", "ETDRK2", "SETDRK2"]), grad=True)
    if kind == 5:  # 3D
        eq = rng.choice(["burgers", "ns_velocity"])
        if rng.random() < 0.6:
            shape = [2 ** rng.randint(5, 7)] * 3 if rng.random() < 0.7 else [2 ** rng.randint(5, 8) for _ in range(3)]
        else:
            shape = [_log_int(rng, 24, 160) for _ in range(3)]
        points = math.prod(shape)
        budget = 2.5e7 if _common(shape) else 5e6
        batch = max(1, min(_log_int(rng, 1, 8), int(budget // points)))
        length = 1.0 if eq == "burgers" else TWO_PI
        return case(eq, shape, batch, length, 0.01, 0.1 * length / max(shape),
                    _steps(rng, budget / (1 if eq == "burgers" else 2), points * batch, 1, 10),
                    "ETDRK2" if eq == "burgers" else "auto")
    if kind == 6:  # long 1D
        n = rng.choice([8192, 16384, 32768, 65536, _log_int(rng, 5000, 60000)])
        batch = max(1, min(_log_int(rng, 1, 16), 2 ** 20 // n))
        if not _is_pow2(n):
            batch = min(batch, 4)
        return case("burgers", [n], batch, n / 512.0, 0.01, 0.15 / 512, rng.randint(5, 20))
    if kind == 7:  # exact diffusion
        dims = rng.choice([1, 2, 2, 3])
        shape = [_axis(rng, *{1: (64, 4096), 2: (48, 1024), 3: (32, 128)}[dims]) for _ in range(dims)]
        batch = max(1, min(_log_int(rng, 1, 64), 2 ** 22 // math.prod(shape)))
        return case("heat", shape, batch, TWO_PI, 0.01, rng.uniform(0.1, 2.0), 1)
    dims = rng.choice([2, 2, 3])  # pressure of a velocity field
    shape = [_axis(rng, *{2: (48, 512), 3: (32, 128)}[dims])] * dims
    batch = max(1, min(_log_int(rng, 1, 16), 2 ** 21 // math.prod(shape)))
    return case("pressure", shape, batch, TWO_PI, 0.0)


# ------------------------------------------------------------------------------ inputs
def _shape(c):
    return [int(n) for n in c["shape"].split("x")]


def _channels(c):
    return len(_shape(c)) if c["eq"] in ("burgers", "ns_velocity", "pressure") else 1


def _noise(shape, batch, channels, kmax, gen):
    """Smooth random fields: complex normal modes with amplitude 1 / |k| for 1 <= |k| <= kmax."""
    ks = [torch.fft.fftfreq(n, 1.0 / n, device="cuda") for n in shape]
    kk = torch.sqrt(sum(k**2 for k in torch.meshgrid(*ks, indexing="ij")))
    amp = torch.where((kk >= 1) & (kk <= kmax), 1.0 / kk.clamp(min=1.0), torch.zeros_like(kk))
    z = torch.randn(batch, channels, *shape, 2, generator=gen, device="cuda")
    dims = tuple(range(2, 2 + len(shape)))
    return torch.fft.ifftn(torch.view_as_complex(z) * amp, dim=dims).real


def _unit_rms(u):
    dims = tuple(range(1, u.dim()))
    return u / torch.sqrt((u**2).mean(dim=dims, keepdim=True))


def _solenoidal(a, length):
    """Curl of a potential: one channel in 2D, three in 3D."""
    dims = a.dim() - 2
    ax = tuple(range(-dims, 0))
    ks = []
    for d in range(dims):
        n = a.shape[2 + d]
        k = torch.fft.fftfreq(n, length / n, device=a.device) * TWO_PI
        if n % 2 == 0:
            k[n // 2] = 0.0
        ks.append(k.reshape([1, 1] + [n if i == d else 1 for i in range(dims)]))
    ah = torch.fft.fftn(a, dim=ax)
    if dims == 2:
        parts = [1j * ks[1] * ah, -1j * ks[0] * ah]
    else:
        x, y, z = ah[:, 0:1], ah[:, 1:2], ah[:, 2:3]
        parts = [1j * (ks[1] * z - ks[2] * y), 1j * (ks[2] * x - ks[0] * z), 1j * (ks[0] * y - ks[1] * x)]
    return torch.fft.ifftn(torch.cat(parts, dim=1), dim=ax).real


def _inputs(c, seed):
    shape, batch = _shape(c), c["batch"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if c["eq"] == "ks":
        u = _noise(shape, batch, 1, 20, gen)
    elif c["eq"] == "ns_vorticity":
        u = _noise(shape, batch, 1, min(32, min(shape) // 6), gen)
    elif c["eq"] == "heat":
        u = torch.randn(batch, 1, *shape, generator=gen, device="cuda")
    elif c["eq"] in ("ns_velocity", "pressure"):
        kmax = 8 if len(shape) == 3 else min(16, min(shape) // 6)
        u = _solenoidal(_noise(shape, batch, 1 if len(shape) == 2 else 3, kmax, gen), c["length"])
    else:
        u = _noise(shape, batch, len(shape), 4 if max(shape) <= 4096 else max(shape) // 512, gen)
    target = _unit_rms(_noise(shape, batch, len(shape), 4, gen)).contiguous() if c["grad"] else None
    return _unit_rms(u).contiguous(), target


def prepare(c, seed):
    shape = _shape(c)
    u0, target = _inputs(c, seed)
    mesh = MeshGrid([(0, c["length"], n) for n in shape], device=u0.device)
    nu = c["nu"]
    if c["grad"]:
        nu = torch.tensor(nu, device=u0.device, requires_grad=True)
        u0.requires_grad_(True)
    if c["eq"] == "burgers":
        op = pde.Burgers(nu)
    elif c["eq"] == "ks":
        op = pde.KuramotoSivashinsky()
    elif c["eq"] == "ns_vorticity":
        op = pde.NavierStokesVorticity(1 / nu, field.kolm_force(mesh.bc_mesh_grid()[1]))
    elif c["eq"] == "ns_velocity":
        op = pde.NavierStokes(1 / nu)
    elif c["eq"] == "heat":
        op = nu * Laplacian()
    else:
        op = Velocity2Pressure()
    if c["scheme"] != "auto":
        op.set_integrator(INTEGRATORS[c["scheme"]])
    op.register_mesh(mesh, _channels(c))
    return {"case": c, "op": op, "u0": u0, "nu": nu, "target": target}


def run(state):
    c, op, u0 = state["case"], state["op"], state["u0"]
    if c["eq"] == "pressure":
        return op(u0)
    if c["record"]:
        return op.integrate(u0, dt=c["dt"], step=c["steps"], trajectory_recorder=AutoRecorder())
    u = op.integrate(u0, dt=c["dt"], step=c["steps"])
    if c["grad"]:
        loss = torch.mean((u - state["target"]) ** 2)
        # the operator's coefficient is one graph node that every roll-out shares
        g_u0, g_nu = torch.autograd.grad(loss, (u0, state["nu"]), retain_graph=True)
        return {"u": u.detach(), "grad_u0": g_u0, "grad_nu": g_nu}
    return u


# ------------------------------------------------------------------------------ work
def work(c):
    """Bytes: the initial field in, every returned field out.  Flops: the real transforms of every
    evaluation of the product term (2.5 n log2 n each) and, for an exact linear step, of the state."""
    shape = _shape(c)
    dims, chans, points = len(shape), _channels(c), math.prod(shape)
    fields = {"burgers": chans + chans * dims, "ks": 2, "ns_vorticity": 4, "ns_velocity": chans + chans * dims,
              "pressure": chans + chans * dims, "heat": 0}[c["eq"]]
    evals = c["steps"] * (4 if c["scheme"] == "auto" else 2)
    if c["eq"] in ("heat", "pressure"):
        evals = 1 if fields else 0
    outs = chans * (c["steps"] + 1 if c["record"] else 1)
    if c["eq"] == "pressure":
        outs = 1
    transforms = evals * (fields + chans) + 2 * chans
    values = chans + outs
    if c["grad"]:
        # the transposed evaluations: the fields and the adjoint's, and their products' spectra
        transforms += evals * (chans + fields + chans + chans * dims) + 2 * chans
        values += 2 * chans
    return {"bytes": 4.0 * c["batch"] * points * values,
            "flops": 2.5 * c["batch"] * points * math.log2(points) * transforms}


# ------------------------------------------------------------------------------ float64
class _Spectral:
    """Symbols, mask and transforms of one box in float64, on the full complex spectrum."""

    def __init__(self, shape, length, device):
        self.dims = tuple(range(-len(shape), 0))
        self.k, keep = [], 1.0
        for d, n in enumerate(shape):
            view = [1, 1] + [n if i == d else 1 for i in range(len(shape))]
            self.k.append((TWO_PI * torch.fft.fftfreq(n, length / n, device=device, dtype=torch.float64)).reshape(view))
            # which modes the 2/3 rule keeps is decided in float32 frequencies, as the framework documents
            f = torch.fft.fftfreq(n, length / n, device=device, dtype=torch.float32).abs()
            keep = keep * (f <= f.max() * (2 / 3)).double().reshape(view)
        self.keep = keep
        self.lap = -sum(k**2 for k in self.k)
        self.inv_lap = torch.where(self.lap == 0, torch.ones_like(self.lap), 1 / torch.where(self.lap == 0, 1.0, self.lap))

    def fft(self, u):
        return torch.fft.fftn(u, dim=self.dims)

    def phys(self, uh):
        return torch.fft.ifftn(uh, dim=self.dims).real

    def convection(self, uh):
        uh = uh * self.keep
        u = self.phys(uh)
        acc = 0.0
        for j, k in enumerate(self.k):
            acc = acc + u[:, j:j + 1] * self.phys(1j * k * uh)
        return self.fft(acc)

    def vorticity_convection(self, wh):
        wh = wh * self.keep
        psi = -wh * self.inv_lap
        kx, ky = self.k
        return self.fft(self.phys(1j * ky * psi) * self.phys(1j * kx * wh) - self.phys(1j * kx * psi) * self.phys(1j * ky * wh))

    def divergence(self, uh):
        return sum(1j * k * uh[:, j:j + 1] for j, k in enumerate(self.k))

    def gradient(self, ph):
        return torch.cat([1j * k * ph for k in self.k], dim=1)


def _phi(dt, L, order, f, points=32):
    """Mean over a unit circle around dt L of f: the removable singularities at 0 do no harm."""
    th = TWO_PI * (torch.arange(points, device=L.device, dtype=torch.float64) + 0.5) / points
    total = 0.0
    for t in th:
        z = dt * L + torch.exp(1j * t)
        total = total + f(z)
    return dt * (total / points).real


def _stepper(name, dt, L, nonlinear):
    E = torch.exp(dt * L)
    if name in ("ETDRK2", "SETDRK2"):
        c1 = _phi(dt, L, 1, lambda z: (torch.exp(z) - 1) / z)
        c2 = _phi(dt, L, 2, lambda z: (torch.exp(z) - 1 - z) / z**2)

        def step(u):
            n0 = nonlinear(u)
            a = E * u + c1 * n0
            return a + c2 * (nonlinear(a) - n0)

        return step
    E2 = torch.exp(0.5 * dt * L)
    q = _phi(dt, L, 1, lambda z: (torch.exp(z / 2) - 1) / z)
    c4 = _phi(dt, L, 3, lambda z: (-4 - z + torch.exp(z) * (4 - 3 * z + z**2)) / z**3)
    c5 = _phi(dt, L, 3, lambda z: (2 + z + torch.exp(z) * (-2 + z)) / z**3)
    c6 = _phi(dt, L, 3, lambda z: (-4 - 3 * z - z**2 + torch.exp(z) * (4 - z)) / z**3)

    def step(u):
        n0 = nonlinear(u)
        a = E2 * u + q * n0
        na = nonlinear(a)
        nb = nonlinear(E2 * u + q * na)
        nc = nonlinear(E2 * a + q * (2 * nb - n0))
        return E * u + c4 * n0 + 2 * c5 * (na + nb) + c6 * nc

    return step


def exact(c, seed):
    shape = _shape(c)
    u0, target = _inputs(c, seed)
    s = _Spectral(shape, c["length"], u0.device)
    u0 = u0.double()
    nu = torch.tensor(c["nu"], device=u0.device, dtype=torch.float64)
    if c["grad"]:
        u0.requires_grad_(True)
        nu.requires_grad_(True)
    if c["eq"] == "heat":
        return s.phys(torch.exp(c["dt"] * nu * s.lap) * s.fft(u0))
    if c["eq"] == "pressure":
        return s.phys(-s.inv_lap * s.divergence(s.convection(s.fft(u0))))
    if c["eq"] == "burgers":
        L, nonlinear = nu * s.lap, lambda uh: -s.convection(uh)
    elif c["eq"] == "ks":
        L, nonlinear = -s.lap - s.lap**2, lambda uh: -s.convection(uh)
    elif c["eq"] == "ns_vorticity":
        y = torch.arange(shape[1], device=u0.device, dtype=torch.float64) * (c["length"] / shape[1])
        force = s.fft((4.0 * torch.cos(4.0 * y)).reshape(1, 1, 1, -1).expand(1, 1, *shape))
        L, nonlinear = nu * s.lap - 0.1, lambda wh: -s.vorticity_convection(wh) - force
    else:
        def nonlinear(uh):
            conv = s.convection(uh)
            return s.gradient(s.inv_lap * s.divergence(conv)) - conv

        L = nu * s.lap
    step = _stepper(c["scheme"], c["dt"], L, nonlinear)
    uh = s.fft(u0)
    frames = [u0]
    for _ in range(c["steps"]):
        uh = step(uh)
        if c["record"]:
            frames.append(s.phys(uh))
    if c["record"]:
        return torch.stack(frames, dim=1)
    u = s.phys(uh)
    if c["grad"]:
        loss = torch.mean((u - target.double()) ** 2)
        g_u0, g_nu = torch.autograd.grad(loss, (u0, nu))
        return {"u": u.detach(), "grad_u0": g_u0, "grad_nu": g_nu}
    return u
