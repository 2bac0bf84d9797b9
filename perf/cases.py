"""The measured work: calls that a program using this package makes, at sizes
from its own configurations, examples and tests, and the sizes around them.

A case is one family of calls (``FAMILIES``) at one size. The equations' own
settings follow the grid so that every size stays resolved: the
Kuramoto-Sivashinsky domains grow with the number of points, the Burgers
viscosities fall with it. ``exact`` restates each call in float64 with torch's
transforms.
"""
import math

import numpy as np
import torch

import exponax_amd as ex
from exponax_amd import autograd, corrector

DEVICE = "cuda:0"


# --------------------------------------------------------------------- cases
def listed():
    return [
        # one state stepped once, as an interactive loop or a host-side scheme does: the smallest call
        dict(name="step_ks1d_n256", family="step_ks1d", points=256, batch=1, steps=1),
        # one long trajectory of the reference's own example size: a serial chain of small steps
        dict(name="rollout_ks1d_n256_b1", family="rollout_ks1d", points=256, batch=1, steps=200),
        # the batched data set: one trajectory per viscosity, every state kept
        dict(name="rollout_burgers1d_n1024_b4096", family="ensemble_burgers1d", points=1024, batch=4096, steps=100),
        # emulator training data on the reference's 100-point grid, a size that is no power of two
        dict(name="rollout_burgers1d_n100_b100", family="rollout_burgers1d", points=100, batch=100, steps=200),
        # the reference's README workload shape: 2-D Kuramoto-Sivashinsky trajectories
        dict(name="rollout_ks2d_n128_b32", family="rollout_ks2d", points=128, batch=32, steps=50),
        # forced 2-D turbulence at the practical 2-D resolution, a Reynolds number per instance
        dict(name="rollout_kolmogorov2d_n512_b8", family="ensemble_kolmogorov2d", points=512, batch=8, steps=40),
        # the same on the odd grid of the reference's spectrum validation
        dict(name="rollout_kolmogorov2d_n513_b8", family="ensemble_kolmogorov2d", points=513, batch=8, steps=20),
        # 3-D incompressible turbulence, velocity form
        dict(name="rollout_ns3d_n64_b8", family="rollout_ns3d", points=64, batch=8, steps=20),
        # 3-D Burgers at the practical 3-D resolution, not a power of two
        dict(name="rollout_burgers3d_n48_b2", family="rollout_burgers3d", points=48, batch=2, steps=20),
        # the gradient of a loss through 50 solver steps, checkpoints every 10
        dict(name="grad_ks2d_n128_b32", family="grad_ks2d", points=128, batch=32, steps=50),
        # one iteration of the learned corrector's training: four unrolled steps, forward and backward
        dict(name="train_corrector_n64_b512", family="train_corrector", points=64, batch=512, steps=4),
        # inference with the corrected coarse solver
        dict(name="rollout_corrector_n64_b8192", family="rollout_corrector", points=64, batch=8192, steps=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A grid size of a multi-dimensional run, odd ones among them, without
    the large prime factors that nobody picks there."""
    while True:
        n = rest = rng.randint(lo, hi)
        for p in (2, 3, 5, 7, 11, 13, 17, 19):
            while rest % p == 0:
                rest //= p
        if rest == 1:
            return n


def draw(rng):
    family = rng.choice(["step_ks1d", "rollout_ks1d", "ensemble_burgers1d", "rollout_burgers1d", "rollout_ks2d",
                         "ensemble_kolmogorov2d", "rollout_ns3d", "rollout_burgers3d", "grad_ks2d",
                         "train_corrector", "rollout_corrector"])
    if family == "step_ks1d":
        points, batch, steps = rng.choice([rng.randint(32, 600), 2 ** rng.randint(5, 11)]), _log_int(rng, 1, 64), 1
    elif family == "rollout_ks1d":
        points, batch, steps = 2 ** rng.randint(5, 11), rng.randint(1, 4), rng.randint(50, 200)
    elif family == "ensemble_burgers1d":
        points, batch, steps = 2 ** rng.randint(7, 10), _log_int(rng, 256, 4096), rng.randint(20, 100)
    elif family == "rollout_burgers1d":
        points, batch, steps = rng.randint(40, 600), _log_int(rng, 4, 200), rng.randint(16, 60)
    elif family == "rollout_ks2d":
        points, batch, steps = rng.choice([32, 64, 128, _grid(rng, 40, 160)]), rng.randint(1, 32), rng.randint(16, 50)
    elif family == "ensemble_kolmogorov2d":
        points = rng.choice([128, 256, 512, _grid(rng, 64, 513)])
        batch, steps = rng.randint(1, 8), rng.randint(16, 20)
    elif family == "rollout_ns3d":
        points, batch, steps = rng.choice([16, 32, 64, _grid(rng, 16, 56)]), rng.randint(1, 8), rng.randint(16, 20)
    elif family == "rollout_burgers3d":
        points, batch, steps = rng.choice([32, 64, _grid(rng, 16, 56)]), rng.randint(1, 3), rng.randint(16, 20)
    elif family == "grad_ks2d":
        points = rng.choice([32, 64, 128, _grid(rng, 32, 100)])
        batch, steps = rng.randint(1, 16), rng.randint(10, 40)
    elif family == "train_corrector":
        points, batch, steps = rng.choice([32, 64, 128]), _log_int(rng, 64, 1024), rng.randint(1, 4)
    else:
        points, batch, steps = rng.choice([32, 64]), _log_int(rng, 128, 8192), rng.randint(5, 20)
    return dict(family=family, points=points, batch=batch, steps=steps)


# ----------------------------------------------------------------- equations
class Equation:
    """One family's equation: how to build its stepper, and what its step is
    in float64 (``linear``: L of |kappa|^2; ``nonlinear``: spectra to spectra)."""

    def __init__(self, kind, dims, channels, extent, dt, cutoff):
        self.kind, self.dims, self.channels, self.extent, self.dt, self.cutoff = kind, dims, channels, extent, dt, cutoff


def equation(case):
    f, n = case["family"], case["points"]
    if "corrector" in f:  # the coarse stepper: dt = 0.5 on the coarse grid
        return Equation("ks_conservative", 1, 1, 100.0 * n / 64, 0.5, 5)
    if f.endswith("ks1d"):
        return Equation("ks_conservative", 1, 1, 100.0 * n / 256, 0.05, 5)
    if f.endswith("burgers1d"):
        return Equation("burgers", 1, 1, 1.0, 1e-3, 5)
    if f.endswith("ks2d"):
        return Equation("ks", 2, 1, 60.0 * n / 128, 0.05, 5)
    if f.endswith("kolmogorov2d"):
        return Equation("kolmogorov", 2, 1, 2 * math.pi, 0.01, 6)
    if f.endswith("ns3d"):
        return Equation("navier_stokes", 3, 3, 2 * math.pi, 0.01, 3)
    return Equation("burgers", 3, 3, 1.0, 1e-3, 2)


def coefficients(case, seed):
    """The members' diffusivities (one where the batch shares it)."""
    eq, n = equation(case), case["points"]
    rng = np.random.default_rng([seed, 17])
    if eq.kind == "burgers" and eq.dims == 1:
        nu = 10.0 ** rng.uniform(-3.0, -2.0, case["batch"]) * (1024 / n)
    elif eq.kind == "kolmogorov":
        nu = 1.0 / rng.uniform(100.0, 1000.0, case["batch"])
    elif eq.kind == "burgers":
        nu = np.array([0.02])
    else:
        nu = np.array([0.01])
    return nu if case["family"].startswith("ensemble") else nu[:1]


def make_stepper(eq, n, nu):
    s = ex.stepper
    if eq.kind == "ks_conservative":
        return s.KuramotoSivashinskyConservative(1, eq.extent, n, eq.dt)
    if eq.kind == "ks":
        return s.KuramotoSivashinsky(2, eq.extent, n, eq.dt)
    if eq.kind == "burgers":
        return s.Burgers(eq.dims, eq.extent, n, eq.dt, diffusivity=float(nu))
    if eq.kind == "kolmogorov":
        return s.KolmogorovFlowVorticity(2, eq.extent, n, eq.dt, diffusivity=float(nu))
    return s.NavierStokesVelocity(3, eq.extent, n, eq.dt, diffusivity=float(nu))


def states(case, seed, stream=0):
    """Seeded smooth fields (batch, C, N, ..., N) of unit maximum: a band of
    Fourier modes with normal amplitudes, made in float64."""
    eq, n = equation(case), case["points"]
    gen = torch.Generator(device="cpu").manual_seed(1000 * int(seed) + stream)
    k = min(eq.cutoff, n // 2 - 1)
    count = case["batch"] * eq.channels
    band = torch.zeros((count,) + (2 * k + 1,) * (eq.dims - 1) + (k + 1,), dtype=torch.complex128)
    band.real = torch.randn(band.shape, generator=gen, dtype=torch.float64)
    band.imag = torch.randn(band.shape, generator=gen, dtype=torch.float64)
    hat = torch.zeros((count,) + (n,) * (eq.dims - 1) + (n // 2 + 1,), dtype=torch.complex128, device=DEVICE)
    at = torch.arange(-k, k + 1) % n
    index = torch.meshgrid(*([at] * (eq.dims - 1) + [torch.arange(k + 1)]), indexing="ij")
    hat[(slice(None),) + tuple(i.to(DEVICE) for i in index)] = band.to(DEVICE)
    hat[(slice(None),) + (0,) * eq.dims] = 0.0
    u = torch.fft.irfftn(hat, s=(n,) * eq.dims, dim=tuple(range(1, eq.dims + 1)))
    u = u / u.abs().amax(dim=tuple(range(1, eq.dims + 1)), keepdim=True)
    return u.reshape((case["batch"], eq.channels) + (n,) * eq.dims).to(torch.float32).contiguous()


def network(seed):
    """Seeded parameters of the trained network's shape, the last layer scaled
    so that its corrections are as small as a trained one's."""
    return corrector.init_params(int(seed) % 1000, scale_last=0.01)


# ------------------------------------------------------------------ the calls
def prepare(case, seed):
    eq, n, family = equation(case), case["points"], case["family"]
    nu = coefficients(case, seed)
    u = states(case, seed)
    if family.startswith("ensemble"):
        stepper = ex.ensemble(lambda v: make_stepper(eq, n, v), nu)
    else:
        stepper = make_stepper(eq, n, nu[0])
    state = dict(case=case, stepper=stepper, u=u)
    if family == "step_ks1d":
        state["call"] = stepper if case["batch"] == 1 else ex.vmap(stepper)
        state["u"] = u[0] if case["batch"] == 1 else u
        state["call"](state["u"])
    elif "corrector" in family:
        cnn = corrector.PeriodicCNN(network(seed))
        state["cnn"] = cnn
        state["corrected"] = corrector.CorrectedStepper(stepper, cnn)
        if family == "train_corrector":
            # what follows the drawn windows' first states in the training data
            state["targets"] = [states(case, seed, stream=j + 1) for j in range(case["steps"])]
    elif family == "grad_ks2d":
        state["target"] = states(case, seed, stream=1)
    else:
        stepper.rollout_batch(u, 16)  # a plan chooses among its kernels on its first rollout of 16 steps
    return state


def run(state):
    case, stepper, u = state["case"], state["stepper"], state["u"]
    family, steps = case["family"], case["steps"]
    if family == "step_ks1d":
        return state["call"](u)
    if family == "train_corrector":
        cnn, loss = state["cnn"], 0.0
        for target in state["targets"]:
            u = cnn.apply(autograd.step(stepper, u))
            loss = loss + ((u - target) ** 2).mean()
        loss = loss / steps
        (grad,) = torch.autograd.grad(loss, cnn.params)
        return {"state": u.detach(), "loss": loss.detach(), "grad": grad}
    if family == "rollout_corrector":
        return state["corrected"].rollout_batch(u, steps)
    if family == "grad_ks2d":
        x = u.clone().requires_grad_(True)
        y = autograd.repeat(stepper, x, steps, checkpoint_every=10)
        loss = ((y - state["target"]) ** 2).mean()
        loss.backward()
        return {"loss": loss.detach(), "grad": x.grad}
    return stepper.rollout_batch(u, steps)


# --------------------------------------------------------------- what it takes
CNN_FLOPS_PER_POINT = 2 * (1 * 32 * 5 + 3 * 32 * 32 * 5 + 32 * 1 * 5)
# real transforms of one nonlinear evaluation, per batch member (fields in, products out)
TRANSFORMS = {"ks_conservative": 2, "ks": 3, "kolmogorov": 5, "navier_stokes": 9}


def work(case):
    eq, n, b, steps = equation(case), case["points"], case["batch"], case["steps"]
    field = n ** eq.dims
    modes = n ** (eq.dims - 1) * (n // 2 + 1)
    transform = 2.5 * field * math.log2(field)
    per_eval = TRANSFORMS.get(eq.kind, 3 if eq.dims == 1 else 15)
    step_flops = b * transform * (2 * per_eval + eq.channels)
    state = 4 * b * eq.channels * field
    tables = 12 * modes * (b if case["family"].startswith("ensemble") else 1)
    cnn = b * n * CNN_FLOPS_PER_POINT
    if case["family"] == "train_corrector":  # backward: the step's transpose, the network's two products per layer
        return {"bytes": state * (2 + steps) + tables, "flops": steps * (3 * cnn + 2 * step_flops)}
    if case["family"] == "rollout_corrector":
        return {"bytes": state * (1 + steps) + tables, "flops": steps * (cnn + step_flops)}
    if case["family"] == "grad_ks2d":  # forward, transposed steps; the states between are recomputed or kept
        return {"bytes": 3 * state + tables, "flops": 2 * steps * step_flops}
    return {"bytes": state * (1 + steps) + tables, "flops": steps * step_flops}


def tolerance(case):
    """About four times what float64 and the float32 (network: bfloat16) paths differ by."""
    return {
        "train_corrector": {"rel": 2e-2, "max": 0.5},
        "rollout_corrector": {"rel": 5e-3, "max": 0.2},
        "rollout_ks1d": {"rel": 3e-5, "max": 3e-4},  # the trajectories part slowly: the equation is chaotic
        "grad_ks2d": {"rel": 2.5e-5, "max": 2.5e-4},
    }.get(case["family"], {"rel": 7e-6, "max": 1e-4})


# ------------------------------------------------------------- float64 restated
class Exact:
    """ETDRK2 in float64 for one equation on one grid."""

    def __init__(self, eq, n, nu):
        self.eq, self.n, D = eq, n, eq.dims
        self.axes = tuple(range(-D, 0))
        full = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=DEVICE)
        half = torch.arange(n // 2 + 1, dtype=torch.float64, device=DEVICE)
        k = torch.stack(torch.meshgrid(*([full] * (D - 1) + [half]), indexing="ij"))
        self.k, self.kappa = k, k * (2 * math.pi / eq.extent)
        # the reference compares with the cutoff in float32
        self.mask = (k.abs() <= float(np.float32((2 / 3) * (n // 2) - 1))).all(dim=0).to(torch.float64)
        k2 = (self.kappa ** 2).sum(dim=0)
        nu = torch.as_tensor(nu, dtype=torch.float64, device=DEVICE).reshape((-1,) + (1,) * (D + 1))
        if eq.kind == "ks_conservative" or eq.kind == "ks":
            # the fourth derivatives are summed along the axes, without mixed ones
            L = k2 - (self.kappa ** 4).sum(dim=0) + 0 * nu
        elif eq.kind == "kolmogorov":
            L = -nu * k2 - 0.1
        else:
            L = -nu * k2
        self.inverse_laplacian = torch.where(k2 > 0, -1.0 / torch.where(k2 > 0, k2, 1.0), 0.0)
        dt = eq.dt
        self.E = torch.exp(L * dt)
        circle = torch.exp(2j * math.pi * (torch.arange(1, 17, dtype=torch.float64, device=DEVICE) - 0.5) / 16)
        self.c1, self.c2 = torch.zeros_like(L), torch.zeros_like(L)
        for z in circle:
            lr = z + L * dt
            self.c1 += dt * ((torch.exp(lr) - 1) / lr).real / 16
            self.c2 += dt * ((torch.exp(lr) - 1 - lr) / lr ** 2).real / 16

    def fft(self, u):
        return self.mask * torch.fft.rfftn(u, dim=self.axes)

    def ifft(self, hat):
        return torch.fft.irfftn(self.mask * hat, s=(self.n,) * self.eq.dims, dim=self.axes)

    def nonlinear(self, hat):
        eq, i = self.eq, 1j
        if eq.kind == "ks_conservative":
            return -0.5 * i * self.kappa * self.fft(self.ifft(hat) ** 2)
        if eq.kind == "ks":
            g = sum(self.ifft(i * kd * hat) ** 2 for kd in self.kappa)
            return -0.5 * self.fft(g - g.mean(dim=self.axes, keepdim=True))
        if eq.kind == "burgers":
            u = self.ifft(hat)
            return -self.fft(sum(u[:, d:d + 1] * self.ifft(i * self.kappa[d] * hat) for d in range(eq.dims)))
        if eq.kind == "kolmogorov":
            psi, (kx, ky) = self.inverse_laplacian * hat, self.kappa
            conv = self.ifft(i * ky * psi) * self.ifft(i * kx * hat) - self.ifft(i * kx * psi) * self.ifft(i * ky * hat)
            forcing = torch.where((self.k[0] == 0) & (self.k[1] == 4), -4.0 * self.n ** 2 / 2, 0.0)
            return -self.fft(conv) + forcing
        kap = self.kappa
        curl = torch.stack([i * (kap[1] * hat[:, 2] - kap[2] * hat[:, 1]), i * (kap[2] * hat[:, 0] - kap[0] * hat[:, 2]),
                            i * (kap[0] * hat[:, 1] - kap[1] * hat[:, 0])], dim=1)
        c = self.fft(torch.cross(self.ifft(hat), self.ifft(curl), dim=1))
        return c + kap * (self.inverse_laplacian * (kap * c).sum(dim=1, keepdim=True))

    def __call__(self, u):
        hat = torch.fft.rfftn(u, dim=self.axes)
        n0 = self.nonlinear(hat)
        a = self.E * hat + self.c1 * n0
        b = a + self.c2 * (self.nonlinear(a) - n0)
        return torch.fft.irfftn(b, s=(self.n,) * self.eq.dims, dim=self.axes)


def _network(params, x):
    """y = x + f(x): five periodic convolutions of width 5, tanh-form GELU between."""
    at, a = 0, x
    shapes = [(32, 1), (32, 32), (32, 32), (32, 32), (1, 32)]
    for layer, (co, ci) in enumerate(shapes):
        w = params[at:at + co * ci * 5].reshape(co, ci, 5)
        b = params[at + co * ci * 5:at + co * ci * 5 + co]
        at += co * ci * 5 + co
        z = b[:, None] + sum((w[None, :, :, j, None] * torch.roll(a, 2 - j, dims=-1)[:, None]).sum(dim=2) if ci == 1
                             else torch.matmul(w[:, :, j].contiguous(), torch.roll(a, 2 - j, dims=-1)) for j in range(5))
        a = torch.nn.functional.gelu(z, approximate="tanh") if layer < 4 else z
    return x + a


def exact(case, seed):
    eq, n, steps, family = equation(case), case["points"], case["steps"], case["family"]
    step = Exact(eq, n, coefficients(case, seed))
    u = states(case, seed).double()
    if family == "step_ks1d":
        out = step(u)
        return out[0] if case["batch"] == 1 else out
    if "corrector" in family:
        params = torch.tensor(network(seed), device=DEVICE).double()
        if family == "train_corrector":
            params.requires_grad_(True)
            loss = 0.0
            for j in range(steps):
                u = _network(params, step(u))
                loss = loss + ((u - states(case, seed, stream=j + 1).double()) ** 2).mean()
            loss = loss / steps
            (grad,) = torch.autograd.grad(loss, params)
            return {"state": u.detach(), "loss": loss.detach(), "grad": grad}
        outs = []
        for _ in range(steps):
            u = _network(params, step(u))
            outs.append(u)
        return torch.stack(outs, dim=1)
    if family == "grad_ks2d":
        u.requires_grad_(True)
        y = u
        for _ in range(steps):
            y = step(y)
        loss = ((y - states(case, seed, stream=1).double()) ** 2).mean()
        (grad,) = torch.autograd.grad(loss, u)
        return {"loss": loss.detach(), "grad": grad}
    out = torch.empty((case["batch"], steps) + tuple(u.shape[1:]), dtype=torch.float64, device=DEVICE)
    for t in range(steps):
        u = step(u)
        out[:, t] = u
    return out
