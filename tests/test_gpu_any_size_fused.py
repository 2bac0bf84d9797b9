"""The fused passes of the runtime grid sizes against the general ones.

1-D: a step, a rollout and a repeat of a size whose lines fit LDS run as one
launch; the same step through fft, step_fourier and ifft runs the separate
passes. 2-D and 3-D: the fields fused with the first inverse axis and the rows
fused with the products, at sizes on both sides of the LDS limit and with an
odd number of rows, against the oracle."""
import numpy as np
import pytest

import exponax_amd as ex
from oracle import stepper as ost
from tests.helpers import RTOL_STEP, ics, max_rel_l2

pytestmark = pytest.mark.gpu

S = ex.stepper


def _steppers_1d(N):
    """Every 1-D kind, order and operator form, with its number of channels."""
    out = []
    for order in (1, 2, 3, 4):
        out.append((f"burgers o{order}", S.Burgers(1, 1.0, N, 1e-3, diffusivity=0.02, order=order), 1))
        out.append((f"kdv o{order}", S.KortewegDeVries(1, 20.0, N, 1e-3, order=order), 1))
    nc = S.Burgers(1, 1.0, N, 1e-3, diffusivity=0.02)
    nc.exact_form = True
    out += [("burgers exact form", nc, 1), ("ks", S.KuramotoSivashinsky(1, 30.0, N, 0.05), 1),
            ("ks o4", S.KuramotoSivashinsky(1, 30.0, N, 0.05, order=4), 1),
            ("general", S.generic.GeneralNonlinearStepper(1, 2.0, N, 1e-3, linear_coefficients=(0.0, 0.0, 0.01),
                                                          nonlinear_coefficients=(0.3, -1.0, -0.5)), 1),
            ("allen-cahn", S.reaction.AllenCahn(1, 1.0, N, 1e-3), 1),
            ("cahn-hilliard", S.reaction.CahnHilliard(1, 1.0, N, 1e-5), 1),
            ("gray-scott", S.reaction.GrayScott(1, 2.5, N, 1.0), 2),
            ("advection o0", S.Advection(1, 2.0, N, 0.01, velocity=0.8), 1)]
    return out


@pytest.mark.parametrize("N", [3, 11, 97, 100, 243, 1023, 1050])
def test_1d_one_launch_equals_separate_passes(device, N):
    """The two routes do the same float32 arithmetic up to the order of the
    transforms' sums: each is within a few eps log2(N) (eps sqrt(R) per
    direct pass of a prime R) of the exact step, the difference within twice
    that; stated at 3e-6."""
    import torch

    B = 5
    for name, st, C in _steppers_1d(N):
        print(f"[case] {name} N={N}", flush=True)
        u0 = ics(B, 1, 1.0, N, min(5, (N - 1) // 2), seed=7 + N, channels=C)[0]
        x = torch.tensor(u0, device=device) * 0.5
        a = st.step(x)
        b = ex.spectral.ifft(st.step_fourier(ex.spectral.fft(x, num_spatial_dims=1)), num_spatial_dims=1,
                             num_points=N)
        e = max_rel_l2(a.cpu().numpy().reshape(B, 1, -1), b.cpu().numpy().reshape(B, 1, -1))
        assert e <= 3e-6, (name, N, e)
        # a rollout's first state is the step; repeat is its last state; a
        # strided batch (the trajectory buffer) steps as a contiguous one
        tr = st.rollout_batch(x, 3, include_init=True)
        assert torch.equal(tr[:, 0], x) and max_rel_l2(tr[:, 1].cpu().numpy().reshape(B, 1, -1),
                                                       a.cpu().numpy().reshape(B, 1, -1)) <= 3e-6
        assert torch.equal(st.repeat_batch(x, 3), tr[:, 3])


@pytest.mark.parametrize("nt", [2, -1])
def test_1d_per_member_tables_and_channels(device, nt):
    """Per-trajectory operators (lin_batch = B) and per-channel ones take each
    workgroup's own tables: a member's bits are those of its own plan with the
    same strategy (the spectrum carried, or a float32 round trip per step:
    other kernels, other bits), and the per-channel ones those of the oracle."""
    import torch

    nus = np.linspace(0.01, 0.05, 7)
    rates = [(2e-5, 1e-5), (4e-5, 1e-5), (3e-5, 2e-5)]
    for name, make, ps, C in (("burgers", lambda nu: S.Burgers(1, 1.0, 77, 1e-3, diffusivity=float(nu)), nus, 1),
                              ("gray-scott", lambda d: S.reaction.GrayScott(1, 2.5, 77, 1.0, diffusivity_1=d[0],
                                                                            diffusivity_2=d[1]), rates, 2)):
        print(f"[case] {name} strategy {nt}", flush=True)
        B = len(ps)
        ens = ex.ensemble(make, ps)
        u0 = torch.tensor(0.5 * ics(B, 1, 1.0, 77, 5, seed=3, channels=C)[0], device=device)
        ens.plan(B).set_rollout_strategy(nt)
        got = ens.rollout_batch(u0, 4)
        for i, v in enumerate(ps):
            one = make(v)
            one.plan(1).set_rollout_strategy(nt)
            assert torch.equal(got[i:i + 1], one.rollout_batch(u0[i:i + 1], 4)), (name, i)
    cpu = ost.GrayScott(1, 2.5, 77, 1.0, diffusivity_1=rates[1][0], diffusivity_2=rates[1][1], dtype=np.float32)
    u = u0[1:2].cpu().numpy()
    for s in range(4):
        u = cpu.step_batch(u)
        assert max_rel_l2(got[1:2, s].cpu().numpy(), u) <= RTOL_STEP


@pytest.mark.parametrize("N", [6, 33, 99, 810, 825, 1025])
def test_2d_rows_with_products(device, N):
    """Kolmogorov flow (four fields): 810 is the largest smooth even size below
    the row kernel's LDS limit (64 KiB of line pairs), which odd sizes reach
    above 1024: 1025 runs the separate passes; 33, 99, 825 and 1025 leave a
    last row alone."""
    import torch

    print(f"[case] kolmogorov N={N}", flush=True)
    L, dt = 2 * np.pi, 0.005
    gpu = S.KolmogorovFlowVorticity(2, L, N, dt, diffusivity=0.01, injection_mode=2)
    cpu = ost.KolmogorovFlowVorticity(2, L, N, dt, diffusivity=0.01, injection_mode=2, dtype=np.float32)
    u0 = ics(2, 2, L, N, min(4, (N - 1) // 2), seed=N)[0]
    got = gpu.rollout_batch(torch.tensor(u0, device=device), 2).cpu().numpy()
    u = u0
    for s in range(2):
        u = cpu.step_batch(u)
        e = max_rel_l2(got[:, s], u)
        assert e <= RTOL_STEP, (N, s, e)


@pytest.mark.parametrize("kind,N,C", [("bz", 15, 3), ("general", 9, 1), ("ns", 10, 3), ("ns", 21, 3), ("gs", 18, 2)])
def test_3d_rows_with_products(device, kind, N, C):
    import torch

    print(f"[case] 3-D {kind} N={N}", flush=True)
    kw = dict(dtype=np.float32)
    if kind == "bz":
        gpu, cpu = S.reaction.BelousovZhabotinsky(3, 1.0, N, 1e-3), ost.BelousovZhabotinsky(3, 1.0, N, 1e-3, **kw)
    elif kind == "gs":
        gpu, cpu = S.reaction.GrayScott(3, 2.5, N, 1.0), ost.GrayScott(3, 2.5, N, 1.0, **kw)
    elif kind == "ns":
        gpu, cpu = S.NavierStokesVelocity(3, 6.0, N, 0.01), ost.NavierStokesVelocity(3, 6.0, N, 0.01, **kw)
    else:
        lin, nonlin = (0.0, 0.0, 0.01), (0.3, -1.0, -0.5)
        gpu = S.generic.GeneralNonlinearStepper(3, 2.0, N, 1e-3, linear_coefficients=lin,
                                                nonlinear_coefficients=nonlin)
        cpu = ost.GeneralStepper(3, 2.0, N, 1e-3, linear_coefficients=lin, nonlinear_scales=nonlin, **kw)
    u0 = 0.5 * ics(3, 3, 1.0, N, 3, seed=N, channels=C)[0]
    got = gpu.rollout_batch(torch.tensor(u0, device=device), 2).cpu().numpy()
    u = u0
    for s in range(2):
        u = cpu.step_batch(u)
        e = max_rel_l2(got[:, s], u)
        assert e <= RTOL_STEP, (kind, N, s, e)
