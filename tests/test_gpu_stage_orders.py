"""Every stage combination of the runtime-size passes against the oracle: ETDRK
orders 1 to 4, real and complex linear operators, one table for all channels,
one per channel and one per trajectory; and the sizes whose rows run fused
while the last forward axis does not fit its workgroup."""
import numpy as np
import pytest

import exponax_amd as ex
from oracle import stepper as ost
from tests.helpers import RTOL_STEP, ics, max_rel_l2

pytestmark = pytest.mark.gpu

KINDS = {  # (maker, channels of dimension D)
    "ks": (lambda m, D, N, o, **k: m.KuramotoSivashinsky(D, 30.0, N, 0.05, order=o, **k), lambda D: 1),
    "kdv": (lambda m, D, N, o, **k: m.KortewegDeVries(D, 20.0, N, 1e-3, order=o, **k), lambda D: D),
    "gray_scott": (lambda m, D, N, o, **k: m.reaction.GrayScott(D, 2.5, N, 1.0, order=o) if m is ex.stepper
                   else m.GrayScott(D, 2.5, N, 1.0, order=o, **k), lambda D: 2),
}


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("D,N", [(2, 33), (2, 60), (3, 12), (3, 15)])
def test_orders(device, kind, order, D, N):
    """Two steps, so that the state behind the cutoff (which the stages alone
    move) is read again; an even and an odd size per dimension."""
    import torch

    print(f"[case] {kind} {D}-D N={N} order {order}", flush=True)
    make, channels = KINDS[kind]
    gpu, cpu = make(ex.stepper, D, N, order), make(ost, D, N, order, dtype=np.float32)
    u0 = 0.5 * ics(3, D, 1.0, N, 4, seed=N + order, channels=channels(D))[0]
    got = gpu.rollout_batch(torch.tensor(u0, device=device), 2).cpu().numpy()
    u = u0
    for s in range(2):
        u = cpu.step_batch(u)
        e = max_rel_l2(got[:, s], u)
        assert e <= RTOL_STEP, (s, e)


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("D,N", [(2, 33), (3, 12)])
def test_tables_per_trajectory_and_channel(device, D, N, order):
    """An ensemble of two-channel reactions: each member's channels have an
    operator of their own."""
    import torch

    print(f"[case] {D}-D N={N} order {order}", flush=True)
    rates = [(2e-5, 1e-5), (4e-5, 1e-5), (3e-5, 2e-5)]
    ens = ex.ensemble(lambda d: ex.stepper.reaction.GrayScott(D, 2.5, N, 1.0, diffusivity_1=d[0], diffusivity_2=d[1],
                                                              order=order), rates)
    u0 = 0.5 * ics(3, D, 1.0, N, 4, seed=N, channels=2)[0]
    got = ens.rollout_batch(torch.tensor(u0, device=device), 2).cpu().numpy()
    for i, d in enumerate(rates):
        cpu = ost.GrayScott(D, 2.5, N, 1.0, diffusivity_1=d[0], diffusivity_2=d[1], order=order, dtype=np.float32)
        u = u0[i:i + 1]
        for s in range(2):
            u = cpu.step_batch(u)
            assert max_rel_l2(got[i:i + 1, s], u) <= RTOL_STEP, (i, s)


@pytest.mark.parametrize("N", [800, 810])
def test_rows_fused_without_the_stage(device, N):
    """Conservative Burgers in 2-D, four products: at 810 a pair of rows fills
    the workgroup's 64 KiB and the last forward axis with its line starts does
    not fit any more, so it runs by itself and the combine reads spectra whose
    entries behind the cutoff were never written; 800 has the fused stage."""
    import torch

    print(f"[case] burgers N={N}", flush=True)
    kw = dict(diffusivity=0.02, conservative=True)
    gpu = ex.stepper.Burgers(2, 1.0, N, 1e-3, **kw)
    cpu = ost.Burgers(2, 1.0, N, 1e-3, dtype=np.float32, **kw)
    u0 = 0.5 * ics(1, 2, 1.0, N, 4, seed=N, channels=2)[0]
    got = gpu.rollout_batch(torch.tensor(u0, device=device), 2).cpu().numpy()
    u = u0
    for s in range(2):
        u = cpu.step_batch(u)
        e = max_rel_l2(got[:, s], u)
        assert e <= RTOL_STEP, (N, s, e)
