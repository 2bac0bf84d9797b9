"""autograd.repeat keeps its checkpoints in the forward pass: the gradient
equals the one whose backward forms them itself (rollout_vjp), for every kind
of plan the repeat has, with a ragged last segment, one segment, and inputs
the kept form does not take."""
import numpy as np
import pytest

import exponax_amd as ex
from tests.helpers import ics

pytestmark = pytest.mark.gpu

S = ex.stepper
CASES = {
    "ks1d_128": (lambda: S.KuramotoSivashinskyConservative(1, 30.0, 128, 0.05), 1, 128, 1),
    "ks1d_100": (lambda: S.KuramotoSivashinskyConservative(1, 30.0, 100, 0.05), 1, 100, 1),
    "ks2d_64": (lambda: S.KuramotoSivashinsky(2, 30.0, 64, 0.05), 2, 64, 1),
    "ks2d_128": (lambda: S.KuramotoSivashinsky(2, 60.0, 128, 0.05), 2, 128, 1),
    "burgers2d_32": (lambda: S.Burgers(2, 1.0, 32, 1e-3, diffusivity=0.02), 2, 32, 2),
    "ks2d_60": (lambda: S.KuramotoSivashinsky(2, 30.0, 60, 0.05), 2, 60, 1),
    "ns3d_16": (lambda: S.NavierStokesVelocity(3, 6.0, 16, 0.01), 3, 16, 3),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("n,every", [(7, 3), (6, 3), (4, 4), (5, 1), (3, 0)])
def test_kept_checkpoints_give_the_gradient(device, name, n, every):
    """Both forms run the same kernels from checkpoints that differ by the
    rounding of one transform round trip per segment; stated at 2e-5 of the
    gradient's norm, as for the rollout gradients."""
    import torch

    print(f"[case] {name} n={n} every={every}", flush=True)
    make, D, N, C = CASES[name]
    st = make()
    u0 = torch.tensor(ics(2, D, 1.0, N, 3, seed=5, channels=C)[0], device=device)
    g = torch.tensor(np.random.default_rng(6).standard_normal(u0.shape).astype(np.float32), device=device)
    x = u0.clone().requires_grad_(True)
    y = ex.autograd.repeat(st, x, n, checkpoint_every=every)
    ref = st.repeat_batch(u0, n)
    assert float((y.detach() - ref).norm() / ref.norm()) <= 5e-6
    (gx,) = torch.autograd.grad(y, x, g, retain_graph=True)
    (again,) = torch.autograd.grad(y, x, g)
    assert torch.equal(gx, again)
    want = st.rollout_vjp(u0, n, g_final=g, checkpoint_every=every)
    assert float((gx - want).norm() / want.norm()) <= 2e-5
    # a strided input takes the other form
    wide = torch.stack([u0, u0], dim=1)[:, 0].requires_grad_(True)
    assert not wide.is_contiguous()
    (gw,) = torch.autograd.grad(ex.autograd.repeat(st, wide, n, checkpoint_every=every), wide, g)
    assert float((gw - want).norm() / want.norm()) <= 2e-5
