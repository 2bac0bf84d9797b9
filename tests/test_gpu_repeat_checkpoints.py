"""autograd.repeat keeps its checkpoints in the forward pass: the gradient
equals the one whose backward forms them itself (rollout_vjp), for every kind
of plan the repeat has, with a ragged last segment, one segment, strided inputs
and saved-tensor hooks. The final state is repeat_batch's, bit for bit."""
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
    "gs1d_100": (lambda: S.reaction.GrayScott(1, 2.5, 100, 1.0), 1, 100, 2),
    "kolmogorov2d_128": (lambda: S.KolmogorovFlowVorticity(2, 6.0, 128, 0.01, diffusivity=0.01), 2, 128, 1),
    "ns3d_32": (lambda: S.NavierStokesVelocity(3, 6.0, 32, 0.01), 3, 32, 3),
    "ns3d_16": (lambda: S.NavierStokesVelocity(3, 6.0, 16, 0.01), 3, 16, 3),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("n,every", [(7, 3), (6, 3), (4, 4), (5, 1), (3, 0)])
def test_kept_checkpoints_give_the_gradient(device, name, n, every):
    """Under every strategy of the plan: keeping the checkpoints changes no bit
    of the final state, and they are states of that rollout. The gradients run
    the same kernels from checkpoints that differ by the rounding of one
    transform round trip per segment; stated at 2e-5 of the gradient's norm, as
    for the rollout gradients."""
    import torch

    print(f"[case] {name} n={n} every={every}", flush=True)
    make, D, N, C = CASES[name]
    st = make()
    u0 = torch.tensor(ics(2, D, 1.0, N, 3, seed=5, channels=C)[0], device=device)
    g = torch.tensor(np.random.default_rng(6).standard_normal(u0.shape).astype(np.float32), device=device)
    wide = torch.stack([u0, u0], dim=1)[:, 0]
    assert not wide.is_contiguous()
    K = every if 0 < every < n else n
    for nt in (0, -1, 1, 2, 3):
        try:
            st.plan(len(u0)).set_rollout_strategy(nt)
        except (NotImplementedError, ValueError):
            continue
        ref = st.repeat_batch(u0, n)
        out, ckpt = st._repeat_checkpointed(u0, n, every)
        assert torch.equal(out, ref), nt
        assert ckpt.shape[0] == -(-n // K) - 1
        if nt != 0 and len(ckpt):  # (a rollout with 0 would choose a strategy)
            states = st.rollout_batch(u0, n)[:, K - 1:n - 1:K].movedim(1, 0)
            if name == "ks1d_128":  # formed by segments of their own
                assert float((ckpt - states).norm() / states.norm()) <= 1e-6, nt
            else:
                assert torch.equal(ckpt, states), nt
        want = st.rollout_vjp(u0, n, g_final=g, checkpoint_every=every)
        for v in (u0, wide):
            x = v.detach().requires_grad_(True)
            y = ex.autograd.repeat(st, x, n, checkpoint_every=every)
            assert torch.equal(y, ref), nt
            (gx,) = torch.autograd.grad(y, x, g, retain_graph=True)
            (again,) = torch.autograd.grad(y, x, g)
            assert torch.equal(gx, again)
            assert float((gx - want).norm() / want.norm()) <= 2e-5, nt


def test_only_a_graph_keeps_checkpoints(device, monkeypatch):
    """Nothing is kept where no gradient can follow, although the input asks
    for one."""
    import torch

    st = S.KuramotoSivashinskyConservative(1, 30.0, 60, 0.05)
    x = torch.tensor(ics(2, 1, 1.0, 60, 3, seed=5)[0], device=device, requires_grad=True)
    ref = st.repeat_batch(x.detach(), 6)
    kept = []
    monkeypatch.setattr(type(st), "_repeat_checkpointed",
                        lambda *a, _f=type(st)._repeat_checkpointed: kept.append(1) or _f(*a))
    with torch.no_grad():
        assert torch.equal(ex.autograd.repeat(st, x, 6, checkpoint_every=2), ref)
    assert torch.equal(ex.autograd.repeat(st, x.detach(), 6, checkpoint_every=2), ref)
    assert not kept
    ex.autograd.repeat(st, x, 6, checkpoint_every=2)
    assert kept == [1]
    # the fused 1-D sizes pass no checkpoints on their way
    fused = S.KuramotoSivashinskyConservative(1, 30.0, 64, 0.05)
    y = torch.tensor(ics(2, 1, 1.0, 64, 3, seed=5)[0], device=device, requires_grad=True)
    assert torch.equal(ex.autograd.repeat(fused, y, 6, checkpoint_every=2), fused.repeat_batch(y.detach(), 6))
    assert kept == [1]


def test_a_steppers_own_repeat_is_called(device):
    """A stepper that repeats or differentiates in its own way keeps doing so."""
    import torch

    class Mine(S.KuramotoSivashinskyConservative):
        def repeat_batch(self, u0, n, **kw):
            return 2.0 * super().repeat_batch(u0, n, **kw)

    class Scaled(S.KuramotoSivashinskyConservative):
        def rollout_vjp(self, *a, **kw):
            return 2.0 * super().rollout_vjp(*a, **kw)

    u0 = torch.tensor(ics(2, 1, 1.0, 60, 3, seed=5)[0], device=device)
    plain = S.KuramotoSivashinskyConservative(1, 30.0, 60, 0.05)
    x = u0.clone().requires_grad_(True)
    assert torch.equal(ex.autograd.repeat(Mine(1, 30.0, 60, 0.05), x, 6, checkpoint_every=2),
                       2.0 * plain.repeat_batch(u0, 6))
    (got,) = torch.autograd.grad(ex.autograd.repeat(Scaled(1, 30.0, 60, 0.05), x, 6, checkpoint_every=2).sum(), x)
    want = 2.0 * plain.rollout_vjp(u0, 6, g_final=torch.ones_like(u0), checkpoint_every=2)
    assert torch.equal(got, want)


def test_saved_tensor_hooks(device):
    """The checkpoints may leave the device between forward and backward; what
    comes back is looked at before a kernel reads it."""
    import torch

    st = S.KuramotoSivashinskyConservative(1, 30.0, 60, 0.05)
    x = torch.tensor(ics(2, 1, 1.0, 60, 3, seed=5)[0], device=device, requires_grad=True)
    y = ex.autograd.repeat(st, x, 6, checkpoint_every=2)
    (want,) = torch.autograd.grad(y.sum(), x)
    hooks = {"cpu": (lambda t: t.cpu(), lambda t: t),
             "strided": (lambda t: t, lambda t: torch.stack([t, t], dim=-1)[..., 0]),
             "double": (lambda t: t.double(), lambda t: t)}
    for name, (pack, unpack) in hooks.items():
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = ex.autograd.repeat(st, x, 6, checkpoint_every=2)
        (got,) = torch.autograd.grad(y.sum(), x)
        assert torch.equal(got, want), name
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t[:1]):
        y = ex.autograd.repeat(st, x, 6, checkpoint_every=2)
    with pytest.raises(ValueError):
        torch.autograd.grad(y.sum(), x)
