"""Differentiable stepping for PyTorch: ``torch.autograd.Function`` wrappers
whose backward passes run the hand-written adjoint kernels.

The reference gets its derivatives from ``jax.grad`` through ``lax.scan``
(``_utils.py:92-254``, README.md:85-91). It keeps every step's residuals. Here
one state every ``checkpoint_every`` steps is kept (by the forward pass of
``repeat`` where it passes them, else by the backward) and each segment is
recomputed on the way back.

    u0 = torch.randn(32, 1, 128, 128, device="cuda", requires_grad=True)
    uT = exponax_amd.autograd.repeat(stepper, u0, 50, checkpoint_every=10)
    loss = ((uT - target) ** 2).mean()
    loss.backward()          # u0.grad via exmi_rollout_vjp
"""
from __future__ import annotations

import torch

from ._base_stepper import BaseStepper, Ensemble
from ._tensor import as_float32


class _Step(torch.autograd.Function):
    @staticmethod
    def forward(ctx, u, stepper):
        ctx.stepper = stepper
        ctx.save_for_backward(u)
        return stepper.step(u.detach())

    @staticmethod
    def backward(ctx, g):
        (u,) = ctx.saved_tensors
        return ctx.stepper.step_vjp(u.detach(), g.contiguous()), None


class _Rollout(torch.autograd.Function):
    @staticmethod
    def forward(ctx, u0, stepper, n, include_init, checkpoint_every):
        ctx.stepper, ctx.n, ctx.include_init, ctx.k = stepper, n, include_init, checkpoint_every
        ctx.save_for_backward(u0)
        return stepper.rollout_batch(u0.detach(), n, include_init=include_init)

    @staticmethod
    def backward(ctx, g_traj):
        (u0,) = ctx.saved_tensors
        g = ctx.stepper.rollout_vjp(u0.detach(), ctx.n, g_traj=g_traj.contiguous(), include_init=ctx.include_init,
                                    checkpoint_every=ctx.k)
        return g, None, None, None, None


class _Repeat(torch.autograd.Function):
    @staticmethod
    def forward(ctx, u0, stepper, n, checkpoint_every, keep):
        ctx.stepper, ctx.n, ctx.k, ctx.keep = stepper, n, checkpoint_every, keep
        # the checkpoints the backward starts its segments from are states
        # this pass goes through: kept here, the backward need not run it again
        if keep:
            out, ckpt = stepper._repeat_checkpointed(as_float32(u0.detach()), n, checkpoint_every)
            ctx.save_for_backward(u0, ckpt)
            return out
        ctx.save_for_backward(u0)
        return stepper.repeat_batch(u0.detach(), n)

    @staticmethod
    def backward(ctx, g):
        if ctx.keep:
            u0, ckpt = ctx.saved_tensors
            return ctx.stepper._repeat_vjp(u0.detach(), ctx.n, ckpt, g, ctx.k), None, None, None, None
        (u0,) = ctx.saved_tensors
        return ctx.stepper.rollout_vjp(u0.detach(), ctx.n, g_final=g.contiguous(), checkpoint_every=ctx.k), None, \
            None, None, None


def _check(u):
    if not (isinstance(u, torch.Tensor) and u.is_cuda):
        raise TypeError("exponax_amd.autograd expects a torch tensor on the HIP device")


def step(stepper, u):
    """One step of a batch ``(..., C, N^D)``, differentiable in ``u``."""
    _check(u)
    return _Step.apply(u, stepper)


def rollout(stepper, u0, n: int, *, include_init: bool = False, checkpoint_every: int = 10):
    """``exponax.rollout(stepper, n, include_init)(u0)`` batched over leading
    axes: ``(..., n[+1], C, N^D)``, differentiable in ``u0``."""
    _check(u0)
    return _Rollout.apply(u0, stepper, n, include_init, checkpoint_every)


def repeat(stepper, u0, n: int, *, checkpoint_every: int = 10):
    """``exponax.repeat(stepper, n)(u0)``, differentiable in ``u0``: the bits
    of ``stepper.repeat_batch``. Where a gradient can follow, the states after
    every ``checkpoint_every`` steps are kept with the graph until its backward
    (ceil(n / checkpoint_every) - 1 batches of states; in 1-D for the runtime
    sizes only)."""
    _check(u0)
    keep = (torch.is_grad_enabled() and u0.requires_grad and 0 < (checkpoint_every or 0) < n and _own_repeat(stepper)
            and _writes_checkpoints(stepper, u0))
    return _Repeat.apply(u0, stepper, n, checkpoint_every, keep)


def _own_repeat(stepper):
    """Whether the stepper's repeat is the library's, on one plan (an ensemble
    of several groups has a plan for each)."""
    return (isinstance(stepper, BaseStepper) and getattr(stepper, "_groups", None) is None
            and type(stepper).repeat_batch in (BaseStepper.repeat_batch, Ensemble.repeat_batch)
            and type(stepper).rollout_vjp is BaseStepper.rollout_vjp)


def _writes_checkpoints(stepper, u0):
    """Whether the steps up to the end pass the checkpoints on their way: not
    the one launch of the fused 1-D sizes, whose backward forms them as
    ``rollout_vjp`` does."""
    if stepper.num_spatial_dims > 1:
        return True
    return stepper.plan(stepper._split(u0, stepper.state_shape)[1]).fft_config() is not None
