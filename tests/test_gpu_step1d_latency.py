"""The 1-D rollout kernels with twice the lanes per transform (strategy 3)
against the ones with the usual number (strategy 1): every size and kind they
are built for, both forms of carrying the state, ragged batches, repeat and
the failure-detecting rollout."""
import numpy as np
import pytest

import exponax_amd as ex
from tests.helpers import ics, max_rel_l2

pytestmark = pytest.mark.gpu

S = ex.stepper


def _stepper(kind, N, physical):
    if kind == "conv":
        st = S.KuramotoSivashinskyConservative(1, 100.0 * N / 256, N, 0.05)
    elif kind == "conv_exact":
        st = S.Burgers(1, 1.0, N, 1e-3, diffusivity=0.02 * 256 / N)
        st.exact_form = True
    else:
        st = S.KuramotoSivashinsky(1, 100.0 * N / 256, N, 0.05)
    if physical:
        st.fourier_resident = False
    return st


@pytest.mark.parametrize("N", [64, 128, 256, 512, 2048])
@pytest.mark.parametrize("kind", ["conv", "conv_exact", "gradnorm"])
def test_latency_variant_equals_the_usual(device, kind, N):
    """Both compute the same step with the transform's passes split another
    way: float32 rounding apart, 1e-6 over 12 steps as between the other
    strategies."""
    import torch

    for physical in (False, True):
        for B in (1, 7):
            print(f"[case] {kind} N={N} physical={physical} B={B}", flush=True)
            st = _stepper(kind, N, physical)
            x = torch.tensor(ics(B, 1, 1.0, N, 5, seed=N + B)[0], device=device)
            plan, outs, reps = st.plan(B), {}, {}
            for nt in (1, 3):
                plan.set_rollout_strategy(nt)
                outs[nt] = st.rollout_batch(x, 12, include_init=True).cpu().numpy()
                reps[nt] = st.repeat_batch(x, 12).cpu().numpy()
                np.testing.assert_array_equal(outs[nt][:, 0], x.cpu().numpy())
                np.testing.assert_array_equal(reps[nt], outs[nt][:, -1])
            for s in range(1, 13):
                assert max_rel_l2(outs[3][:, s], outs[1][:, s]) <= 1e-6, s
            tr, bad = st.rollout_checked(x, 3)
            assert bool((bad == -1).all())
            tr, bad = st.rollout_checked(x, 3, bound=1e-3)
            assert bool((bad == 0).all())


def test_not_built_elsewhere(device):
    """Sizes, orders and kinds without the variant refuse the strategy."""
    for st in (S.KuramotoSivashinskyConservative(1, 100.0, 48, 0.05),
               S.KuramotoSivashinskyConservative(1, 400.0, 1024, 0.05),
               S.KuramotoSivashinskyConservative(1, 100.0, 4096, 0.01),
               S.KuramotoSivashinskyConservative(1, 100.0, 256, 0.05, order=4),
               S.KortewegDeVries(1, 20.0, 256, 1e-3), S.reaction.AllenCahn(1, 1.0, 256, 1e-3)):
        with pytest.raises(NotImplementedError):
            st.plan(2).set_rollout_strategy(3)


@pytest.mark.parametrize("N,B", [(64, 8192), (64, 8193), (256, 2048), (256, 2049), (2048, 512), (2048, 513)])
def test_untuned_repeat_takes_it_up_to_one_wavefront_per_simd(device, N, B):
    """A repeat before any rollout was timed: strategy 3 as long as its
    wavefronts (two per transform at N = 2048) are no more than the 1024 SIMDs,
    2 above. The strategies' bits tell which one ran."""
    import torch

    st = S.KuramotoSivashinskyConservative(1, 100.0 * N / 256, N, 0.05)
    x = torch.tensor(ics(8, 1, 1.0, N, 5, seed=N)[0], device=device).repeat(B // 8 + 1, 1, 1)[:B].contiguous()
    got = st.repeat_batch(x, 20)
    bits = {}
    for nt in (2, 3):
        st.plan(B).set_rollout_strategy(nt)
        bits[nt] = st.repeat_batch(x, 20)
    assert not torch.equal(bits[2], bits[3])
    assert torch.equal(got, bits[2 if B % 2 else 3])
