"""The network's launch shapes: four- and eight-wave workgroups (up to 1024
samples and above), more samples than resident wavefronts, and the
weight-gradient pass above and below one sample per wavefront, against the
bfloat16 oracle."""
import numpy as np
import pytest

from oracle import cnn as ocnn

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = np.asarray(a, np.float64).ravel(), np.asarray(b, np.float64).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("N,count", [(64, 1024), (64, 1025), (64, 8193), (32, 4100), (128, 2049)])
def test_forward_counts(device, N, count):
    """Every sample equals the same sample run in a batch of at most 8 (the
    arithmetic of a sample does not depend on the launch), and those equal the
    oracle at the tolerance of the parity test."""
    import torch

    from exponax_amd import corrector as cr

    print(f"[case] forward N={N} count={count}", flush=True)
    p = torch.tensor(cr.init_params(N, scale_last=1.0), device=device)
    x = torch.tensor(np.random.default_rng(count).standard_normal((count, 1, N)).astype(np.float32), device=device)
    y = cr.cnn_forward(p, x)
    for i in (0, 7, count // 2, count - 8):
        assert torch.equal(y[i:i + 8], cr.cnn_forward(p, x[i:i + 8].contiguous()))
    ref, _ = ocnn.forward(p.cpu().numpy(), x[-8:].cpu().numpy(), bf16_model=True)
    assert _rel(y[-8:].cpu().numpy() - x[-8:].cpu().numpy(), ref - x[-8:].cpu().numpy()) <= 1e-3


@pytest.mark.parametrize("N,count", [(64, 4), (64, 511), (64, 513), (32, 700), (128, 130)])
def test_backward_counts(device, N, count):
    import torch

    from exponax_amd import corrector as cr

    print(f"[case] backward N={N} count={count}", flush=True)
    cnn = cr.PeriodicCNN(cr.init_params(N, scale_last=1.0))
    rng = np.random.default_rng(count)
    x = torch.tensor(rng.standard_normal((count, 1, N)).astype(np.float32), device=device, requires_grad=True)
    dy = torch.tensor(rng.standard_normal((count, 1, N)).astype(np.float32), device=device)
    gx, gp = torch.autograd.grad(cnn.apply(x), (x, cnn.params), dy)
    rp, rx = ocnn.backward(cnn.params.detach().cpu().numpy(), x.detach().cpu().numpy(), dy.cpu().numpy(),
                           bf16_model=True)
    # the tolerance of the parity test: float32 summation order and the rare
    # bfloat16 rounding it flips
    d = dy.cpu().numpy()
    ep, ex_ = _rel(gp.cpu().numpy(), rp), _rel(gx.cpu().numpy() - d, rx - d)
    print(f"  params {ep:.2e}, input {ex_:.2e}", flush=True)
    assert ep <= 5e-3 and ex_ <= 5e-3
