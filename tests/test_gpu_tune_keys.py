"""The tuning cache's keys say what was timed: choices made on a step belong to
one equation and shape, and an entry of another is not taken for them."""
import numpy as np
import pytest

import exponax_amd as ex
from tests.helpers import ics

pytestmark = pytest.mark.gpu

S = ex.stepper
# equal D, N and number of fields within each row
PAIRS = {
    "kinds": [(lambda: S.KuramotoSivashinsky(2, 30.0, 60, 0.05), 3, 1),
              (lambda: S.KolmogorovFlowVorticity(2, 2 * np.pi, 60, 0.01, diffusivity=0.01), 3, 1)],
    "orders": [(lambda: S.KuramotoSivashinsky(2, 30.0, 60, 0.05, order=2), 3, 1),
               (lambda: S.KuramotoSivashinsky(2, 30.0, 60, 0.05, order=4), 3, 1)],
    "channels": [(lambda: S.Burgers(3, 1.0, 12, 1e-3, diffusivity=0.02), 2, 3),
                 (lambda: S.KuramotoSivashinsky(3, 30.0, 12, 0.05), 6, 1)],
}


@pytest.mark.parametrize("pair", list(PAIRS))
def test_each_is_timed_for_itself(device, pair, tmp_path, monkeypatch):
    import torch

    path = tmp_path / "tune.txt"
    monkeypatch.setenv("EXMI_TUNE_CACHE", str(path))
    # what a library that timed bare transforms left for this D, N and count
    S.Burgers(1, 1.0, 100, 1e-3).fft_config(batch=1)
    arch = path.read_text().split("|")[0]
    make, B, C = PAIRS[pair][0]
    st = make()
    old = f"{arch}|gfft|D{st.num_spatial_dims}|N{st.num_points}|I{B * C}"
    path.write_text(f"{old} 100800256\n")
    for make, B, C in PAIRS[pair]:
        st = make()
        print(f"[case] {pair} {type(st).__name__} B={B}", flush=True)
        first = st.fft_config(batch=B)
        assert first["source"] == "timed"
        again = make().fft_config(batch=B)
        assert again["source"] == "cache" and again["code"] == first["code"]
        D, N = st.num_spatial_dims, st.num_points
        st.rollout_batch(torch.tensor(ics(B, D, 1.0, N, 3, seed=1, channels=C)[0], device=device) * 0.1, 16)
    keys = [ln.rsplit(" ", 1)[0] for ln in path.read_text().split("\n") if ln.strip()]
    # the old entry; a transform choice and a rollout strategy of each
    assert len(keys) == len(set(keys)) == 5, keys


def test_the_reported_code_given_back_changes_nothing(device, tmp_path, monkeypatch):
    """1-D plans step with radices of their own: reading a plan's knobs and
    setting them again leaves every bit alone, another code is used there too."""
    import torch

    path = tmp_path / "tune.txt"
    monkeypatch.setenv("EXMI_TUNE_CACHE", str(path))
    make = lambda: S.Burgers(1, 1.0, 100, 1e-3, diffusivity=0.02)  # noqa: E731
    make().fft_config(batch=3)
    key = path.read_text().split("\n")[0].rsplit(" ", 1)[0]
    path.write_text(f"{key} 101002048\n")  # two passes of ten points
    st = make()
    plan = st.plan(3)
    cfg = plan.fft_config()
    assert cfg["source"] == "cache" and cfg["radices"] == [10, 10]
    plan.set_rollout_strategy(2)
    u0 = torch.tensor(ics(3, 1, 1.0, 100, 5, seed=3)[0], device=device)
    want = st.rollout_batch(u0, 8)
    plan.set_fft_config(cfg["code"])
    assert plan.fft_config()["code"] == cfg["code"]
    assert torch.equal(st.rollout_batch(u0, 8), want)
    plan.set_fft_config(200000 + 1024)  # 2 2 5 5
    got = st.rollout_batch(u0, 8)
    assert not torch.equal(got, want) and float((got - want).norm() / want.norm()) <= 3e-6
