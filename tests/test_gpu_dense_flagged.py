"""The bf16 dense step's flagged components (a hidden unit wider than 3 in z over one moment
bin), whose gates are evaluated exactly, one token per lane: none, a few sharing waves with
unflagged ones, and every component; token counts that end inside a wave and inside a
block of the passes. Against the oracle's float64 step at the bf16 tolerance."""

import numpy as np
import pytest
import torch

from oracle import pd_oracle as po
from oracle import threefry as tf
from param_decomp_amd.dense_step import DenseSiteStep
from param_decomp_amd.losses import ImpMin

pytestmark = pytest.mark.gpu
RTOL = 2e-2


@pytest.mark.parametrize("T,d_in,d_out,C", [(8, 64, 64, 72), (328, 64, 96, 200), (1032, 40, 64, 136)])
@pytest.mark.parametrize("wide", ["none", "some", "all"])
@pytest.mark.parametrize("sl0", [False, True])
def test_dense_step_flagged_components(device, T, d_in, d_out, C, wide, sl0):
    rng = np.random.default_rng(T + C)
    f = lambda t: t.float().cpu().numpy().astype(np.float64)  # noqa: E731
    t = lambda a, dt: torch.tensor(np.asarray(a, np.float32), device=device).to(dt)  # noqa: E731
    x, W, V, U = (t(a, torch.bfloat16) for a in (
        rng.normal(size=(T, d_in)), rng.normal(size=(d_out, d_in)) / d_in**0.5, rng.normal(size=(d_in, C)) / d_in**0.5,
        rng.normal(size=(C, d_out)) / C**0.5))
    w_in = rng.normal(size=(C, 16)) * 1.4
    h = f(x) @ f(V)
    span = (h.max(0) - h.min(0)) / 16
    w_in *= np.minimum(1.0, 2.0 / (np.abs(w_in).max(1) * span))[:, None]  # none flagged
    which = {"none": [], "some": [0, 5, 33, C - 1], "all": list(range(C))}[wide]
    w_in[which] *= (4.5 / (np.abs(w_in[which]).max(1) * span[which]))[:, None]
    gate = [t(a, torch.float32) for a in (w_in, np.zeros((C, 16)), rng.normal(size=(C, 16)) * 0.35, np.full(C, 0.3))]
    kw = dict(coeff=0.7, gamma=0.5, frequency_coeff=0.05, reference_datapoint_count=64.0)
    step = DenseSiteStep(T, d_in, d_out, C, device=device, use_delta=True,
                         imp_min=ImpMin.smooth_l0(**kw) if sl0 else None)
    key = tf.fold_in(tf.prng_key(3), T)
    g = step.step(x, W, V, U, tuple(gate), *step.site_keys(key, 0))
    spec = po.ImpMin("smooth_l0", coeff=0.7, gamma=0.5, freq_coeff=0.05, ref_count=64.0) if sl0 else None
    r = po.dense_site_step(f(x), f(W), f(V), f(U), po.GateParams(*(f(a) for a in gate)), key, mask_dtype="bfloat16",
                           use_delta=True, bf16_storage=True, **({"imp_min": spec} if sl0 else {}))
    np.testing.assert_allclose(g.losses.cpu().numpy(), [r.loss, r.recon, r.imp, r.freq], rtol=RTOL, atol=1e-7)
    for got, want, name in [(g.dU, r.dU, "dU"), (g.dV, r.dV, "dV"),
                            *zip((g.dw_in, g.db_in, g.dw_out, g.db_out), r.dgate, ("dw_in", "db_in", "dw_out", "db_out"))]:
        err = np.abs(f(got) - want)
        assert (err <= RTOL * np.abs(want) + 1e-2 * np.abs(want).max()).all(), (name, err.max(), np.abs(want).max())
