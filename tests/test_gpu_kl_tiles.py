"""The bf16 streamed KL's tiles: the summation order of a tied head's statistics, and
contractions that fill one, two or three of the two-head ring's three stages.

A position's statistics over one 128 x 256 tile are fixed sums: each of two waves adds 128
columns (per lane half the 4-column groups 8g + 4h in order, the two halves added), and the
waves are added. Logits that fp32 holds exactly make those sums reproducible outside the
kernel, bit for bit: another order moves the last bits of logZ, and through the bf16
cotangents behind them the LM step's gradients by 1e-3 to 8e-3."""

import numpy as np
import pytest
import torch

from oracle import pd_oracle as po
from param_decomp_amd import _lib as L
from param_decomp_amd.losses import streamed_position_kl

pytestmark = pytest.mark.gpu


def _ordered_sum(ex):
    """Sum over the columns of ex [N, V], V <= 256, in the tile's order."""
    N, V = ex.shape
    ex = torch.nn.functional.pad(ex, (0, 256 - V))  # adding the missing columns' 0 changes nothing
    waves = []
    for w in range(2):
        halves = []
        for h in range(2):
            acc = torch.zeros(N, device=ex.device)
            for g in range(w * 16, w * 16 + 16):  # 8 columns each
                for e in range(4):
                    acc = acc + ex[:, 8 * g + 4 * h + e]
            halves.append(acc)
        waves.append(halves[0] + halves[1])
    return waves[0] + waves[1]


@pytest.mark.parametrize("N,V", [(512, 256), (300, 203), (64, 40)])
def test_tied_head_statistics_order(device, N, V):
    d = 72
    g = torch.Generator(device=device).manual_seed(V)
    quarters = lambda *s: (torch.randint(-4, 5, s, device=device, generator=g) / 4).to(torch.bfloat16)
    act_q, act_p, head = quarters(N, d), quarters(N, d), quarters(V, d)
    kl, stats = torch.empty(N, device=device), torch.empty(N, 5, device=device)
    dt = L.dtype_code(torch.bfloat16)
    ws = L.workspace(L.load().pd_streamed_kl_workspace_size(dt, N, d, V, 1), device)
    L.call("pd_streamed_kl_fwd", dt, N, d, V, 1, L.ptr(act_q), L.ptr(head), L.ptr(act_p), L.ptr(head), L.ptr(kl),
           L.ptr(stats), L.ptr(ws), ws.numel(), L.stream())
    for act, m_col, s_col in ((act_p, 0, 1), (act_q, 3, 4)):
        z = act.float() @ head.float().t()  # sixteenths below 2^7: exact in any order
        m = z.amax(1)
        assert torch.equal(stats[:, m_col], m)
        assert torch.equal(stats[:, s_col], _ordered_sum(torch.exp2((z - m[:, None]) * np.float32(1.44269504088896341))))


@pytest.mark.parametrize("d", [8, 64, 72, 136])
@pytest.mark.parametrize("n_chunks,V", [(1, 263), (3, 999)])
@pytest.mark.parametrize("shared", [False, True])
def test_short_contractions(device, d, n_chunks, V, shared):
    """Against the float64 oracle on the same bf16 inputs; the gradient passes through bf16
    (q - p) g on its way into its product: 2e-2 of a value or 1e-2 of the largest."""
    N = 150
    rng = np.random.default_rng(d + V)
    bf = lambda *s: torch.tensor(rng.normal(size=s) * 0.5, device=device).to(torch.bfloat16)  # noqa: E731
    n64 = lambda t: t.detach().float().cpu().numpy().astype(np.float64)  # noqa: E731
    aq, ap, hq = bf(N, d).requires_grad_(True), bf(N, d), bf(V, d)
    hp = hq if shared else bf(V, d)
    kl = streamed_position_kl(aq, hq, ap, hp, n_chunks)
    want, _ = po.streamed_position_kl(n64(aq), n64(hq), n64(ap), n64(hp), n_chunks)
    np.testing.assert_allclose(n64(kl), want, rtol=1e-3, atol=1e-4 * np.abs(want).max())
    g = rng.normal(size=N)
    (da,) = torch.autograd.grad(kl, aq, torch.tensor(g, dtype=torch.float32, device=device))
    want_da = po.streamed_position_kl_vjp(n64(aq), n64(hq), n64(ap), n64(hp), g)
    np.testing.assert_allclose(n64(da), want_da, rtol=2e-2, atol=1e-2 * np.abs(want_da).max())
