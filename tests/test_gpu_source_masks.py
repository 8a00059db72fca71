"""The mask kernels' source-table reads and column sums where their paths divide: tables
whose base is not aligned to a four-value load, tiles holding many (expert, source row)
groups with more experts than lanes, and source rows of more jobs than a wave takes."""

import pytest
import torch

from oracle import moe_oracle as mo
from test_gpu_moe import _make
from test_gpu_moe_sources import _tables

pytestmark = pytest.mark.gpu

U = 2.0**-24  # fp32 rounding: a sum of n terms is within n U of the sum of their magnitudes


def _step(cfg, rps, inputs, src, srcd):
    from param_decomp_amd.moe_step import MoEStackStep

    w, ci, x0 = inputs
    step = MoEStackStep(cfg.T, cfg.d, cfg.f, cfg.E, cfg.k, cfg.c, cfg.L, device=x0.device, p=2.0, imp_coeff=1e-3,
                        recon_coeff=1.5, rows_per_source=rps)
    step.step_sources(x0, w, ci, src, srcd)
    torch.cuda.synchronize()
    return {n: getattr(step, n).clone() for n in ("losses", "d_src", "d_src_delta", "d_ci_pre")}


def _per_token(t, rps):
    wide = t.to(torch.int32) if t.dtype == torch.uint16 else t
    return wide.repeat_interleave(rps, dim=2).to(t.dtype)


@pytest.mark.parametrize("T,E,k,rps,dtype", [(520, 70, 3, 520, torch.float32), (520, 70, 3, 8, torch.bfloat16),
                                             (1024, 5, 2, 512, torch.uint16), (520, 70, 3, 1, torch.float32),
                                             (520, 9, 2, 104, torch.bfloat16)])
def test_moe_table_alignment_and_groups(device, T, E, k, rps, dtype):
    cfg = mo.MoEConfig(T=T, d=64, f=32, E=E, k=k, c=72, L=1)
    _, _, _, w, ci, x0 = _make(cfg, 0, device)
    src, srcd, _, _ = _tables(cfg, rps, dtype, True, 5, device)
    raw = torch.empty(src.numel() + 1, dtype=dtype, device=device)
    off = raw[1:].view(src.shape)  # one element past the allocation's alignment
    off.copy_(src)
    a = _step(cfg, rps, (w, ci, x0), src, srcd)
    b = _step(cfg, rps, (w, ci, x0), off, srcd)
    for n in a:
        assert torch.equal(a[n], b[n]), n
    # the same sources as one table row per token: each row's gradient is its tokens' sum
    one = _step(cfg, 1, (w, ci, x0), _per_token(src, rps), _per_token(srcd, rps))
    assert torch.equal(one["losses"], a["losses"]) and torch.equal(one["d_ci_pre"], a["d_ci_pre"])
    for n, terms, slack in (("d_src", rps, 1), ("d_src_delta", rps * k, 16)):
        # (a token's delta gradient is a sum of k terms that may cancel: 16 times its magnitude)
        parts = one[n].double().unflatten(2, (-1, rps))
        bound = slack * terms * U * parts.abs().sum(3) + 1e-30
        assert ((a[n].double() - parts.sum(3)).abs() <= bound).all(), n
