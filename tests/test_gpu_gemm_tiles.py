"""The bf16 products in 256x256 tiles (`big_tiles`): contractions of one partial stage up to
a few, ragged outputs, ragged and empty groups, and the two-segment product with k tails.

Against fp32 products of the same bf16 operands: an fp32 output's error is the order of an
fp32 sum over K <= 1000 terms (below 1e-6 of the result's norm), a bf16 output adds one
rounding (2^-9 of a value at most, 1.7e-3 of the norm for uniform mantissas)."""

import pytest
import torch

from param_decomp_amd import ops
from param_decomp_amd.decomposed_linear import SiteWeights, site_forward

pytestmark = pytest.mark.gpu


def _rel(got, want):
    return float((got.float() - want).norm() / want.norm())


def _rand(device, seed, *shape):
    g = torch.Generator(device=device).manual_seed(seed)
    return torch.randn(*shape, device=device, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("K", [8, 64, 72, 128, 136, 320])
@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
def test_big_tile_short_contractions(device, ta, tb, K):
    M, N = 3000, 4104
    a, b = _rand(device, 1, *((K, M) if ta else (M, K))), _rand(device, 2, *((N, K) if tb else (K, N)))
    want = (a.t() if ta else a).float() @ (b.t() if tb else b).float()
    assert _rel(ops.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb), out_dtype=torch.float32), want) < 1e-6
    assert _rel(ops.gemm(a, b, trans_a=bool(ta), trans_b=bool(tb)), want) < 2e-3


@pytest.mark.parametrize("K", [72, 256])
@pytest.mark.parametrize("sizes", [[20000, 0, 1, 300, 257], [4000, 4001, 3999, 4096, 4100]])
def test_big_tile_groups(device, sizes, K):
    E, J, N = len(sizes), sum(sizes), 520
    offs = torch.tensor([0] + sizes, device=device).cumsum(0).to(torch.int32)
    lhs, rhs = _rand(device, 3, J, K), _rand(device, 4, E, N, K)
    got = ops.grouped_gemm(lhs, rhs, offs, trans_rhs=True)
    want = torch.cat([x.float() @ rhs[e].float().t() for e, x in enumerate(lhs.split(sizes))])
    assert _rel(got, want) < 2e-3


@pytest.mark.parametrize("trans_rhs", [True, False])
@pytest.mark.parametrize("K", [72, 512])
def test_groups_of_few_rows(device, K, trans_rhs):
    sizes, N = [3, 0, 1, 130, 17, 0, 128, 64], 264
    offs = torch.tensor([0] + sizes, device=device).cumsum(0).to(torch.int32)
    lhs, rhs = _rand(device, 3, sum(sizes), K), _rand(device, 4, len(sizes), *((N, K) if trans_rhs else (K, N)))
    got = ops.grouped_gemm(lhs, rhs, offs, trans_rhs=trans_rhs)
    want = torch.cat([x.float() @ (rhs[e].float().t() if trans_rhs else rhs[e].float())
                      for e, x in enumerate(lhs.split(sizes))])
    assert _rel(got, want) < 2e-3


@pytest.mark.parametrize("d_in,C", [(200, 136), (64, 72), (8, 128)])
def test_big_tile_two_segments(device, d_in, C):
    T, d_out = 4000, 3072
    x, V, U, W = (_rand(device, 5 + i, *s) for i, s in enumerate([(T, d_in), (d_in, C), (C, d_out), (d_out, d_in)]))
    m, d = torch.rand(T, C, device=device).to(torch.bfloat16), torch.rand(T, device=device).to(torch.bfloat16)
    route = torch.arange(T, device=device) % 3 != 0
    out = site_forward(x, SiteWeights(W, V, U), m, d, route.to(torch.uint8)).output
    target = x.float() @ W.float().t()
    xV = (x.float() @ V.float()).to(torch.bfloat16).float()
    acts = (xV * (m.float() - d.float()[:, None])).to(torch.bfloat16).float()
    want = torch.where(route[:, None], acts @ U.float() + d.float()[:, None] * target, target)
    # the stored xV may round to the neighbouring bf16 value in another order of its sum
    assert _rel(out, want) < 4e-3


@pytest.mark.parametrize("K", [768, 776, 1000, 1032])
@pytest.mark.parametrize("M,N", [(1, 8), (300, 264), (2048, 2048)])
def test_four_stage_ring(device, M, N, K):
    a, b = _rand(device, 7, M, K), _rand(device, 8, N, K)
    got = ops.gemm(a, b, trans_b=True, out_dtype=torch.float32)
    # two fp32 sums of K terms in different orders, each within sqrt(K) 2^-24 = 1.9e-6
    assert _rel(got, a.float() @ b.float().t()) < 4e-6


@pytest.mark.parametrize("N", [1023, 1025, 1537, 3001])  # one slice, then a ragged last one
def test_ci_mlp_sliced_weight_gradient(device, N):
    dims = (72, 136, 64)
    x, g = _rand(device, 9, N, dims[0]), _rand(device, 10, N, dims[2])
    w = [_rand(device, 11 + i, dims[i], dims[i + 1]) for i in range(2)]
    b = [torch.zeros(d, dtype=torch.bfloat16, device=device) for d in dims[1:]]
    _, ws = ops.ci_mlp_fwd(x, w, b)
    dW, _, _ = ops.ci_mlp_bwd(x, w, g, ws, True)
    # the head's: the hidden activations round to bf16 from either order of their sum
    a = torch.nn.functional.gelu((x.float() @ w[0].float()).to(torch.bfloat16).float()).to(torch.bfloat16).float()
    assert _rel(dW[1], a.t() @ g.float()) < 4e-3


def _gelu_grad(z):
    return 0.5 * (1 + torch.erf(z * 0.5**0.5)) + z * torch.exp(-0.5 * z * z) * (2 * torch.pi)**-0.5


# 256x256 tiles with ragged edges in both directions (hidden layer, head and the pullback into
# the hidden layer); the four-stage ring with a k tail in the backward, with and without GELU'
@pytest.mark.parametrize("N,dims", [(3000, (72, 4104, 4104)), (300, (72, 776, 840))])
def test_ci_mlp_tiles(device, N, dims):
    x, g = _rand(device, 20, N, dims[0]), _rand(device, 21, N, dims[2])
    w = [(_rand(device, 22 + i, dims[i], dims[i + 1]).float() / dims[i]**0.5).to(torch.bfloat16) for i in range(2)]
    b = [_rand(device, 24 + i, dims[i + 1]) for i in range(2)]
    pre, ws = ops.ci_mlp_fwd(x, w, b)
    dW, db, dx = ops.ci_mlp_bwd(x, w, g, ws, True)
    r = lambda t: t.to(torch.bfloat16).float()  # noqa: E731
    wf, gf = [t.float() for t in w], g.float()
    z = r(r(x.float() @ wf[0]) + b[0].float())
    a = r(torch.nn.functional.gelu(z))
    dz = r(r(gf @ wf[1].t()) * _gelu_grad(z))
    want = dict(pre=r(r(a @ wf[1]) + b[1].float()), dx=r(dz @ wf[0].t()), dW0=x.float().t() @ dz, dW1=a.t() @ gf,
                db0=dz.sum(0), db1=gf.sum(0))
    got = dict(pre=pre, dx=dx, dW0=dW[0], dW1=dW[1], db0=db[0], db1=db[1])
    # values rounded to bf16 on the way may take the neighbour in another order of their sum
    for k in want:
        assert _rel(got[k], want[k]) < 4e-3, k
