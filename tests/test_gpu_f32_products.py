"""The fp32 products' direct form: K-contiguous operands in loads of 4, 2 and 1 floats (by K,
row stride and base alignment), contractions that end inside a batch and outputs inside a
tile; and the native ResidualMLP step where its products change form: one contraction slice
and several, weight gradients one at a time, products on the LDS-staged form.

Tolerance of a product: an fp32 sum of K unit-variance terms in slices is below
sqrt(K) * 2^-24 of the result's norm, under 3e-6 for K <= 2048. The step against the same
step composed of separate products under autograd: a few such sums one after another, 1e-5
of each gradient's norm (the bound of the oracle comparison)."""

import pytest
import torch

from param_decomp_amd import _lib as L, ops, toys

pytestmark = pytest.mark.gpu


def _rel(got, want):
    return float((got.double() - want.double()).norm() / want.double().norm())


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (33, 65, 17), (64, 31, 50), (300, 70, 100), (40, 33, 1026), (2048, 1000, 50),
                                   (100, 70, 2048)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 0), (2, 0), (1, 0), (4, 2), (4, 1)])
def test_direct_form_load_widths(device, M, N, K, pad, shift):
    g = torch.Generator(device=device).manual_seed(M + K)

    def operand(r, c):  # a view with row stride c + pad, `shift` floats into its storage
        buf = torch.randn(shift + r * (c + pad), device=device, generator=g)
        return buf[shift:].as_strided((r, c), (c + pad, 1), shift)

    for ta in (False, True):
        for tb in (False, True):
            a, b = operand(*((K, M) if ta else (M, K))), operand(*((N, K) if tb else (K, N)))
            got = torch.empty(M, N, device=device)
            L.call("pd_gemm", L.dtype_code(a.dtype), M, N, K, a.data_ptr(), a.stride(0), int(ta), b.data_ptr(),
                   b.stride(0), int(tb), L.ptr(got), N, L.dtype_code(got.dtype), 1.0, 0.0, L.stream())
            assert _rel(got, (a.t() if ta else a).double() @ (b.t() if tb else b).double()) < 3e-6, (ta, tb)


# one to five 16-deep batches per wave and none, whole and ragged, in blocks of 8 and 16 waves
# (70 x 40) and of one wave per tile (2048 x 1024)
@pytest.mark.parametrize("M,N,K", [(70, 40, k) for k in (16, 31, 130, 256, 257, 300, 384, 511, 512, 700, 1100, 1300)] +
                         [(2048, 1024, k) for k in (5, 16, 33, 48, 64, 250)])
def test_direct_form_batches(device, M, N, K):
    g = torch.Generator(device=device).manual_seed(K)
    for ta in (False, True):
        for tb in (False, True):
            a = torch.randn(*((K, M) if ta else (M, K)), device=device, generator=g)
            b = torch.randn(*((N, K) if tb else (K, N)), device=device, generator=g)
            got = ops.gemm(a, b, trans_a=ta, trans_b=tb, out_dtype=torch.float32)
            assert _rel(got, (a.t() if ta else a).double() @ (b.t() if tb else b).double()) < 3e-6, (ta, tb)


@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
def test_no_contraction(device, ta, tb, beta):
    """K = 0 with padded rows leaves beta C, plain and batched, and reads neither operand."""
    M, N, ld = 40, 33, 64
    a, b = torch.ones(8, ld, device=device), torch.ones(8, ld, device=device)
    for call, z in ((lambda c: L.call("pd_gemm", L.dtype_code(a.dtype), M, N, 0, L.ptr(a), ld, ta, L.ptr(b), ld, tb,
                                      L.ptr(c), N, L.dtype_code(c.dtype), 1.0, beta, L.stream()), 1),
                    (lambda c: L.call("pd_gemm_strided_batched", L.dtype_code(a.dtype), 2, M, N, 0, L.ptr(a), ld, ld,
                                      ta, L.ptr(b), ld, ld, tb, L.ptr(c), N, M * N, L.dtype_code(c.dtype), 1.0, beta,
                                      L.stream()), 2)):
        c = torch.randn(z, M, N, device=device)
        want = beta * c
        call(c)
        assert torch.equal(c, want)


@pytest.mark.parametrize("B,F,D,M,C,n_layers", [(3, 20, 100, 10, 20, 2), (511, 33, 101, 13, 37, 2), (1030, 33, 102, 14, 36, 3),
                                         (64, 24, 1000, 20, 520, 1), (33000, 20, 300, 30, 20, 1)])
def test_resid_mlp_step_product_forms(device, B, F, D, M, C, n_layers):
    g = torch.Generator(device=device).manual_seed(B)
    target, sites = toys.init_resid_mlp(F, D, M, n_layers, C, device=device, generator=g)
    x = toys.sparse_features(B, F, 0.1, -1.0, device=device, generator=g)
    params = [p for s in sites for p in s.parameters()]
    want = toys.ToyDecompositionStep(target, sites, p=2.0).step(x, (5, 6))
    want = [want["loss"].clone(), want["out"].clone()] + [p.grad.clone() for p in params]
    res = toys.ResidMLPFusedStep(target, sites, p=2.0).step(x, (5, 6))
    got = [res["loss"], res["out"]] + [p.grad for p in params]
    for i, (a, b) in enumerate(zip(got, want)):
        assert _rel(a, b) < 1e-5, i
