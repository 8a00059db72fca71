"""The calls whose speed this repository is measured on, over the sizes and options they are used at.

`listed()` and `draw(rng)` give cases (dicts of plain values), `prepare(case, seed)` what a
program holds before the call, `run(state)` one pass through the public entry points,
`work(case)` the bytes and operations a pass cannot do without, `tolerance(case)` how far
another correct implementation may be, and `exact(case, seed)` the same outputs in 64 bits
from plain torch operations.

Inputs follow the repository's benchmark: targets N(0, 1/d_in), components V N(0, 1/d_in) and
U N(0, 1/C), CI preactivations uniform on (-0.3, 1.3) (every branch of both squashings,
their ties in bf16 included), unit-scale activations, Kaiming gates.
"""

from __future__ import annotations

import math

import torch

from param_decomp_amd import toys
from param_decomp_amd.ci_fn import SiteMLP
from param_decomp_amd.decomposed_linear import SiteWeights, site_forward
from param_decomp_amd.dense_step import DenseSiteStep
from param_decomp_amd.faithfulness import FaithfulnessLoss
from param_decomp_amd.lm_step import KINDS, LMStackStep, LMWeights, site_dims
from param_decomp_amd.losses import ImpMin, streamed_position_kl
from param_decomp_amd.moe_step import SITE_NAMES, MoEStackStep, MoEWeights

F64 = torch.float64
BF16 = torch.bfloat16
HEAD = 64  # head width of the LM stack
GATE = 16  # hidden width of a component's gate
SL0 = dict(coeff=0.7, gamma=0.5, frequency_coeff=0.05, reference_datapoint_count=256.0)


# ------------------------------------------------------------------------------------ cases
def listed():
    return [
        # TMS 5-2 training step at its configured batch: the smallest call, a latency case
        dict(name="tms_5_2", kind="tms", B=4096, use_delta=False, p=1.0),
        # ResidualMLP training step at its configured size (fp32, 1000-wide, C = 100)
        dict(name="resid_mlp_1l", kind="resid", B=2048, F=100, D=1000, M=50, C=100, L=1, p=2.0),
        # one decomposed dense linear's training step at the benchmark's size
        dict(name="dense_step_768x3072", kind="dense", T=4096, d_in=768, d_out=3072, C=4096, dtype="bf16",
             use_delta=False, smooth_l0=False),
        # a down-projection site inside a caller's own autograd model, ragged token count,
        # with the delta channel and per-token routes
        dict(name="site_3072x768_routed", kind="site", T=3001, d_in=3072, d_out=768, C=4096, dtype="bf16", delta=True,
             route=True),
        # the engine's layerwise CI MLP of one site, forward and backward
        dict(name="ci_mlp_768_1024_4096", kind="ci_mlp", T=4096, d_in=768, hidden=1024, C=4096),
        # faithfulness of every expert gate matrix of the MoE stack, forward and backward (fp32)
        dict(name="faith_moe_gate", kind="faith", g=4, E=42, d_in=512, d_out=256, C=512, w_dtype="bf16"),
        # the streamed KL over an untied pair of heads, forward and backward
        dict(name="streamed_kl_50277", kind="kl", N=2048, d=768, V=50277, chunks=3),
        # the MoE stack's training step, the configuration the throughput figure is quoted on
        dict(name="moe_4l", kind="moe", T=8192, d=512, f=256, E=42, k=8, c=512, L=4, smooth_l0=False, use_delta=True,
             routes=False, rps=0),
        # a small MoE batch with the engine's smooth-L0 loss and per-token routes
        dict(name="moe_2l_small_routed", kind="moe", T=520, d=256, f=128, E=16, k=4, c=128, L=2, smooth_l0=True,
             use_delta=True, routes=True, rps=0),
        # the source half of a persistent-PGD step over the MoE stack: one warmup scoring
        # (source gradients alone), then the final call with every gradient
        dict(name="moe_4l_sources", kind="moe", T=8192, d=512, f=256, E=42, k=8, c=512, L=4, smooth_l0=False,
             use_delta=True, routes=False, rps=512),
        # the Llama-style LM stack's training step at the benchmark's size
        dict(name="lm_4l", kind="lm", B=16, T=512, H=12, KV=12, f=3072, V=50277, L=4, Ca=1024, Cm=4096, chunks=3,
             smooth_l0=False, use_delta=True, routes=False, rps=0),
        # a small LM batch: grouped-query attention, smooth-L0, per-token routes
        dict(name="lm_2l_small_gqa", kind="lm", B=3, T=192, H=6, KV=2, f=1024, V=8001, L=2, Ca=384, Cm=768, chunks=3,
             smooth_l0=True, use_delta=True, routes=True, rps=0),
    ]


def _log(rng, lo, hi, step=1):
    """An integer in [lo, hi], spread over its logarithm, a multiple of `step`."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step
    return min(max(v, -(-lo // step) * step), hi // step * step)


def draw(rng):
    kind = rng.choice(["tms", "resid", "dense", "site", "ci_mlp", "faith", "kl", "moe", "moe", "lm", "lm"])
    coin = lambda p=0.5: rng.random() < p  # noqa: E731
    if kind == "tms":
        return dict(kind=kind, B=_log(rng, 64, 16384), use_delta=coin(), p=rng.choice([1.0, 2.0]))
    if kind == "resid":
        return dict(kind=kind, B=_log(rng, 128, 4096), F=_log(rng, 20, 128), D=_log(rng, 100, 1200),
                    M=_log(rng, 10, 100), C=_log(rng, 20, 160), L=rng.choice([1, 2, 3]), p=rng.choice([1.0, 2.0]))
    if kind == "dense":
        fp32 = coin(0.25)
        return dict(kind=kind, T=_log(rng, 256, 2048 if fp32 else 8192, 8), d_in=_log(rng, 64, 3072, 8),
                    d_out=_log(rng, 64, 3072, 8), C=_log(rng, 128, 1024 if fp32 else 8192, 8),
                    dtype="fp32" if fp32 else "bf16", use_delta=coin(), smooth_l0=coin())
    if kind == "site":
        fp32 = coin(0.25)
        return dict(kind=kind, T=_log(rng, 64, 2048 if fp32 else 8192), d_in=_log(rng, 64, 3072, 8),
                    d_out=_log(rng, 64, 3072, 8), C=_log(rng, 64, 1024 if fp32 else 4096, 8),
                    dtype="fp32" if fp32 else "bf16", delta=coin(), route=coin())
    if kind == "ci_mlp":
        return dict(kind=kind, T=_log(rng, 128, 8192), d_in=_log(rng, 64, 3072, rng.choice([1, 8])),
                    hidden=_log(rng, 64, 2048, 8), C=_log(rng, 64, 4096, 8))
    if kind == "faith":
        E = _log(rng, 1, 42)
        return dict(kind=kind, g=rng.choice([1, 2, 4]), E=E, d_in=_log(rng, 64, 768), d_out=_log(rng, 64, 1024),
                    C=_log(rng, 64, 4096 if E < 4 else 768), w_dtype=rng.choice(["bf16", "fp32"]))
    if kind == "kl":
        chunks = rng.choice([1, 2, 3])
        return dict(kind=kind, N=_log(rng, 64, 8192), d=_log(rng, 64, 1024, 8), V=chunks * _log(rng, 300, 16759),
                    chunks=chunks)
    if kind == "moe":
        E = _log(rng, 4, 64)
        T = _log(rng, 128, 8192, 64)
        rps = rng.choice([0, 0, T, 64, 1 if T <= 512 else 0])
        return dict(kind=kind, T=T, d=_log(rng, 64, 640, 8), f=_log(rng, 32, 384, 8), E=E,
                    k=rng.randint(1, min(E, 8)), c=_log(rng, 16, 512, 8), L=rng.randint(1, 4), smooth_l0=coin(),
                    use_delta=coin(0.7), routes=rps == 0 and coin(0.3), rps=rps)
    H = rng.choice([2, 4, 6, 8, 12])
    chunks = rng.choice([1, 3])
    B, T = rng.randint(1, 8), 64 * rng.randint(1, 9)
    rps = rng.choice([0, 0, 0, T, B * T])
    return dict(kind="lm", B=B, T=T, H=H, KV=H // rng.choice([1, 2]), f=64 * _log(rng, 2, 48),
                V=chunks * _log(rng, 300, 16759), L=rng.randint(1, 3), Ca=_log(rng, 64, 1024, 8),
                Cm=_log(rng, 64, 4096, 8), chunks=chunks, smooth_l0=coin(), use_delta=coin(0.7),
                routes=rps == 0 and coin(0.3), rps=rps)


# ---------------------------------------------------------------------------- inputs in hand
class _Draws:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed((seed * 1000003 + 17) % (1 << 31))
        self.key = (0, (seed * 2654435761 + 12345) % (1 << 32))

    def n(self, *shape, scale=1.0, dtype=BF16):
        return (torch.randn(*shape, device="cuda", generator=self.gen) * scale).to(dtype)

    def u(self, *shape, lo=0.0, hi=1.0, dtype=BF16):
        return (torch.rand(*shape, device="cuda", generator=self.gen) * (hi - lo) + lo).to(dtype)

    def ci(self, *shape):
        return self.u(*shape, lo=-0.3, hi=1.3)

    def coin(self, *shape, p=0.7):
        return (torch.rand(*shape, device="cuda", generator=self.gen) < p).to(torch.uint8)


def _dtype(name):
    return torch.float32 if name == "fp32" else BF16


def _imp(case):
    return ImpMin.smooth_l0(**SL0) if case["smooth_l0"] else ImpMin("pnorm", p=2.0, coeff=1.0)


def _inputs(case, seed):
    """Every tensor of a case, from the seed alone (what prepare() and exact() both start from)."""
    r, c, kind = _Draws(seed), case, case["kind"]
    x = {"key": r.key}
    if kind in ("tms", "resid"):
        if kind == "tms":
            target, sites = toys.init_tms(5, 2, 20, generator=r.gen)
            x["x"] = toys.sparse_features(c["B"], 5, 0.05, 0.0, generator=r.gen)
        else:
            target, sites = toys.init_resid_mlp(c["F"], c["D"], c["M"], c["L"], c["C"], generator=r.gen)
            x["x"] = toys.sparse_features(c["B"], c["F"], 0.01, -1.0, generator=r.gen)
        x.update(target=target, sites=sites)
    elif kind == "dense":
        dt, T, di, do, C = _dtype(c["dtype"]), c["T"], c["d_in"], c["d_out"], c["C"]
        x.update(x=r.n(T, di, dtype=dt), W=r.n(do, di, scale=di**-0.5, dtype=dt), V=r.n(di, C, scale=di**-0.5, dtype=dt),
                 U=r.n(C, do, scale=C**-0.5, dtype=dt))
        f32 = dict(dtype=torch.float32)
        x["gate"] = (r.n(C, GATE, scale=2**0.5, **f32), torch.zeros(C, GATE, device="cuda"),
                     r.n(C, GATE, scale=(2 / GATE)**0.5, **f32), torch.zeros(C, device="cuda"))
    elif kind == "site":
        dt, T, di, do, C = _dtype(c["dtype"]), c["T"], c["d_in"], c["d_out"], c["C"]
        x.update(x=r.n(T, di, dtype=dt), W=r.n(do, di, scale=di**-0.5, dtype=dt), V=r.n(di, C, scale=di**-0.5, dtype=dt),
                 U=r.n(C, do, scale=C**-0.5, dtype=dt), mask=r.u(T, C, dtype=dt), g=r.n(T, do, dtype=dt),
                 delta=r.u(T, dtype=dt) if c["delta"] else None, route=r.coin(T) if c["route"] else None)
    elif kind == "ci_mlp":
        mlp = SiteMLP((c["d_in"], c["hidden"], c["C"]), device="cuda", generator=r.gen)
        x.update(mlp=mlp, x=r.n(c["T"], c["d_in"]), g=r.n(c["T"], c["C"]))
    elif kind == "faith":
        g, E, di, do, C = c["g"], c["E"], c["d_in"], c["d_out"], c["C"]
        x.update(W=r.n(g, E, do, di, scale=di**-0.5, dtype=_dtype(c["w_dtype"])),
                 V=r.n(g, E, di, C, scale=di**-0.5, dtype=torch.float32),
                 U=r.n(g, E, C, do, scale=C**-0.5, dtype=torch.float32))
        x["norms"] = [float(v) for v in x["W"].double().square().sum((1, 2, 3)).tolist()]
    elif kind == "kl":
        N, d, V = c["N"], c["d"], c["V"]
        x.update(am=r.n(N, d), ac=r.n(N, d), hm=r.n(V, d, scale=d**-0.5), hc=r.n(V, d, scale=d**-0.5),
                 g=r.u(N, lo=0.5, hi=1.5, dtype=torch.float32) / N)
    elif kind == "moe":
        T, d, f, E, k, cc, L = (c[n] for n in ("T", "d", "f", "E", "k", "c", "L"))
        x["w"] = MoEWeights(
            ln=r.n(L, d, scale=0.1, dtype=torch.float32), router=r.n(L, E, d, scale=d**-0.5),
            Wg=r.n(L, E, d, f, scale=d**-0.5), Wu=r.n(L, E, d, f, scale=d**-0.5), Wd=r.n(L, E, f, d, scale=f**-0.5),
            Vg=r.n(L, E, d, cc, scale=d**-0.5), Ug=r.n(L, E, cc, f, scale=(E * cc)**-0.5),
            Vu=r.n(L, E, d, cc, scale=d**-0.5), Uu=r.n(L, E, cc, f, scale=(E * cc)**-0.5),
            Vd=r.n(L, E, f, cc, scale=f**-0.5), Ud=r.n(L, E, cc, d, scale=(E * cc)**-0.5))
        x.update(x0=r.n(T, d), ci=r.ci(L, 3, T, k, cc), routes=r.coin(L, 3, T) if c["routes"] else None)
        if c["rps"]:
            S = T // c["rps"]
            x["src"] = (r.u(L, 3, S, E, cc, hi=65535.0, dtype=torch.float32)).to(torch.int32).to(torch.uint16)
            x["srcd"] = r.u(L, 3, S, dtype=torch.float32) if c["use_delta"] else None
    elif kind == "lm":
        N, d, L, V, C = c["B"] * c["T"], c["H"] * HEAD, c["L"], c["V"], _lm_C(c)
        dims = _lm_dims(c)
        x["w"] = LMWeights(
            wte=r.n(V, d, scale=d**-0.5), ln1=1 + r.n(L, d, scale=0.1).float(), ln2=1 + r.n(L, d, scale=0.1).float(),
            norm=torch.ones(d, device="cuda"),
            W={n: r.n(L, dims[n][1], dims[n][0], scale=dims[n][0]**-0.5) for n in KINDS},
            V={n: r.n(L, dims[n][0], C[n], scale=dims[n][0]**-0.5) for n in KINDS},
            U={n: r.n(L, C[n], dims[n][1], scale=C[n]**-0.5) for n in KINDS})
        x["tokens"] = torch.randint(0, V, (N,), device="cuda", generator=r.gen, dtype=torch.int32)
        x["ci"] = {n: r.ci(L, N, C[n]) for n in KINDS}
        x["routes"] = r.coin(L, 6, N) if c["routes"] else None
        if c["rps"]:
            S = N // c["rps"]
            x["src"] = {n: r.u(L, S, C[n], dtype=torch.float32) for n in KINDS}
            x["srcd"] = r.u(L, 6, S, dtype=torch.float32) if c["use_delta"] else None
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return x


def _lm_C(c):
    return {n: c["Cm"] if n in ("c_fc", "down_proj") else c["Ca"] for n in KINDS}


def _lm_dims(c):
    return {n: site_dims(n, c["H"] * HEAD, c["H"], c["KV"], c["f"]) for n in KINDS}


def prepare(case, seed):
    x, c, kind = _inputs(case, seed), case, case["kind"]
    x["case"] = c
    if kind == "tms":
        x["step"] = toys.TMSFusedStep(x["target"], x["sites"], p=c["p"], use_delta=c["use_delta"])
    elif kind == "resid":
        x["step"] = toys.ResidMLPFusedStep(x["target"], x["sites"], p=c["p"])
    elif kind == "dense":
        x["step"] = DenseSiteStep(c["T"], c["d_in"], c["d_out"], c["C"], dtype=_dtype(c["dtype"]), imp_min=_imp(c),
                                  use_delta=c["use_delta"])
        x["keys"] = x["step"].site_keys(x["key"], 0)
    elif kind == "site":
        x["leaves"] = [x[n].requires_grad_(True) for n in ("x", "V", "U", "mask")]
    elif kind == "faith":
        x["loss"] = FaithfulnessLoss({"gate": None}, {"gate": x["norms"]}, c["g"])
        x["leaves"] = [x[n].requires_grad_(True) for n in ("V", "U")]
    elif kind == "kl":
        x["am"].requires_grad_(True)
    elif kind == "moe":
        x["step"] = MoEStackStep(c["T"], c["d"], c["f"], c["E"], c["k"], c["c"], c["L"], imp_min=_imp(c),
                                 use_delta=c["use_delta"], rows_per_source=c["rps"] or None)
    elif kind == "lm":
        x["step"] = LMStackStep(c["B"], c["T"], c["H"] * HEAD, c["H"], c["KV"], c["f"], c["V"], c["L"], _lm_C(c),
                                imp_min=_imp(c), use_delta=c["use_delta"], n_kl_chunks=c["chunks"],
                                routed=c["routes"], rows_per_source=c["rps"] or None)
    return x


# ---------------------------------------------------------------------------------- one pass
def _toy_outputs(res, sites):
    grads = [[p.grad for p in s.parameters()] for s in sites]
    return {"losses": [res["loss"], res["recon"], res["imp"]], "grads": grads}


def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind in ("tms", "resid"):
        res = s["step"].step(s["x"], s["key"])
        out = _toy_outputs(res, s["sites"])
        return dict(out, out=res["out"]) if kind == "resid" else out
    if kind == "dense":
        g = s["step"].step(s["x"], s["W"], s["V"], s["U"], s["gate"], *s["keys"])
        return {"losses": g.losses, "dV": g.dV, "dU": g.dU, "gate": [g.dw_in, g.db_in, g.dw_out, g.db_out]}
    if kind == "site":
        y = site_forward(s["x"], SiteWeights(s["W"], s["V"], s["U"]), s["mask"], s["delta"], s["route"])
        return [y.output, y.component_activation, *torch.autograd.grad(y.output, s["leaves"], s["g"])]
    if kind == "ci_mlp":
        y = s["mlp"](s["x"])
        return [y, *torch.autograd.grad(y, list(s["mlp"].parameters()), s["g"])]
    if kind == "faith":
        loss = s["loss"]({"gate": (s["W"], s["V"], s["U"])})
        return [loss, *torch.autograd.grad(loss, s["leaves"])]
    if kind == "kl":
        kl = streamed_position_kl(s["am"], s["hm"], s["ac"], s["hc"], c["chunks"])
        return [kl, *torch.autograd.grad(kl, [s["am"]], s["g"])]
    st = s["step"]
    if kind == "moe":
        out = {"losses": st.losses, "dV": st.dV, "dU": st.dU, "d_ci": st.d_ci_pre, "top_idx": st.top_idx}
        args = (s["x0"], s["w"], s["ci"])
    else:
        out = {"losses": st.losses, "dV": st.dV, "dU": st.dU, "d_ci": st.d_ci_pre}
        args = (s["tokens"], s["w"], s["ci"])
    if not c["rps"]:
        st.step(*args, s["key"], routes=s["routes"])
        return out
    st.step_sources(*args, s["src"], s["srcd"], want_weight_grads=False)
    st.step_sources(*args, s["src"], s["srcd"], reuse_clean=True)
    out["d_src"] = st.d_src
    if s["srcd"] is not None:
        out["d_src_delta"] = st.d_src_delta
    return out


# ---------------------------------------------------------------------------- work, tolerance
def work(case):
    """Inputs read once and outputs written once; products by the reference's rule (forward,
    the input gradients that are needed, the factor gradients; frozen products included)."""
    c, kind = case, case["kind"]
    if kind in ("tms", "resid"):
        B, C = c["B"], 20 if kind == "tms" else c["C"]
        if kind == "tms":
            dims, clean, io = [(5, 2), (2, 5)], 2 * B * (5 * 2 + 2 * 5), 4 * B * 5
        else:
            F, D, M = c["F"], c["D"], c["M"]
            dims = [(D, M), (M, D)] * c["L"]
            clean, io = 2 * B * (3 * F * D + 2 * c["L"] * D * M) + 2 * B * F * D, 4 * (B * F * 2 + 2 * F * D)
        flops = clean
        nbytes = io
        for i, (di, do) in enumerate(dims):
            inp, out = 2 * B * di * C, 2 * B * C * do
            # the gate reads the clean input's activations, the mask the masked input's
            flops += inp + (inp if i else 0) + out + 2 * out + inp * (2 if i else 1) + (inp if i else 0)
            flops += 3 * 4 * GATE * B * C
            nbytes += 4 * (di * do + 2 * (di * C + C * do + C * (3 * GATE + 1)))
        return {"bytes": nbytes, "flops": flops}
    if kind in ("dense", "site"):
        T, di, do, C = c["T"], c["d_in"], c["d_out"], c["C"]
        es = 4 if c["dtype"] == "fp32" else 2
        i, o, f = 2 * T * di * C, 2 * T * C * do, 2 * T * di * do
        if kind == "dense":
            nbytes = es * (T * di + di * do + di * C + C * do) + 4 * (di * C + C * do + 2 * C * (3 * GATE + 1))
            return {"bytes": nbytes, "flops": f + 2 * i + 3 * o + 3 * 4 * GATE * T * C}
        frozen = c["delta"] or c["route"]
        nbytes = es * (2 * T * di + 2 * T * do + di * do * frozen + 2 * (di * C + C * do) + 3 * T * C)
        return {"bytes": nbytes, "flops": 3 * i + 3 * o + 2 * f * frozen}
    if kind == "ci_mlp":
        T, di, h, C = c["T"], c["d_in"], c["hidden"], c["C"]
        P = di * h + h * C + h + C
        return {"bytes": 2 * T * (di + 2 * C) + 8 * P, "flops": 2 * T * (2 * di * h + 3 * h * C)}
    if kind == "faith":
        n, di, do, C = c["g"] * c["E"], c["d_in"], c["d_out"], c["C"]
        es = 4 if c["w_dtype"] == "fp32" else 2
        return {"bytes": n * (es * di * do + 8 * C * (di + do)), "flops": 6 * n * di * do * C}
    if kind == "kl":
        N, d, V = c["N"], c["d"], c["V"]
        return {"bytes": 2 * (2 * N * d + 2 * V * d) + 8 * N + 2 * N * d, "flops": 2 * N * d * V * 3}
    calls = [True] if not c["rps"] else [False, True]  # with the factor gradients or without
    if kind == "moe":
        T, d, f, E, k, cc, L = (c[n] for n in ("T", "d", "f", "E", "k", "c", "L"))
        J, frozen = T * k, c["use_delta"] or c["routes"]
        i, o, fr = 2 * J * d * cc, 2 * J * cc * f, 2 * J * d * f * frozen  # gate and up; the down site mirrors them
        flops = L * 3 * 2 * J * d * f  # the clean pass, formed once
        for grads in calls:
            for layer in range(L):
                flops += 3 * (i + o + fr) + 2 * o + i + (2 * (i + fr) if layer else 0) + (o + fr)
                flops += 3 * (i + o) * grads
        nfac, nw = L * E * cc * 3 * (d + f), L * E * 3 * d * f
        nbytes = 2 * (nfac + nw + T * d + L * E * d) + 4 * nfac + 2 * 2 * L * 3 * J * cc
        if c["rps"]:
            nbytes += (2 + 4) * L * 3 * (T // c["rps"]) * E * cc
        return {"bytes": nbytes, "flops": flops}
    N, d, C, V, L = c["B"] * c["T"], c["H"] * HEAD, _lm_C(c), c["V"], c["L"]
    frozen = c["use_delta"] or c["routes"]
    attn = 2 * N * c["T"] // 2 * d  # one causal product over all heads
    flops, nbytes = 0, 0
    for n, (di, do) in _lm_dims(c).items():
        nbytes += L * (2 * di * do + 6 * C[n] * (di + do) + 4 * N * C[n])
        flops += L * 2 * N * di * do  # the frozen pass
        for layer in range(L):
            i, o, fr = 2 * N * di * C[n], 2 * N * C[n] * do, 2 * N * di * do * frozen
            need_x = layer > 0 or n not in ("q_proj", "k_proj", "v_proj")
            for grads in calls:
                flops += i + o + fr + o + (i + fr) * need_x + (i + o) * grads
        if c["rps"]:
            nbytes += 8 * L * (N // c["rps"]) * C[n]
    flops += L * attn * (2 + 7 * len(calls)) + 2 * N * d * V * (1 + 2 * len(calls))
    return {"bytes": nbytes + 2 * V * d, "flops": flops}


def tolerance(case):
    """About four times the distance from exact(): measured 2e-8 to 6e-7 in fp32, 1e-3 to 3e-3
    where a pass stores a few tensors in bf16, and 4e-3 to 2e-2 down a stack of layers."""
    kind = case["kind"]
    if kind in ("tms", "resid", "faith") or case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind in ("moe", "lm"):
        return {"rel": 3e-2, "max": 0.9, "differ": 1e-3}
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------------- the same in 64 bits
M32 = 0xFFFFFFFF
ROTATIONS = (13, 15, 26, 6, 17, 29, 16, 24)


def _threefry(key, x0, x1):
    """Threefry-2x32 with 20 rounds (Salmon et al. 2011), on Python integers or int64 tensors."""
    ks = (key[0], key[1], key[0] ^ key[1] ^ 0x1BD11BDA)
    x0, x1 = (x0 + ks[0]) & M32, (x1 + ks[1]) & M32
    for block in range(5):
        for r in ROTATIONS[4 * (block & 1):4 * (block & 1) + 4]:
            x0 = (x0 + x1) & M32
            x1 = (((x1 << r) | (x1 >> (32 - r))) & M32) ^ x0
        x0, x1 = (x0 + ks[(block + 1) % 3]) & M32, (x1 + ks[(block + 2) % 3] + block + 1) & M32
    return x0, x1


def _fold(key, *data):
    for d in data:
        key = _threefry(key, 0, d)
    return key


def _uniform(key, shape, bf16):
    """A draw of jax.random.uniform: 7 of 8 bits in bf16, 23 of 32 in fp32, counter i for element i."""
    i = torch.arange(math.prod(shape), device="cuda", dtype=torch.int64)
    y0, y1 = _threefry(key, 0, i)
    bits = y0 ^ y1
    u = ((bits & 0xFF) >> 1).to(F64) * 2.0**-7 if bf16 else (bits >> 9).to(F64) * 2.0**-23
    return u.reshape(shape)


class _Lower(torch.autograd.Function):
    """clip(x, 0, 1); backward: the gradient on (0, 1], 0.01 of a negative one at or below 0."""

    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return x.clamp(0.0, 1.0)

    @staticmethod
    def backward(ctx, g):
        (x,) = ctx.saved_tensors
        return torch.where(x <= 0, 0.01 * g.clamp(max=0.0), torch.where(x <= 1, g, 0.0 * g))


class _Upper(torch.autograd.Function):
    """clip(x, 0, 1), leaking with slope 0.01 above 1; half the gradient at the two ties."""

    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return torch.where(x > 1, 1 + 0.01 * (x - 1), x.clamp(0.0, 1.0))

    @staticmethod
    def backward(ctx, g):
        (x,) = ctx.saved_tensors
        inner = torch.where((x == 0) | (x == 1), 0.5, ((x > 0) & (x < 1)).to(g.dtype))
        return g * torch.where(x > 1, 0.01, inner)


def _activity(case, up, rows, scatter=None):
    """(activity, frequency penalty) of one site's upper CI [rows, C], summed over components;
    `scatter(psi)` adds selected values up into their expert's components."""
    if not case.get("smooth_l0"):
        return up.pow(case.get("p", 2.0)).sum() / rows, 0.0
    psi = up**2 / (up**2 + SL0["gamma"]**2)
    f = (scatter(psi) if scatter else psi.sum(0)) / rows
    return f.sum(), (f * torch.log2(1.0 + SL0["reference_datapoint_count"] * f)).sum()


def _total(case, recon, act, freq):
    coeff, fc = (SL0["coeff"], SL0["frequency_coeff"]) if case.get("smooth_l0") else (1.0, 0.0)
    total = recon + coeff * act + fc * freq
    freq = freq if torch.is_tensor(freq) else recon * 0
    return total, torch.stack([total, recon, act, freq]).detach()


def _leaf(t):
    return t.detach().to(F64).requires_grad_(True)


def _gate(h, w_in, b_in, w_out, b_out):
    g = b_out + 0.0 * h
    for j in range(GATE):
        g = g + w_out[:, j] * torch.nn.functional.gelu(h * w_in[:, j] + b_in[:, j])
    return g


def _exact_toy(c, x):
    tms = c["kind"] == "tms"
    t, sites = x["target"], x["sites"]
    P = [[_leaf(p) for p in s.parameters()] for s in sites]
    W = [s.W.to(F64) for s in sites]
    batch, n = x["x"].to(F64), len(sites)
    mk, dk = _threefry(x["key"], 0, 0), _threefry(x["key"], 0, 1)

    def forward(site):
        if tms:
            return torch.relu(site(1, site(0, batch)) + t.b2.to(F64))
        r = batch @ t.W_E.to(F64)
        for i in range(n // 2):
            r = r + site(2 * i + 1, torch.relu(site(2 * i, r)))
        return r @ t.W_U.to(F64)

    seen = []

    def frozen(i, a):
        seen.append(a)
        return a @ W[i].T

    clean = forward(frozen)
    coef, delta, act = [], [], 0.0
    for i, (V, U, *gate) in enumerate(P):
        g = _gate(seen[i] @ V, *gate)
        lo = _Lower.apply(g)
        m = lo + (1 - lo) * _uniform(_fold(mk, i), g.shape, False)
        d = _uniform(_fold(dk, i), g.shape[:1], False)[:, None] if c.get("use_delta") else None
        coef.append(m if d is None else m - d)
        delta.append(d)
        act = act + _activity(c, _Upper.apply(g), g.shape[0])[0]

    def masked(i, a):
        y = ((a @ P[i][0]) * coef[i]) @ P[i][1]
        return y if delta[i] is None else y + delta[i] * (a @ W[i].T)

    out = forward(masked)
    recon = (out - clean).square().mean()
    loss = recon + act
    flat = torch.autograd.grad(loss, [p for q in P for p in q])
    grads = [list(flat[6 * i:6 * i + 6]) for i in range(n)]
    res = {"losses": [loss.detach(), recon.detach(), act.detach()], "grads": grads}
    return res if tms else dict(res, out=out.detach())


def _exact_dense(c, x):
    bf = c["dtype"] == "bf16"
    X, W, V, U = x["x"].to(F64), x["W"].to(F64), _leaf(x["V"]), _leaf(x["U"])
    gate = [_leaf(p) for p in x["gate"]]
    keys = [_fold(_threefry(x["key"], 0, i), 0) for i in range(2)]
    target = X @ W.T
    h = X @ V
    if bf:  # the gate and the squashings' branches read the stored activation
        h = h + (h.detach().to(BF16).to(F64) - h.detach())
    g = _gate(h, *gate)
    lo = _Lower.apply(g)
    m = lo + (1 - lo) * _uniform(keys[0], g.shape, bf)
    d = _uniform(keys[1], g.shape[:1], bf)[:, None] if c["use_delta"] else 0.0
    y = (h * (m - d)) @ U + d * target
    recon = (y - target).square().mean()
    loss, losses = _total(c, recon, *_activity(c, _Upper.apply(g), g.shape[0]))
    dV, dU, *dg = torch.autograd.grad(loss, [V, U, *gate])
    return {"losses": losses, "dV": dV, "dU": dU, "gate": dg}


def _exact_site(c, x):
    leaves = [_leaf(x[n]) for n in ("x", "V", "U", "mask")]
    X, V, U, m = leaves
    d = x["delta"].to(F64)[:, None] if c["delta"] else 0.0
    xV = X @ V
    y = (xV * (m - d)) @ U
    if c["delta"] or c["route"]:
        target = X @ x["W"].to(F64).T
        y = y + d * target
        if c["route"]:
            y = torch.where(x["route"].bool()[:, None], y, target)
    return [y.detach(), xV.detach(), *torch.autograd.grad(y, leaves, x["g"].to(F64))]


def _exact_ci_mlp(c, x):
    # the engine computes in bf16 from fp32 masters cast once
    P = [_leaf(p.detach().to(BF16)) for p in x["mlp"].parameters()]
    (w0, w1), (b0, b1) = P[:2], P[2:]
    y = torch.nn.functional.gelu(x["x"].to(F64) @ w0 + b0) @ w1 + b1
    return [y.detach(), *torch.autograd.grad(y, P, x["g"].to(F64))]


def _exact_faith(c, x):
    V, U = _leaf(x["V"]), _leaf(x["U"])
    W = x["W"].to(F64)
    err = (W - (V @ U).transpose(-1, -2)).square().sum((1, 2, 3))
    loss = (err / torch.tensor(x["norms"], device="cuda", dtype=F64)).sum() / c["g"]
    return [loss.detach(), *torch.autograd.grad(loss, [V, U])]


def _kl(masked, clean):
    log_q, log_p = torch.log_softmax(masked, -1), torch.log_softmax(clean, -1)
    return (log_p.exp() * (log_p - log_q)).sum(-1)


def _exact_kl(c, x):
    am = _leaf(x["am"])
    kl = _kl(am @ x["hm"].to(F64).T, x["ac"].to(F64) @ x["hc"].to(F64).T)
    return [kl.detach(), *torch.autograd.grad(kl, [am], x["g"].to(F64))]


def _site_masks(c, key, ci, kind, layer, rows, u=None, d=None):
    """(coefficient, delta [rows, 1], upper) of a stack's site: drawn, or from source rows u, d."""
    lo = _Lower.apply(ci)
    if u is None:
        u = _uniform(_fold(_threefry(key, 0, 0), kind, layer), ci.shape, True)
        d = _uniform(_fold(_threefry(key, 0, 1), kind, layer), (rows,), True) if c["use_delta"] else None
    return lo + (1 - lo) * u, 0.0 if d is None else d, _Upper.apply(ci)


class _Stored(torch.autograd.Function):
    """A bf16 read of a wider stored value (straight gradient)."""

    @staticmethod
    def forward(ctx, x):
        return x.to(BF16).to(F64)

    @staticmethod
    def backward(ctx, g):
        return g


def _exact_moe(c, x):
    T, E, k, L, w, cc = c["T"], c["E"], c["k"], c["L"], x["w"], c["c"]
    bf = lambda t: t.to(BF16).to(F64)  # noqa: E731
    norm = lambda r, ln: r * torch.rsqrt(r.square().mean(-1, keepdim=True) + 1e-6) * (1.0 + ln)  # noqa: E731
    silu = torch.nn.functional.silu

    def jobs_of(idx):
        flat = idx.reshape(-1)
        order = torch.sort(flat, stable=True)[1]
        return order, order.argsort(), torch.bincount(flat, minlength=E).tolist()

    def gmm(lhs, rhs, sizes):
        return torch.cat([a @ rhs[e] for e, a in enumerate(lhs.split(sizes))])

    # the frozen pass: which experts are taken is decided by bf16 logits of bf16 activations,
    # so it rounds what the path stores
    rc, tops = x["x0"].to(F64), []
    for l in range(L):
        h2 = bf(norm(rc, w.ln[l].to(F64)))
        probs = torch.softmax(bf(h2 @ w.router[l].to(F64).T), -1)
        idx = torch.sort(-probs, dim=-1, stable=True)[1][:, :k]
        order, inv, sizes = jobs_of(idx)
        xj = h2.index_select(0, order // k)
        din = bf(silu(bf(gmm(xj, w.Wg[l].to(F64), sizes))) * bf(gmm(xj, w.Wu[l].to(F64), sizes)))
        down = bf(gmm(din, w.Wd[l].to(F64), sizes))
        mix = probs.gather(1, idx)
        mix = mix / mix.sum(-1, keepdim=True)
        rc = bf(rc + bf((down[inv].reshape(T, k, -1) * mix[..., None]).sum(1)))
        tops.append(idx)
    V = {s: _leaf(getattr(w, "V" + s[0])) for s in SITE_NAMES}
    U = {s: _leaf(getattr(w, "U" + s[0])) for s in SITE_NAMES}
    ci = _leaf(x["ci"])
    wrt = [V[s] for s in SITE_NAMES] + [U[s] for s in SITE_NAMES] + [ci]
    if c["rps"]:
        doc = torch.arange(T, device="cuda") // c["rps"]
        # tables are read in the CI's dtype
        src = _leaf(x["src"].to(torch.int32).to(F64) / 65535.0)
        wrt.append(src)
        srcd = None
        if x["srcd"] is not None:
            srcd = _leaf(x["srcd"])
            wrt.append(srcd)
    r, act, freq = x["x0"].to(F64), 0.0, 0.0
    for l in range(L):
        h2, idx = norm(r, w.ln[l].to(F64)), tops[l]
        mix = torch.softmax(h2 @ w.router[l].to(F64).T, -1).gather(1, idx)
        mix = mix / mix.sum(-1, keepdim=True)
        order, inv, sizes = jobs_of(idx)
        tok = order // k
        xj = h2.index_select(0, tok)

        def site(si, a):
            s = SITE_NAMES[si]
            u = d = None
            if c["rps"]:
                at = (doc[:, None] * E + idx).reshape(-1)
                u = _Stored.apply(src[l, si].reshape(-1, cc).index_select(0, at)).reshape(T, k, cc)
                d = None if srcd is None else _Stored.apply(srcd[l, si].index_select(0, doc))
            m, d, up = _site_masks(c, x["key"], ci[l, si].reshape(T, k * cc), 11 + si, l, T,
                                   None if u is None else u.reshape(T, k * cc), d)
            m = m.reshape(T * k, cc).index_select(0, order)
            dj = d.index_select(0, tok)[:, None] if torch.is_tensor(d) else 0.0
            out = gmm(gmm(a, V[s][l], sizes) * (m - dj), U[s][l], sizes)
            if torch.is_tensor(dj) or c["routes"]:
                frozen = gmm(a, getattr(w, "W" + s[0])[l].to(F64), sizes)
                out = out + dj * frozen
                if c["routes"]:
                    out = torch.where(x["routes"][l, si].bool()[tok][:, None], out, frozen)
            scatter = lambda p: torch.zeros(E, cc, device="cuda", dtype=F64).index_add(  # noqa: E731
                0, idx.reshape(-1), p.reshape(T * k, cc))
            return out, _activity(c, up, T, scatter)

        (g, a0), (u_, a1) = site(0, xj), site(1, xj)
        down, a2 = site(2, silu(g) * u_ * mix.reshape(-1).index_select(0, order)[:, None])
        act, freq = act + a0[0] + a1[0] + a2[0], freq + a0[1] + a1[1] + a2[1]
        r = r + down.index_select(0, inv).reshape(T, k, -1).sum(1)
    loss, losses = _total(c, (r - rc).square().mean(), act, freq)
    got = torch.autograd.grad(loss, wrt)
    out = {"losses": losses, "dV": dict(zip(SITE_NAMES, got[:3])), "dU": dict(zip(SITE_NAMES, got[3:6])),
           "d_ci": got[6], "top_idx": None}
    if c["rps"]:
        out["d_src"] = got[7]
        if srcd is not None:
            out["d_src_delta"] = got[8]
    return out


def _exact_lm(c, x):
    B, T, H, KV, L, w = c["B"], c["T"], c["H"], c["KV"], c["L"], x["w"]
    N, C, d = B * T, _lm_C(c), H * HEAD
    norm = lambda r, g: g.to(F64) * r * torch.rsqrt(r.square().mean(-1, keepdim=True) + 1e-6)  # noqa: E731
    inv_freq = 10000.0 ** (-torch.arange(0, HEAD, 2, device="cuda", dtype=F64) / HEAD)
    ang = torch.arange(T, device="cuda", dtype=F64)[:, None] * inv_freq
    ang = torch.cat([ang, ang], -1)
    cos, sin = (f().to(BF16).to(F64) for f in (ang.cos, ang.sin))  # the tables are bf16
    causal = torch.ones(T, T, device="cuda", dtype=torch.bool).tril()
    rot = lambda t: torch.cat([-t[..., HEAD // 2:], t[..., :HEAD // 2]], -1)  # noqa: E731

    def attention(q, k, v):
        q, k, v = (t.reshape(B, T, -1, HEAD).transpose(1, 2).contiguous() for t in (q, k, v))
        q, k = q * cos + rot(q) * sin, k * cos + rot(k) * sin
        k, v = (t.repeat_interleave(H // KV, 1) for t in (k, v))
        s = (q @ k.transpose(-1, -2).contiguous()) * HEAD**-0.5
        a = torch.softmax(s.masked_fill(~causal, float("-inf")), -1) @ v
        return a.transpose(1, 2).reshape(N, d)

    def forward(site):
        r = w.wte.to(F64)[x["tokens"].long()]
        for l in range(L):
            h = norm(r, w.ln1[l])
            a = attention(*(site(l, n, h) for n in ("q_proj", "k_proj", "v_proj")))
            r = r + site(l, "o_proj", a)
            fc = site(l, "c_fc", norm(r, w.ln2[l]))
            r = r + site(l, "down_proj", torch.nn.functional.gelu(fc, approximate="tanh"))
        return norm(r, w.norm) @ w.wte.to(F64).T

    with torch.no_grad():
        clean = forward(lambda l, n, a: a @ w.W[n][l].to(F64).T)
    V, U, ci = ({n: _leaf(t[n]) for n in KINDS} for t in (w.V, w.U, x["ci"]))
    wrt = [t[n] for t in (V, U, ci) for n in KINDS]
    if c["rps"]:
        doc = torch.arange(N, device="cuda") // c["rps"]
        src = {n: _leaf(x["src"][n]) for n in KINDS}
        wrt += [src[n] for n in KINDS]
        srcd = None
        if x["srcd"] is not None:
            srcd = _leaf(x["srcd"])
            wrt.append(srcd)
    sums = [0.0, 0.0]

    def masked(l, n, a):
        ki, u, dl = KINDS.index(n), None, None
        if c["rps"]:  # tables are read in the CI's dtype
            u = _Stored.apply(src[n][l].index_select(0, doc))
            dl = None if srcd is None else _Stored.apply(srcd[l, ki].index_select(0, doc))
        m, dl, up = _site_masks(c, x["key"], ci[n][l], ki, l, N, u, dl)
        dl = dl[:, None] if torch.is_tensor(dl) else dl
        a0, a1 = _activity(c, up, N)
        sums[0], sums[1] = sums[0] + a0, sums[1] + a1
        y = ((a @ V[n][l]) * (m - dl)) @ U[n][l]
        if torch.is_tensor(dl) or c["routes"]:
            frozen = a @ w.W[n][l].to(F64).T
            y = y + dl * frozen
            if c["routes"]:
                y = torch.where(x["routes"][l, ki].bool()[:, None], y, frozen)
        return y

    loss, losses = _total(c, _kl(forward(masked), clean).mean(), *sums)
    got = torch.autograd.grad(loss, wrt)
    out = {"losses": losses}
    for i, key in enumerate(("dV", "dU", "d_ci")):
        out[key] = dict(zip(KINDS, got[6 * i:6 * i + 6]))
    if c["rps"]:
        out["d_src"] = dict(zip(KINDS, got[18:24]))
        if srcd is not None:
            out["d_src_delta"] = got[24]
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    return {"tms": _exact_toy, "resid": _exact_toy, "dense": _exact_dense, "site": _exact_site,
            "ci_mlp": _exact_ci_mlp, "faith": _exact_faith, "kl": _exact_kl, "moe": _exact_moe,
            "lm": _exact_lm}[case["kind"]](case, x)
