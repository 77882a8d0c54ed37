"""Performance cases of the FP8 mixture-of-experts path and its dense GEMMs.

Each case is one call, or the short chain of calls, that a user's program makes
per step on tensors already on the GPU:

  kind "moe"    an MoE feed-forward layer: hkmoe.MoELayer (per-tensor or
                128x128 / 1x128 block scales) or hkmoe.MoELayerMX (1x32 e8m0).
                With ``from_f32`` the step starts from fp32 hidden states and
                quantises them first, as a layer behind a norm does.
  kind "gemm"   hkmoe.gemm_fp8, per-tensor scales, bf16 or fp32 output
  kind "mx"     an MX linear layer: quantise fp32 activations, pack their
                exponents, gemm_mx against packed weights
  kind "quant"  one quantiser over a tensor

Inputs are made here with plain torch (weights N(0, 1/fan_in), activations
N(0, 1), quantised by the formats' rules), so that ``exact`` can evaluate the
same inputs in 64 bits.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "distributed-hipkittens_amd"))
import hkmoe  # noqa: E402

F8 = torch.float8_e4m3fn
DEV = "cuda"

# Expert shapes (experts, top-k, hidden, inter): the benchmark's decode,
# prefill and 8-expert layers, and two generic layers with uneven K-step counts
# (inter = 11 * 128 and 9 * 128).
SHAPES = {
    "e128": dict(E=128, k=8, H=4096, I=1536),
    "e256": dict(E=256, k=8, H=7168, I=2048),
    "e8": dict(E=8, k=2, H=4096, I=14336),
    "e64": dict(E=64, k=6, H=2048, I=1408),
    "e16": dict(E=16, k=4, H=2560, I=1152),
}


def _moe(shape, T, scales, skew=False, from_f32=False, packed=True):
    return dict(kind="moe", T=T, scales=scales, skew=skew, from_f32=from_f32, packed=packed, **SHAPES[shape])


def listed():
    return [
        # one token of one sequence: interactive decoding, all launches and latency
        dict(name="moe_block_decode_1", **_moe("e128", 1, "block", from_f32=True)),
        # the benchmark's decode batch: weight streaming
        dict(name="moe_block_decode_64", **_moe("e128", 64, "block")),
        # a prefill chunk of odd length beside nothing else: experts of few rows
        dict(name="moe_block_chunk_777", **_moe("e256", 777, "block", skew=True, from_f32=True)),
        # the benchmark's flagship layer: large-batch prefill with skewed routing
        dict(name="moe_block_prefill_8192", **_moe("e256", 8192, "block", skew=True)),
        # a small decode batch through 8 large experts, per-tensor scales
        dict(name="moe_tensor_decode_29", **_moe("e8", 29, "tensor", from_f32=True)),
        # the benchmark's 8-expert prefill, from fp32 hidden states
        dict(name="moe_tensor_prefill_4096", **_moe("e8", 4096, "tensor", from_f32=True)),
        # MX checkpoints: a decode batch and a ragged prefill
        dict(name="moe_mx_decode_48", **_moe("e128", 48, "mx", from_f32=True)),
        dict(name="moe_mx_prefill_3001", **_moe("e256", 3001, "mx", skew=True)),
        # dense projections: the benchmark's square and tensor-parallel shapes,
        # and that tensor-parallel weight with a decode batch
        dict(name="gemm_2048", kind="gemm", M=2048, N=2048, K=2048, out="bf16"),
        dict(name="gemm_8192x8192x2048", kind="gemm", M=8192, N=8192, K=2048, out="bf16"),
        dict(name="gemm_17x8192x2048", kind="gemm", M=17, N=8192, K=2048, out="bf16"),
        # the MX GEMM harness's shape as a linear layer, fp32 out
        dict(name="mx_linear_8192", kind="mx", M=8192, N=8192, K=8192, out="f32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dense(rng):
    """M, N, K of a dense product of at most 8192^3, N in 256s and K in 128s."""
    while True:
        m, n, k = _log_int(rng, 1, 16384), 256 * _log_int(rng, 1, 64), 128 * _log_int(rng, 1, 128)
        if m * n * k <= 8192 ** 3:
            return m, n, k


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "gemm", "gemm", "mx", "quant"])
    if kind == "moe":
        shape = rng.choice(sorted(SHAPES))
        # the e8 layer's rows carry 8192 tokens' work of the e256 layer at T = 4096
        T = _log_int(rng, 1, 4096 if shape == "e8" else 8192)
        return _moe(shape, T, rng.choice(["block", "tensor", "mx"]), skew=rng.random() < 0.5,
                    from_f32=rng.random() < 0.5, packed=rng.random() < 0.8)
    if kind in ("gemm", "mx"):
        m, n, k = _dense(rng)
        return dict(kind=kind, M=m, N=n, K=k, out=rng.choice(["bf16", "f32"]))
    what = rng.choice(["group", "tensor", "mx", "block"])
    rows = 128 * _log_int(rng, 1, 128) if what == "block" else _log_int(rng, 1, 16384)
    return dict(kind="quant", what=what, rows=rows, cols=128 * _log_int(rng, 1, 128))


# ---------------------------------------------------------------------------
# inputs: plain torch
# ---------------------------------------------------------------------------
def _scale(amax):
    # a tensor divisor: torch multiplies by the reciprocal of a scalar one
    return torch.where(amax > 0, (amax / torch.full_like(amax, 448.0)).clamp_min(2.0 ** -126), torch.ones_like(amax))


def _q_tensor(x):
    s = _scale(x.abs().amax().reshape(1))
    return (x / s).to(F8), s


def _q_group(x):
    v = x.view(x.shape[0], -1, 128)
    s = _scale(v.abs().amax(2))
    return (v / s[..., None]).to(F8).view(x.shape), s


def _q_block(w):
    """[B, R, C] -> e4m3, scales [B, R/128, C/128]."""
    v = w.view(w.shape[0], w.shape[1] // 128, 128, w.shape[2] // 128, 128)
    s = _scale(v.abs().amax((2, 4)))
    return (v / s[:, :, None, :, None]).to(F8).view(w.shape), s


def _q_mx(x):
    """[..., C] -> e4m3, e8m0 bytes [..., C/32]: 2^floor(log2 amax) per 32 columns."""
    v = x.view(*x.shape[:-1], -1, 32)
    amax = v.abs().amax(-1)
    e = torch.where(amax > 0, torch.frexp(amax)[1] - 1 + 127, torch.zeros((), dtype=torch.int32, device=x.device))
    e = e.clamp(0, 254)
    q = torch.ldexp(v, (127 - e)[..., None]).to(F8).view(x.shape)
    return q, e.to(torch.uint8)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _weights(g, E, N, K, scales):
    """E expert weights [N, K] with their scales, a few experts at a time."""
    q = torch.empty((E, N, K), dtype=F8, device=DEV)
    shape = {"tensor": (E,), "block": (E, N // 128, K // 128), "mx": (E, N, K // 32)}[scales]
    s = torch.empty(shape, dtype=torch.uint8 if scales == "mx" else torch.float32, device=DEV)
    step = max(1, (1 << 27) // (N * K))
    for e0 in range(0, E, step):
        e1 = min(E, e0 + step)
        w = _randn(g, e1 - e0, N, K) * K ** -0.5
        if scales == "tensor":
            for e in range(e0, e1):
                q[e], s[e:e + 1] = _q_tensor(w[e - e0])
        else:
            q[e0:e1], s[e0:e1] = (_q_block if scales == "block" else _q_mx)(w)
    return q, s


def _logits(g, case, device=DEV):
    """Router logits N(0, 1), with ``skew`` a Zipf(1.1) bias over the experts."""
    x = torch.randn((case["T"], case["E"]), generator=g, device=device, dtype=torch.float32)
    if case["skew"]:
        rank = torch.randperm(case["E"], generator=g, device=device).float() + 1.0
        x = x - 1.1 * torch.log(rank)
    return x


def _moe_inputs(case, seed):
    g = _gen(seed)
    T, E, H, I = case["T"], case["E"], case["H"], case["I"]
    d = dict(x=_randn(g, T, H), logits=_logits(g, case))
    d["x_q"], d["x_s"] = {"tensor": _q_tensor, "block": _q_group, "mx": _q_mx}[case["scales"]](d["x"])
    d["w13"], d["s13"] = _weights(g, E, 2 * I, H, case["scales"])
    d["w2"], d["s2"] = _weights(g, E, H, I, case["scales"])
    return d


def _gemm_inputs(case, seed):
    g = _gen(seed)
    d = {}
    d["a"], d["sa"] = _q_tensor(_randn(g, case["M"], case["K"]))
    d["b"], d["sb"] = _q_tensor(_randn(g, case["N"], case["K"]) * case["K"] ** -0.5)
    return d


def _mx_inputs(case, seed):
    g = _gen(seed)
    d = dict(x=_randn(g, case["M"], case["K"]))
    d["w"], d["sw"] = _q_mx(_randn(g, case["N"], case["K"]) * case["K"] ** -0.5)
    return d


def _quant_input(case, seed):
    return _randn(_gen(seed), case["rows"], case["cols"])


QUANT = {"group": hkmoe.quant_group, "tensor": hkmoe.quant_tensor, "mx": hkmoe.quant_mx, "block": hkmoe.quant_block}


# ---------------------------------------------------------------------------
# a user's step
# ---------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "moe":
        d = _moe_inputs(case, seed)
        cls = hkmoe.MoELayerMX if case["scales"] == "mx" else hkmoe.MoELayer
        layer = cls(d["w13"], d["s13"], d["w2"], d["s2"], case["k"], pack=case["packed"])
        state = dict(layer=layer, logits=d["logits"])
        if case["from_f32"]:
            quant = {"tensor": hkmoe.quant_tensor, "block": hkmoe.quant_group, "mx": hkmoe.quant_mx}[case["scales"]]
            state.update(quant=quant, x=d["x"])
        else:
            state.update(quant=None, x=(d["x_q"], d["x_s"]))
        return state
    if case["kind"] == "gemm":
        d = _gemm_inputs(case, seed)
        return dict(gemm=d, out=torch.bfloat16 if case["out"] == "bf16" else torch.float32)
    if case["kind"] == "mx":
        d = _mx_inputs(case, seed)
        return dict(mx=d, packed=hkmoe.mx_pack_scales(d["sw"]),
                    out=torch.bfloat16 if case["out"] == "bf16" else torch.float32)
    return dict(fn=QUANT[case["what"]], x=_quant_input(case, seed))


def run(state):
    if "layer" in state:
        x_q, x_s = state["quant"](state["x"]) if state["quant"] else state["x"]
        return state["layer"](x_q, x_s, state["logits"])
    if "gemm" in state:
        d = state["gemm"]
        return hkmoe.gemm_fp8(d["a"], d["b"], d["sa"], d["sb"], out_dtype=state["out"])
    if "mx" in state:
        d = state["mx"]
        x_q, x_e = hkmoe.quant_mx(d["x"])
        return hkmoe.gemm_mx(x_q, hkmoe.mx_pack_scales(x_e), d["w"], state["packed"], out_dtype=state["out"])
    q, s = state["fn"](state["x"])
    return q, s


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _deq(q, s, scales):
    """e4m3 [R, C] with the scales of one matrix, in 64 bits."""
    v = q.double()
    if scales == "tensor":
        return v * s.double().reshape(1, 1)
    if scales == "mx":
        return (v.view(v.shape[0], -1, 32) * torch.exp2(s.double() - 127.0)[..., None]).view(v.shape)
    if scales == "group":
        return (v.view(v.shape[0], -1, 128) * s.double()[..., None]).view(v.shape)
    r, c = v.shape
    return (v.view(r // 128, 128, c // 128, 128) * s.double()[:, None, :, None]).view(r, c)


def _exact_moe(case, seed):
    d = _moe_inputs(case, seed)
    T, k, sc = case["T"], case["k"], case["scales"]
    xs = "group" if sc == "block" else sc
    x = _deq(d["x_q"], d["x_s"], xs)
    val, idx = torch.topk(d["logits"], k, dim=1)
    wgt = torch.softmax(val.double(), 1)
    inter = case["I"]
    hs = {}
    for e in idx.unique().tolist():
        t, j = (idx == e).nonzero(as_tuple=True)
        gu = x[t] @ _deq(d["w13"][e], d["s13"][e], sc).T
        gate, up = gu[:, :inter], gu[:, inter:]
        # the intermediate is bf16, then requantised: both are the path's formats
        hs[e] = (t, j, (gate * torch.sigmoid(gate) * up).to(torch.bfloat16).float())
    if sc == "tensor":
        s = _scale(torch.stack([h.abs().amax() for _, _, h in hs.values()]).amax().reshape(1))
    out = torch.zeros((T, case["H"]), dtype=torch.float64, device=DEV)
    for e, (t, j, h) in hs.items():
        if sc == "tensor":
            hq, h_s = (h / s).to(F8), s
        else:
            hq, h_s = (_q_group if sc == "block" else _q_mx)(h)
        y = _deq(hq, h_s, xs) @ _deq(d["w2"][e], d["s2"][e], sc).T
        out.index_add_(0, t, y.to(torch.bfloat16).double() * wgt[t, j][:, None])
    return out


def exact(case, seed):
    if case["kind"] == "moe":
        return _exact_moe(case, seed)
    if case["kind"] == "gemm":
        d = _gemm_inputs(case, seed)
        return (d["a"].double() @ d["b"].double().T) * (d["sa"].double() * d["sb"].double())
    if case["kind"] == "mx":
        d = _mx_inputs(case, seed)
        x_q, x_e = _q_mx(d["x"])
        return _deq(x_q, x_e, "mx") @ _deq(d["w"], d["sw"], "mx").T
    x = _quant_input(case, seed)
    if case["what"] == "block":
        q, s = _q_block(x[None])
        return q.view(x.shape).double(), s[0].double()
    q, s = {"group": _q_group, "tensor": _q_tensor, "mx": _q_mx}[case["what"]](x)
    return q.double(), None if case["what"] == "mx" else s.double()


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close it has to be
# ---------------------------------------------------------------------------
def _scale_bytes(rows, cols, scales):
    """Bytes of the scales of rows x cols activations (or of one weight matrix)."""
    return {"tensor": 4, "group": rows * cols // 128 * 4, "block": rows // 128 * (cols // 128) * 4,
            "mx": rows * cols // 32}[scales]


def work(case):
    if case["kind"] == "moe":
        T, k, E, H, I, sc = (case[n] for n in ("T", "k", "E", "H", "I", "scales"))
        g = torch.Generator()
        g.manual_seed(0)
        active = torch.topk(_logits(g, case, "cpu"), k, dim=1)[1].unique().numel()
        weights = active * (3 * I * H + _scale_bytes(2 * I, H, sc) + _scale_bytes(H, I, sc))
        x = T * H * 4 if case["from_f32"] else T * H + _scale_bytes(T, H, "group" if sc == "block" else sc)
        return {"bytes": weights + x + T * E * 4 + T * H * 2, "flops": 6 * T * k * H * I}
    if case["kind"] in ("gemm", "mx"):
        M, N, K = case["M"], case["N"], case["K"]
        a = M * K if case["kind"] == "gemm" else 4 * M * K
        b = N * K + (0 if case["kind"] == "gemm" else N * K // 32)
        return {"bytes": a + b + M * N * (2 if case["out"] == "bf16" else 4), "flops": 2 * M * N * K}
    n = case["rows"] * case["cols"]
    return {"bytes": 5 * n + _scale_bytes(case["rows"], case["cols"], case["what"]), "flops": 3 * n}


def tolerance(case):
    """About four times what the path measures against ``exact``: quantisers none
    (bytes and scales), layers 1.7e-3 .. 2.5e-3 and at most 5.5e-2 on one element
    (a requantised intermediate that moves by one e4m3 step), bf16 products
    1.7e-3 and 3.9e-3, fp32 products 1.2e-5 .. 1.6e-5 and 1e-4 (the matrix
    instruction's own sums)."""
    if case["kind"] == "quant":
        return "exact"
    if case["kind"] == "moe":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 7e-3, "max": 1.6e-2} if case["out"] == "bf16" else {"rel": 6e-5, "max": 4e-4}
