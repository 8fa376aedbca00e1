"""The work that users of this package have it do, as cases that can be timed and checked.

A case is a dict of plain values; ``path`` names the entry points it goes through:

* ``layer``     ``HyperConnection``: ``bi, add = hc(H); H_new = add(branch_output)``, either alone under
                ``torch.no_grad`` (``mode`` "infer") or followed by the backward of both outputs into H,
                the branch output and every parameter ("train").  ``graph`` replays the same calls from a
                HIP graph captured once, as a serving loop or a launch-bound training loop does.
* ``ops``       the four stream ops composed by hand: ``expand_streams``, ``fused_stream_mix``,
                ``fused_add_residual``, ``collapse_streams``, forward and backward.
* ``sinkhorn``  ``sinkhorn_knopp`` over a batch of 4x4 matrices, forward and backward.
* ``weights``   ``fused_dynamic_weights`` over rows of hidden states, forward and backward.

Sizes are the benchmark's, the tests' and the README example's, or plain round and odd numbers between
them.  Gradients are dropped at the start of a training pass, as ``zero_grad(set_to_none=True)`` does.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mhc-triton_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mhc  # noqa: E402
from mhc import streams  # noqa: E402

_DT = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_SIZE = {"fp32": 4, "bf16": 2, "fp16": 2}


def _layer(name, B, S, D, dtype, weights="dynamic", mode="train", graph=False, params="fp32"):
    return {"name": name, "path": "layer", "B": B, "S": S, "D": D, "dtype": dtype, "weights": weights,
            "mode": mode, "graph": graph, "params": params}


def listed():
    return [
        # one token of one sequence, called eagerly: interactive decoding, where latency is all there is
        _layer("decode one", 1, 1, 4096, "bf16", mode="infer"),
        # one token of each of 64 sequences from a captured graph: a serving loop
        _layer("decode batch, graph", 64, 1, 4096, "bf16", mode="infer", graph=True),
        # the prompt of one sequence of odd length
        _layer("prefill", 1, 1999, 4096, "bf16", mode="infer"),
        # the README's example layer at its size, in fp32: a small experiment or a unit test
        _layer("train small fp32", 2, 128, 512, "fp32"),
        # a micro-batch of a mid-sized model whose step is captured in a graph
        _layer("train mid, graph", 4, 512, 2048, "bf16", graph=True),
        # many short sequences (classification, packed dialogue turns), also captured
        _layer("train short, graph", 512, 8, 2048, "bf16", graph=True),
        # the headline workload: dim 4096 bf16, batch 4, sequence 4096
        _layer("train large", 4, 4096, 4096, "bf16"),
        # static weights in a half-precision module, as the reference's own benchmark casts it
        _layer("train static fp16", 16, 2048, 2048, "fp16", weights="static", params="same"),
        # a width that is not a whole number of 16-byte vectors, and an odd length
        _layer("train ragged", 3, 1023, 1500, "bf16"),
        # the stream ops composed by hand around a branch, at a mid-sized model's micro-batch
        {"name": "ops", "path": "ops", "B": 4, "S": 2048, "D": 2048, "dtype": "bf16"},
        # a million matrices at the default 20 rounds: per-token mixing matrices of a long batch
        {"name": "sinkhorn", "path": "sinkhorn", "n": 1 << 20, "iters": 20, "dtype": "fp32"},
        # weights for every token of a long batch
        {"name": "weights of tokens", "path": "weights", "R": 16384, "K": 16384, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_any(rng):
    path = rng.choice(["layer"] * 6 + ["ops", "sinkhorn", "weights"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if path == "sinkhorn":
        return {"path": path, "n": _log(rng, 1024, 1 << 20), "iters": rng.choice([7, 10, 20, 20, 32]), "dtype": dtype}
    if path == "weights":
        return {"path": path, "R": _log(rng, 4, 16384), "K": 4 * 8 * _log(rng, 16, 512), "dtype": dtype}
    # widths: mostly whole 16-byte vectors, now and then any number
    D = _log(rng, 100, 7168)
    if rng.random() < 0.75:
        D = max(8, D // 8 * 8)
    if path == "ops":
        return {"path": path, "B": _log(rng, 1, 16), "S": _log(rng, 16, 4096), "D": D, "dtype": dtype}
    mode = rng.choice(["infer", "train", "train"])
    weights = rng.choice(["dynamic"] * 4 + ["static", "unfused"])
    short = rng.random() < 0.3
    B, S = (_log(rng, 1, 512), rng.randint(1, 16)) if short else (_log(rng, 1, 16), _log(rng, 16, 8192))
    return {"path": path, "B": B, "S": S, "D": D, "dtype": dtype, "weights": weights, "mode": mode,
            "graph": weights != "unfused" and rng.random() < 0.4, "params": rng.choice(["fp32", "fp32", "same"])}


def draw(rng):
    most = max(work(c)["bytes"] for c in listed())
    while True:
        case = _draw_any(rng)
        if work(case)["bytes"] <= most:
            return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(shape, g, dtype, scale=1.0):
    t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (t.mul_(scale) if scale != 1.0 else t).to(dtype)


def _hidden(B, S, D, g, dtype):
    """Hidden states of four streams: unit noise around a mean of each channel's own."""
    H = torch.randn((B, S, 4, D), generator=g, device="cuda", dtype=torch.float32)
    H += torch.randn((4, D), generator=g, device="cuda").mul_(0.5)
    return H.to(dtype)


def _module(case, g):
    """The layer with trained-looking parameters: every one off its initial value."""
    hc = mhc.HyperConnection(case["D"], dynamic=case["weights"] != "static",
                             use_fused_weights=case["weights"] != "unfused").to("cuda")
    with torch.no_grad():
        for name, p in hc.named_parameters():
            noise = torch.randn(p.shape, generator=g, device="cuda")
            if name == "phi" or name.startswith("W_"):
                p.copy_(noise * 0.02)
            else:
                p.add_(noise * 0.05)
    return hc.to(_DT[case["dtype"]]) if case["params"] == "same" else hc


def _inputs(case, seed):
    """Everything that a pass reads, by name."""
    g = _gen(seed)
    dt = _DT[case["dtype"]]
    if case["path"] == "sinkhorn":
        n = case["n"]
        return {"M": _randn((n, 4, 4), g, dt), "dP": _randn((n, 4, 4), g, dt)}
    if case["path"] == "weights":
        R, K = case["R"], case["K"]
        return {"x": _randn((R, K), g, dt), "phi": _randn((K, 24), g, torch.float32, 0.02),
                "bias": _randn((24,), g, torch.float32, 0.5),
                "alpha": [torch.full((1,), 0.1, device="cuda") for _ in range(3)],
                "g_pre": _randn((R, 4), g, torch.float32), "g_post": _randn((R, 4), g, torch.float32),
                "g_res": _randn((R, 4, 4), g, torch.float32)}
    B, S, D = case["B"], case["S"], case["D"]
    if case["path"] == "ops":
        return {"x": _randn((B, S, D), g, dt), "bo": _randn((B, S, D), g, dt),
                "H_pre": torch.rand((B, 4), generator=g, device="cuda") * 0.5,
                "H_post": torch.rand((B, 4), generator=g, device="cuda") * 2,
                "H_res": torch.rand((B, 4, 4), generator=g, device="cuda") * 0.5,
                "d_bi": _randn((B, S, D), g, dt), "d_y": _randn((B, S, D), g, dt)}
    got = {"hc": _module(case, g), "H": _hidden(B, S, D, g, dt), "bo": _randn((B, S, D), g, dt)}
    if case["mode"] == "train":
        got["dH_new"] = _randn((B, S, 4, D), g, dt)
        got["d_bi"] = _randn((B, S, D), g, dt)
    return got


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _infer(s):
    with torch.no_grad():
        bi, add = s["hc"](s["H"])
        return [bi, add(s["bo"])]


def _train(s):
    for t in s["leaves"]:
        t.grad = None
    bi, add = s["hc"](s["H"])
    H_new = add(s["bo"])
    torch.autograd.backward([H_new, bi], [s["dH_new"], s["d_bi"]])
    return [bi.detach(), H_new.detach()] + [t.grad for t in s["leaves"]]


def _pass_ops(s):
    for t in s["leaves"]:
        t.grad = None
    H = streams.expand_streams(s["x"])
    bi, H_residual = mhc.fused_stream_mix(H, s["H_pre"], s["H_res"])
    H_new = mhc.fused_add_residual(H_residual, s["bo"], s["H_post"])
    y = streams.collapse_streams(H_new)
    torch.autograd.backward([bi, y], [s["d_bi"], s["d_y"]])
    return [bi.detach(), H_new.detach(), y.detach()] + [t.grad for t in s["leaves"]]


def _pass_sinkhorn(s):
    s["M"].grad = None
    P = mhc.sinkhorn_knopp(s["M"], s["iters"])
    P.backward(s["dP"])
    return [P.detach(), s["M"].grad]


def _pass_weights(s):
    for t in s["leaves"]:
        t.grad = None
    out = mhc.fused_dynamic_weights(s["x"], s["phi"], s["bias"], *s["alpha"])
    torch.autograd.backward(out, [s["g_pre"], s["g_post"], s["g_res"]])
    return [t.detach() for t in out] + [t.grad for t in s["leaves"]]


def prepare(case, seed):
    s = _inputs(case, seed)
    path = case["path"]
    if path == "sinkhorn":
        s["M"].requires_grad_(True)
        s.update(iters=case["iters"], go=_pass_sinkhorn)
    elif path == "weights":
        s["leaves"] = [s["x"], s["phi"], s["bias"], *s["alpha"]]
        s["go"] = _pass_weights
    elif path == "ops":
        s["leaves"] = [s["x"], s["bo"], s["H_pre"], s["H_post"], s["H_res"]]
        s["go"] = _pass_ops
    elif case["mode"] == "train":
        s["leaves"] = [s["H"], s["bo"], *s["hc"].parameters()]
        s["go"] = _train
    else:
        s["go"] = _infer
    for t in s.get("leaves", []):
        t.requires_grad_(True)
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                s["go"](s)
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        for t in s.get("leaves", []):
            t.grad = None
        with torch.cuda.graph(s["graph"]):
            s["out"] = s["go"](s)
    return s


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return state["go"](state)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how close two correct ones are
# ---------------------------------------------------------------------------

def work(case):
    path, e = case["path"], _SIZE[case["dtype"]]
    if path == "sinkhorn":
        n, it = case["n"], case["iters"]
        return {"bytes": n * 16 * 4 * e, "flops": n * it * (64 + 112)}
    if path == "weights":
        R, K = case["R"], case["K"]
        return {"bytes": 2 * R * K * e + 2 * K * 24 * 4 + 2 * R * 24 * 4, "flops": R * K * (2 * 25 + 4 * 24 + 2)}
    T, D = case["B"] * case["S"], case["D"]
    if path == "ops":  # in: x, bo, d_bi, d_y; out: bi, H_new, y, dx, d_bo
        return {"bytes": 12 * T * D * e, "flops": 150 * T * D}
    phi = 4 * D * 24 * 4 if case["weights"] != "static" else 0
    if case["mode"] == "infer":  # in: H, bo; out: bi, H_new
        return {"bytes": 10 * T * D * e + phi, "flops": 51 * T * D + 50 * 4 * D * case["B"]}
    # in: H, bo, dH_new, d_bi; out: bi, H_new, dH, d_bo
    return {"bytes": 20 * T * D * e + 2 * phi, "flops": 150 * T * D + 150 * 4 * D * case["B"]}


def tolerance(case):
    # 16-bit outputs: one rounding of an fp32 value (against 64 bits 1.7e-3 in bf16, 2.1e-4 in fp16), which
    # two correct evaluations may place one unit in the last place apart.  The fp32 gradients among them are
    # sums in another order (up to 2e-5 where a sum cancels).
    if case["dtype"] == "bf16":
        return {"rel": 7e-3, "max": 3e-2}
    if case["dtype"] == "fp16":
        return {"rel": 1e-3, "max": 4e-3}
    return {"rel": 7e-5, "max": 7e-4}


# ---------------------------------------------------------------------------
# The same passes in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _sinkhorn64(M, iters, eps):
    P = M.abs() + eps
    for _ in range(iters):
        P = P / (P.sum(dim=-1, keepdim=True) + eps)
        P = P / (P.sum(dim=-2, keepdim=True) + eps)
    return P


def _weights64(x, phi, bias, a_pre, a_post, a_res, iters=20, eps=1e-6):
    raw = (x @ phi) / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)
    sg = torch.sigmoid(a_pre * raw[:, 0:4] + bias[0:4])
    return (sg / (sg.sum(dim=-1, keepdim=True) + eps), 2 * torch.sigmoid(a_post * raw[:, 4:8] + bias[4:8]),
            _sinkhorn64((a_res * raw[:, 8:24] + bias[8:24]).reshape(-1, 4, 4), iters, eps))


def _mix64(H, w):
    """sum_n w[:, n] H[:, :, n] for w [B, 4]."""
    return sum(w[:, n, None, None] * H[:, :, n] for n in range(4))


def _layer_weights64(p, H, kind, iters=20, eps=1e-6):
    """(H_pre, H_post, H_res) of the three kinds of layer."""
    B = H.shape[0]
    if kind == "static":
        sg = torch.sigmoid(p["H_pre_base"])
        return ((sg / (sg.sum() + 1e-8)).expand(B, 4), torch.sigmoid(p["H_post_base"]).expand(B, 4),
                _sinkhorn64(p["H_res_base"][None], iters, 1e-8).expand(B, 4, 4))
    x = H.mean(dim=1).reshape(B, -1)
    if kind == "dynamic":
        bias = torch.cat([p["H_pre_base"], p["H_post_base"], p["H_res_base"].flatten()])
        return _weights64(x, p["phi"], bias, p["alpha_pre"], p["alpha_post"], p["alpha_res"], iters, eps)
    x = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)
    sg = torch.sigmoid(p["H_pre_base"] + (x @ p["W_pre.weight"].T) * p["scale_pre"])
    return (sg / (sg.sum(dim=-1, keepdim=True) + 1e-8),
            torch.sigmoid(p["H_post_base"] + (x @ p["W_post.weight"].T) * p["scale_post"]),
            _sinkhorn64(p["H_res_base"] + (x @ p["W_res.weight"].T).reshape(B, 4, 4) * p["scale_res"], iters, 1e-8))


def _leaf64(t):
    return t.detach().double().requires_grad_(True)


def exact(case, seed):
    s = _inputs(case, seed)
    path = case["path"]
    if path == "sinkhorn":
        M = _leaf64(s["M"])
        P = _sinkhorn64(M, case["iters"], 1e-8)
        P.backward(s["dP"].double())
        return [P.detach(), M.grad]
    if path == "weights":
        leaves = [_leaf64(t) for t in (s["x"], s["phi"], s["bias"], *s["alpha"])]
        out = _weights64(*leaves)
        torch.autograd.backward(out, [s[k].double() for k in ("g_pre", "g_post", "g_res")])
        return [t.detach() for t in out] + [t.grad for t in leaves]
    if path == "ops":
        x, bo, pre, post, res = leaves = [_leaf64(s[k]) for k in ("x", "bo", "H_pre", "H_post", "H_res")]
        H = x[:, :, None].expand(-1, -1, 4, -1)
        bi = _mix64(H, pre)
        H_new = torch.stack([_mix64(H, res[:, n]) + post[:, n, None, None] * bo for n in range(4)], dim=2)
        y = H_new.mean(dim=2)
        torch.autograd.backward([bi, y], [s["d_bi"].double(), s["d_y"].double()])
        return [bi.detach(), H_new.detach(), y.detach()] + [t.grad for t in leaves]
    train = case["mode"] == "train"
    names = [n for n, _ in s["hc"].named_parameters()]
    with torch.set_grad_enabled(train):
        p = {n: _leaf64(t) for n, t in s["hc"].named_parameters()}
        H, bo = _leaf64(s["H"]), _leaf64(s["bo"])
        pre, post, res = _layer_weights64(p, H, case["weights"])
        bi = _mix64(H, pre)
        H_new = torch.stack([_mix64(H, res[:, n]) + post[:, n, None, None] * bo for n in range(4)], dim=2)
        if train:
            torch.autograd.backward([H_new, bi], [s["dH_new"].double(), s["d_bi"].double()])
            return [bi.detach(), H_new.detach(), H.grad, bo.grad] + [p[n].grad for n in names]
    return [bi, H_new]
