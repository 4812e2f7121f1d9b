"""The performance cases: calls through the public Python surface, over the
sizes that the repository's benchmark, tests and published tables use.

A case is a dict of plain values; its "kind" says which entry point it calls:

* mm         a resident GEMM session: launch-only batch, then the result
             downloaded (fp32, bf16 or f16 compute)
* mm_call    matmul2d with host arrays in and out
* attn       a resident attention session: launch-only batch, then a forward
             that downloads (fp32, bf16 or f16; batch x heads)
* attn_call  attention2d with host arrays in and out
* train      dV-only SGD training: upload, resident steps, last step downloads
             the output, the updated V and the loss
* vit        a ViT block session: image uploaded, resident forwards, tokens
             downloaded
* conv_attn  the integrated conv -> attention call with host arrays

`passes` is how many launches of the resident work one pass makes: the
benchmark's resident loops (100 GEMMs) and the reference's batch calls.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lightining-core_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import lightning_core as lc  # noqa: E402


def listed():
    return [
        # The smallest call: the reference's published conv -> attention pipeline, one request at a time.
        {"name": "conv_attn_seq96_d48", "kind": "conv_attn", "n": 1, "cin": 3, "cout": 16, "hw": 8, "s": 96, "d": 48},
        # One attention2d call on numpy arrays, the reference's headline attention size.
        {"name": "attn_call_f32_256x64", "kind": "attn_call", "s": 256, "d": 64, "causal": False},
        # fp32 multi-head attention kept resident, a sequence that is no multiple of a tile.
        {"name": "attn_f32_h8_s1000_d64", "kind": "attn", "dtype": "f32", "b": 1, "h": 8, "s": 1000, "d": 64,
         "causal": True, "passes": 20},
        # The reference's training benchmark: one head trained in a resident loop.
        {"name": "train_f32_512x64", "kind": "train", "s": 512, "d": 64, "causal": False, "passes": 50},
        # matmul2d on numpy arrays, ragged in every dimension.
        {"name": "mm_call_f32_ragged", "kind": "mm_call", "m": 1000, "k": 777, "n": 1030},
        # The default-precision resident GEMM at the reference's headline size.
        {"name": "mm_f32_1024", "kind": "mm", "dtype": "f32", "m": 1024, "k": 1024, "n": 1024, "passes": 100},
        # The largest rectangular shape of the reference's published fp32 sweep.
        {"name": "mm_f32_4096x1024x4096", "kind": "mm", "dtype": "f32", "m": 4096, "k": 1024, "n": 4096,
         "passes": 100},
        # The large 16-bit GEMM that the benchmark's headline is quoted on.
        {"name": "mm_bf16_8192", "kind": "mm", "dtype": "bf16", "m": 8192, "k": 8192, "n": 8192, "passes": 100},
        # An ordinary 16-bit projection of a few sequences' tokens, sizes off the tile.
        {"name": "mm_f16_1500x3000x2000", "kind": "mm", "dtype": "f16", "m": 1500, "k": 3000, "n": 2000,
         "passes": 100},
        # A decode step's projection: 16 rows against a large resident weight.
        {"name": "mm_bf16_16x8192x8192", "kind": "mm", "dtype": "bf16", "m": 16, "k": 8192, "n": 8192,
         "passes": 100},
        # Prefill: batched causal multi-head attention in 16 bits.
        {"name": "attn_bf16_b4h16_s2048_d128", "kind": "attn", "dtype": "bf16", "b": 4, "h": 16, "s": 2048,
         "d": 128, "causal": True, "passes": 100},
        # Vision inference: image batch in, block output out.
        {"name": "vit_f16_b8", "kind": "vit", "dtype": "f16", "b": 8, "image": 224, "patch": 16, "embed": 768,
         "heads": 12, "passes": 100},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mm", "mm", "mm", "mm_call", "attn", "attn", "attn_call", "train", "vit", "conv_attn"])
    if kind == "mm":
        dtype = rng.choice(["f32", "bf16", "f16"])
        top = 4096 if dtype == "f32" else 8192
        # rows from one decode step's to a prefill's; weights of an ordinary layer
        m, k, n = _log(rng, 1 if dtype != "f32" else 64, top), _log(rng, 256, top), _log(rng, 256, top)
        if rng.random() < 0.5:  # half of them at multiples of 64, as most layers are
            m, k, n = (max(64, v // 64 * 64) if v > 64 else v for v in (m, k, n))
        return {"kind": kind, "dtype": dtype, "m": m, "k": k, "n": n, "passes": 100}
    if kind == "mm_call":
        return {"kind": kind, "m": _log(rng, 32, 2048), "k": _log(rng, 32, 2048), "n": _log(rng, 32, 2048)}
    if kind == "attn":
        dtype = rng.choice(["f32", "bf16", "f16"])
        s = _log(rng, 128, 2048 if dtype == "f32" else 4096)
        return {"kind": kind, "dtype": dtype, "b": rng.randint(1, 4), "h": rng.choice([1, 4, 8, 12, 16]), "s": s,
                "d": rng.choice([64, 128]), "causal": rng.random() < 0.5, "passes": 20}
    if kind == "attn_call":
        return {"kind": kind, "s": _log(rng, 32, 1024), "d": rng.choice([32, 48, 64, 128]),
                "causal": rng.random() < 0.5}
    if kind == "train":
        return {"kind": kind, "s": _log(rng, 64, 2048), "d": rng.choice([32, 64, 128]),
                "causal": rng.random() < 0.5, "passes": 50}
    if kind == "vit":
        return {"kind": kind, "dtype": rng.choice(["f16", "bf16"]), "b": rng.randint(1, 32),
                "image": rng.choice([112, 160, 192, 224]), "patch": 16, "embed": 768, "heads": 12, "passes": 100}
    hw = rng.choice([8, 16, 32])
    return {"kind": kind, "n": 1, "cin": 3, "cout": rng.choice([16, 32]), "hw": hw, "s": _log(rng, 48, 256),
            "d": rng.choice([8, 16, 32, 48, 64])}


# --- inputs ---------------------------------------------------------------------

def _sizes(case):
    """The input tensors of a case: name -> (shape, standard deviation)."""
    kind = case["kind"]
    if kind in ("mm", "mm_call"):  # normalised activations times weights scaled by their fan-in
        return {"a": ((case["m"], case["k"]), 1.0), "b": ((case["k"], case["n"]), case["k"] ** -0.5)}
    if kind == "attn":
        shape = (case["b"], case["h"], case["s"], case["d"])
        return {x: (shape, 1.0) for x in "qkv"}
    if kind in ("attn_call", "train"):
        names = ("q", "k", "v", "target") if kind == "train" else ("q", "k", "v")
        return {x: ((case["s"], case["d"]), 1.0) for x in names}
    if kind == "vit":
        e, p = case["embed"], case["patch"]
        return {"x": ((case["b"], 3, case["image"], case["image"]), 1.0),
                "w_conv": ((e, 3, p, p), (3 * p * p) ** -0.5), "w_qkv": ((e, 3 * e), e ** -0.5),
                "w_o": ((e, e), e ** -0.5)}
    return {"x": ((case["n"], case["cin"], case["hw"], case["hw"]), 1.0),
            "w": ((case["cout"], case["cin"], 3, 3), (9 * case["cin"]) ** -0.5), "bias": ((case["cout"],), 0.1)}


def _inputs(case, seed):
    """fp32 inputs on the GPU, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return {name: torch.randn(shape, generator=gen, device="cuda").mul_(std)
            for name, (shape, std) in _sizes(case).items()}


def _learning_rate(case):
    # The loss is a mean over S*D values; the rate takes that factor back.
    return 0.125 * case["s"] * case["d"]


def prepare(case, seed):
    host = {name: t.cpu().numpy() for name, t in _inputs(case, seed).items()}
    kind = case["kind"]
    state = {"case": dict(case)}
    if kind == "mm":
        state["out"] = np.empty(case["m"] * case["n"], np.float32)
        state["session"] = lc.matmul2d_resident_session(host["a"], host["b"], compute_dtype=case["dtype"])
        state["session"].start_into(host["a"], host["b"], state["out"])
    elif kind == "attn":
        state.update(host)
        state["out"] = np.empty(case["b"] * case["h"] * case["s"] * case["d"], np.float32)
        state["session"] = lc.AttentionSession.batched(case["b"], case["h"], case["s"], case["d"],
                                                       causal=case["causal"], compute_dtype=case["dtype"])
        state["resident"] = lc.AttentionIoPolicy(upload_q=False, upload_k=False, upload_v=False)
        state["session"].forward_with_policy_into(host["q"], host["k"], host["v"], state["out"],
                                                  lc.AttentionIoPolicy())
    elif kind == "train":
        state.update(host)
        state["session"] = lc.AttentionSession(case["s"], case["d"], causal=case["causal"])
        state["first"] = lc.AttentionIoPolicy(download_out=False, download_v=False, synchronize=False)
        state["last"] = lc.AttentionIoPolicy(upload_q=False, upload_k=False, upload_v=False, upload_target=False,
                                             download_v=True, loss_every=1)
    elif kind == "vit":
        state["x"] = host["x"]
        state["session"] = lc.VitBlockSession(case["b"], 3, case["image"], case["image"], case["patch"],
                                              case["embed"], case["heads"], compute_dtype=case["dtype"])
        state["session"].set_weights(host["w_conv"], host["w_qkv"], host["w_o"])
    else:
        state.update(host)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mm":
        state["session"].run_batch_sync_cached_no_download(case["passes"] - 1)
        return state["session"].finish_into(out=state["out"])
    if kind == "mm_call":
        return lc.matmul2d(state["a"], state["b"])
    if kind == "attn":
        state["session"].run_cached(case["passes"] - 1)
        state["session"].forward_with_policy_into(state["q"], state["k"], state["v"], state["out"],
                                                  state["resident"])
        return state["out"]
    if kind == "attn_call":
        return lc.attention2d(state["q"], state["k"], state["v"], causal=case["causal"])
    if kind == "train":
        s, lr = state["session"], _learning_rate(case)
        args = (state["q"], state["k"], state["v"], state["target"], lr)
        s.train_step_with_policy(*args, state["first"])
        s.train_run_cached(lr, case["passes"] - 2)
        return s.train_step_with_policy(*args, state["last"])
    if kind == "vit":
        state["session"].forward(state["x"], download=False)
        state["session"].run_cached(case["passes"] - 2)
        return state["session"].forward()
    return lc.api.conv_attention_torchstrong_nchw(state["x"], state["w"], state["bias"], case["s"], case["d"],
                                                  pad_h=1, pad_w=1)


# --- what a pass cannot do without ------------------------------------------------

def _attention_flops(heads, s, d, causal):
    return 2.0 * heads * d * s * (s + 1) if causal else 4.0 * heads * d * s * s


def work(case):
    kind = case["kind"]
    if kind in ("mm", "mm_call"):
        m, k, n = case["m"], case["k"], case["n"]
        size = 2 if case.get("dtype", "f32") != "f32" else 4
        times = case.get("passes", 1)
        return {"bytes": times * (size * (m * k + k * n) + 4.0 * m * n), "flops": times * 2.0 * m * k * n}
    if kind in ("attn", "attn_call"):
        heads = case.get("b", 1) * case.get("h", 1)
        size = 2 if case.get("dtype", "f32") != "f32" else 4
        times = case.get("passes", 1)
        return {"bytes": times * heads * case["s"] * case["d"] * (3.0 * size + 4),
                "flops": times * _attention_flops(heads, case["s"], case["d"], case["causal"])}
    if kind == "train":  # scores and output, then dV: three products; q, k, v, target in, v out
        n = case["s"] * case["d"]
        return {"bytes": case["passes"] * 5.0 * 4 * n,
                "flops": case["passes"] * 1.5 * _attention_flops(1, case["s"], case["d"], case["causal"])}
    if kind == "vit":
        e, p, b = case["embed"], case["patch"], case["b"]
        t = (case["image"] // p) ** 2
        rows, heads = b * t, b * case["heads"]
        flops = 2.0 * rows * e * (3 * p * p + 4 * e) + _attention_flops(heads, t, e // case["heads"], False)
        size = 2.0 * (rows * 3 * p * p + e * 3 * p * p + 4 * e * e) + 4.0 * rows * e
        return {"bytes": case["passes"] * size, "flops": case["passes"] * flops}
    n, cin, cout, hw, s, d = (case[x] for x in ("n", "cin", "cout", "hw", "s", "d"))
    return {"bytes": 4.0 * (n * cin * hw * hw + 9 * cin * cout + cout + s * d),
            "flops": 18.0 * n * cin * cout * hw * hw + _attention_flops(1, s, d, False)}


def tolerance(case):
    kind, dtype = case["kind"], case.get("dtype", "f32")
    if kind == "mm":  # the operands' rounding is fixed; sums are 32 bits wide for every dtype
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "vit" or dtype != "f32":  # probabilities and tokens between the stages are 16 bits wide
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 1e-5, "max": 1e-4}


# --- the same in 64 bits ----------------------------------------------------------

def _softmax_scores(q, k, causal):
    scores = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        s = scores.shape[-1]
        scores.masked_fill_(torch.ones(s, s, dtype=torch.bool, device=scores.device).triu_(1), -math.inf)
    return torch.softmax(scores, -1)


def _heads_attention(q, k, v, causal):
    out = torch.empty_like(q)
    for i in range(q.shape[0]):
        out[i] = torch.matmul(_softmax_scores(q[i], k[i], causal), v[i])
    return out


def exact(case, seed):
    kind = case["kind"]
    t = {name: x.double() for name, x in _inputs(case, seed).items()}
    if kind in ("mm", "mm_call"):
        c = torch.matmul(t["a"], t["b"])
        return c.reshape(-1) if kind == "mm" else c
    if kind == "attn":
        flat = (x.reshape(-1, case["s"], case["d"]) for x in (t["q"], t["k"], t["v"]))
        return _heads_attention(*flat, case["causal"]).reshape(-1)
    if kind == "attn_call":
        return torch.matmul(_softmax_scores(t["q"], t["k"], case["causal"]), t["v"])
    if kind == "train":
        p, v = _softmax_scores(t["q"], t["k"], case["causal"]), t["v"]
        step = 2.0 * _learning_rate(case) / v.numel()
        for _ in range(case["passes"]):
            out = torch.matmul(p, v)
            diff = out - t["target"]
            v = v - step * torch.matmul(p.t().contiguous(), diff)
        return out.reshape(-1), v, float(diff.square().mean())
    if kind == "vit":
        e, h = case["embed"], case["heads"]
        conv = torch.nn.functional.unfold(t["x"], case["patch"], stride=case["patch"])  # [B, C*P*P, T]
        tokens = torch.relu(torch.matmul(conv.transpose(1, 2).contiguous(), t["w_conv"].reshape(e, -1).t().contiguous()))
        b, n = tokens.shape[:2]
        qkv = torch.matmul(tokens, t["w_qkv"]).reshape(b, n, 3, h, e // h).permute(2, 0, 3, 1, 4)
        q, k, v = (x.reshape(b * h, n, e // h).contiguous() for x in qkv)
        out = _heads_attention(q, k, v, False).reshape(b, h, n, e // h).permute(0, 2, 1, 3).reshape(b, n, e)
        return torch.matmul(out.contiguous(), t["w_o"])
    n, s, d = case["n"], case["s"], case["d"]
    cols = torch.nn.functional.unfold(t["x"], 3, padding=1)  # [N, C*9, H*W]
    conv = torch.relu(torch.matmul(t["w"].reshape(case["cout"], -1), cols) + t["bias"][:, None]).reshape(-1)
    packed = conv.repeat(-(-3 * s * d // conv.numel()))[: 3 * s * d].reshape(3, s, d)
    return torch.matmul(_softmax_scores(packed[0], packed[1], False), packed[2]).reshape(-1)
