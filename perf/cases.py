"""Performance cases of the framework: what its users have it do, through its public entry points.

``kind`` of a case:
  train    conv-attention module, forward and autograd backward (O, dQ, dK, dV and the gradient of
           the window weights); ``dtype`` "bf16", or "fp32" for compute_dtype=torch.float32
  forward  the same module without gradients (prefill, evaluation)
  decode   one decode step over a dense KV cache (fwd_conv_attn_inference)
  serve    one decode step over a serving cache with sequences of their own lengths: pages of
           ``page`` keys (decode_paged), or a view of a preallocated cache when page is 0
           (decode_gqa); ``H_kv`` KV heads shared by ``H`` query heads
  mix      head-mixing attention module, forward and autograd backward

Q, K, V and dO are N(0, 1); window weights are the identity tap plus N(0, 0.05), mixing weights
N(0, 1 / H), as in the benchmark workloads of synthetic.py and benchmarks.py.
"""
import math

import torch

from flash_multi_token_attention_amd.conv_attn import ConvAttentionCUDA, fwd_conv_attn_inference
from flash_multi_token_attention_amd.conv_attn import ops
from flash_multi_token_attention_amd.head_conv_attn import HeadConvAttention

_DTYPE = {"bf16": torch.bfloat16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp32": 4}


def _attention(name, kind, B, H, N, d, c_q, c_k, dtype="bf16", causal=True):
    return {"name": name, "kind": kind, "B": B, "H": H, "N": N, "d": d, "c_q": c_q, "c_k": c_k, "dtype": dtype,
            "causal": causal}


def _decode(name, B, H, Nk, d, rows, c_q, c_k, splits):
    return {"name": name, "kind": "decode", "B": B, "H": H, "Nk": Nk, "d": d, "rows": rows, "c_q": c_q, "c_k": c_k,
            "splits": splits}


def _serve(name, B, H, H_kv, Nk, d, c_q, c_k, page):
    return {"name": name, "kind": "serve", "B": B, "H": H, "H_kv": H_kv, "Nk": Nk, "d": d, "c_q": c_q, "c_k": c_k,
            "page": page}


def _mix(name, B, H, N, d, causal=True):
    return {"name": name, "kind": "mix", "B": B, "H": H, "N": N, "d": d, "causal": causal}


def listed():
    return [
        # the first step of the training sweep: a short sequence, launches and host time count
        _attention("train_short", "train", 1, 8, 256, 64, 3, 3),
        # a mid-size batch of an odd length with the largest square window of the sweep
        _attention("train_ragged", "train", 2, 8, 1531, 64, 11, 11),
        # the headline training step (c3_fwd_bwd)
        _attention("train_headline", "train", 4, 16, 4096, 128, 6, 11),
        # long-context training (c5_long)
        _attention("train_long", "train", 1, 32, 16384, 128, 6, 11),
        # prefill / evaluation forward (c2_fwd)
        _attention("prefill", "forward", 4, 16, 2048, 64, 6, 11),
        # full-precision training: checks of a model against fp32, small models
        _attention("train_fp32", "train", 1, 8, 1024, 64, 6, 11, dtype="fp32"),
        # a decode step of a small model: the configuration of the reference's decode figure
        _decode("decode_small", 2, 2, 2048, 64, 16, 7, 7, 32),
        # the headline decode step (c4_decode), the split count left to the library
        _decode("decode_headline", 32, 32, 8192, 128, 6, 6, 11, 0),
        # serving: a batch of sequences of different lengths, shared KV heads, paged cache
        _serve("serve_paged", 32, 32, 8, 8192, 128, 6, 11, 64),
        # head mixing at the reference's own check size: odd length, launches count
        _mix("mix_short", 2, 16, 201, 32),
        # head mixing with 32 heads, mid-size
        _mix("mix_32_heads", 2, 32, 2048, 64),
        # the largest head-mixing step of the sweep
        _mix("mix_large", 4, 16, 4096, 128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(max(lo, hi))))))


def draw(rng):
    """One more case of the listed ones' ranges; no costlier than the costliest of them."""
    kind = rng.choice(["train", "train", "forward", "train_fp32", "decode", "serve", "mix", "mix"])
    if kind in ("train", "forward", "train_fp32"):
        causal = rng.random() < 0.85
        c_q, c_k = rng.choice([(3, 3), (3, 5), (6, 11), (6, 11), (7, 7), (11, 11)])
        if kind == "train_fp32":
            B, H = rng.choice([(1, 2), (1, 8), (2, 4)])
            d, longest, dtype = rng.choice([64, 128]), 2048, "fp32"
        else:
            B, H = rng.choice([(1, 8), (2, 8), (2, 12), (4, 16), (1, 32)])
            d, dtype = rng.choice([64, 128] if c_q > 8 else [32, 64, 64, 128, 128]), "bf16"
            # (score products and window products per pair; c5_long has 9.6e11 of these units)
            per_pair = (d + 16 * c_q) * B * H * (0.5 if causal else 1.0)
            longest = min(16384, int(math.sqrt(6e11 / per_pair)))
        c = _attention("", "forward" if kind == "forward" else "train", B, H, _log_int(rng, 200, longest), d, c_q, c_k, dtype, causal)
    elif kind == "decode":
        B, H = rng.choice([(1, 8), (2, 2), (4, 16), (8, 32), (32, 32)])
        d = rng.choice([64, 128])
        Nk = _log_int(rng, 500, min(65536, 4.2e9 / (4 * B * H * d)))
        c_q, c_k = rng.choice([(3, 3), (6, 11), (7, 7), (11, 11)])
        c = _decode("", B, H, Nk, d, rng.choice([c_q, 16]), c_q, c_k, rng.choice([0, 0, 32]))
    elif kind == "serve":
        B = rng.choice([1, 4, 16, 32])
        H, H_kv = rng.choice([(8, 8), (16, 4), (32, 8), (32, 32)])
        d = rng.choice([64, 128])
        Nk = _log_int(rng, 500, min(65536, 4.2e9 / (4 * B * H_kv * d)))
        c_q, c_k = rng.choice([(3, 3), (6, 11), (6, 11), (11, 11)])
        c = _serve("", B, H, H_kv, Nk, d, c_q, c_k, rng.choice([0, 16, 64, 256]))
    else:
        B, H, d = rng.choice([1, 2, 4]), rng.choice([16, 16, 32]), rng.choice([32, 64, 128])
        causal = rng.random() < 0.85
        most = 9e11 if H == 16 else 2.5e11
        per_pair = (14 * max(d, 64) + 8 * H) * B * H * (0.5 if causal else 1.0)
        c = _mix("", B, H, _log_int(rng, 100, min(4096, int(math.sqrt(most / per_pair)))), d, causal)
    del c["name"]
    return c


def _window(c, normal):
    """Identity tap (current query row, same key) plus noise, [H, c_q, c_k] fp32."""
    W = 0.05 * normal(c["H"], c["c_q"], c["c_k"], dtype=torch.float32)
    W[:, c["c_q"] - 1, c["c_k"] // 2] += 1.0
    return W


def prepare(case, seed):
    c = dict(case)
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(int(seed))

    def normal(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g, device=dev, dtype=dtype)

    s = {"case": c}
    B, H, d = c["B"], c["H"], c["d"]
    if c["kind"] in ("train", "forward", "mix"):
        dt = _DTYPE[c.get("dtype", "bf16")]
        s["Q"], s["K"], s["V"], s["dO"] = (normal(B, H, c["N"], d, dtype=dt) for _ in range(4))
        if c["kind"] == "mix":
            s["module"] = HeadConvAttention(H, dtype=torch.float32).to(dev)
            with torch.no_grad():
                s["module"].head_conv_weights.copy_(normal(H, H, dtype=torch.float32) / math.sqrt(H))
        else:
            s["module"] = ConvAttentionCUDA(H, c["c_q"], c["c_k"], compute_dtype=dt).to(dev)
            with torch.no_grad():
                s["module"].conv_weight.copy_(_window(c, normal))
        if c["kind"] != "forward":
            for n in ("Q", "K", "V"):
                s[n].requires_grad_(True)
        return s
    s["scale"] = 1.0 / math.sqrt(d)
    s["W"] = _window(c, normal)
    if c["kind"] == "decode":
        s["Q"] = normal(B, H, c["rows"], d)
        s["K"], s["V"] = normal(B, H, c["Nk"], d), normal(B, H, c["Nk"], d)
        return s
    s["Q"] = normal(B, H, c["c_q"], d)
    # every sequence has its own length, the longest is full
    lens = [c["Nk"]] + [int(x) for x in torch.randint(max(1, c["Nk"] // 4), c["Nk"] + 1, (B - 1,),
                                                      generator=torch.Generator().manual_seed(int(seed)))]
    s["lens"] = torch.tensor(lens, dtype=torch.int32, device=dev)
    if c["page"]:
        pages = -(-c["Nk"] // c["page"])
        s["K"], s["V"] = (normal(B * pages, c["H_kv"], c["page"], d) for _ in range(2))
        s["table"] = torch.randperm(B * pages, generator=g, device=dev).to(torch.int32).reshape(B, pages).contiguous()
    else:
        room = c["Nk"] + 64
        s["K"], s["V"] = (normal(B, c["H_kv"], room, d)[:, :, :c["Nk"]] for _ in range(2))
    return s


def run(state):
    c = state["case"]
    if c["kind"] == "forward":
        with torch.no_grad():
            return state["module"](state["Q"], state["K"], state["V"], causal=c["causal"])
    if c["kind"] in ("train", "mix"):
        m = state["module"]
        O = m(state["Q"], state["K"], state["V"], causal=c["causal"])
        w = m.head_conv_weights if c["kind"] == "mix" else m.conv_weight
        return (O,) + torch.autograd.grad(O, (state["Q"], state["K"], state["V"], w), state["dO"])
    if c["kind"] == "decode":
        return fwd_conv_attn_inference(state["Q"], state["K"], state["V"], state["W"], c["splits"], state["scale"],
                                       c["c_q"] - 1, (c["c_k"] - 1) // 2, False)
    if c["page"]:
        return ops.decode_paged(state["Q"], state["K"], state["V"], state["table"], state["lens"], c["Nk"],
                                state["W"], 0, state["scale"])[:3]
    return ops.decode_gqa(state["Q"], state["K"], state["V"], state["W"], 0, state["scale"], seq_lens=state["lens"])[:3]


def work(case):
    c = case
    B, H, d = c["B"], c["H"], c["d"]
    if c["kind"] in ("train", "forward", "mix"):
        N = c["N"]
        pairs = B * H * (N * (N + 1) / 2 if c["causal"] else float(N) * N)
        taps = 0 if c["kind"] == "mix" else c["c_q"] * c["c_k"]
        mix = H if c["kind"] == "mix" else 0
        weights = 4 * (H * H if c["kind"] == "mix" else H * taps)
        rows = B * H * N * d * _BYTES[c.get("dtype", "bf16")]
        if c["kind"] == "forward":   # Q, K, V -> O
            return {"bytes": 4 * rows + weights, "flops": pairs * (4 * d + 2 * taps)}
        # Q, K, V, dO -> O, dQ, dK, dV; Q K^T, P V, then S, dP, dQ, dK, dV; the window (or the mix) once
        # forward, once again and transposed backward, and its gradient
        return {"bytes": 8 * rows + 2 * weights, "flops": pairs * (14 * d + 8 * taps + 8 * mix)}
    if c["kind"] == "decode":
        keys, rows, kv_heads = B * c["Nk"], c["rows"], H
    else:
        # the longest sequence is full, the others are 5/8 of it in the mean
        keys, rows, kv_heads = c["Nk"] * (1 + (B - 1) * 0.625), c["c_q"], c["H_kv"]
    return {"bytes": 2 * keys * kv_heads * d * 2 + B * H * (rows * d * 2 + d * 4 + 8) + 4 * H * c["c_q"] * c["c_k"],
            "flops": keys * H * (2 * d * c["c_q"] + 2 * c["c_q"] * c["c_k"] + 2 * d)}


def tolerance(case):
    if case["kind"] in ("decode", "serve"):
        return {"rel": 2e-5}   # bf16 inputs, fp32 arithmetic and results
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1e-2}       # bf16 operands and results
