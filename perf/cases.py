"""What this library is timed on: the calls a program makes of it, at the sizes such programs have.

A case is one call (or the two or three calls that belong together) on inputs that sit where the program has them: in
HBM for the device entries, in host memory for the host-slice entries.  The kinds:

    prefill   bf16 self-attention over a prompt: [B,H,N,D] or [B,N,H,D] tensors, grouped kv heads, any mask
    padded    bf16 causal prefill of a batch padded to its longest sequence
    window    bf16 causal self-attention with a sliding window
    masked    bf16 attention between the projections of a MultiHeadAttention with an additive mask; cross-attention
    prompt    what precedes a prompt's attention: q/k norm, rotary embedding and the append to the cache
    token     what a decode loop runs per layer and token for one sequence: the same preparation, then attention
    decode    one new token for every sequence of a serving batch, caches filled to different lengths
    chunk     several new positions per sequence against the cache (a prompt taken in pieces, drafted tokens)
    forward   f32 attention forward on device tensors
    train     f32 forward that keeps its row statistic, then the gradients from it
    host      f32 attention forward on host slices: upload, kernel, download
"""
import math

import torch

import rustorch_amd as ra

K = ra.LlmKernels


def listed():
    return [
        # a batch of four long prompts on a 32-head model without grouped kv heads
        {"name": "prefill_b4_h32_n4096_d128", "kind": "prefill", "batch": 4, "heads": 32, "kv_heads": 32, "seq": 4096,
         "dim": 128, "mask": "causal", "layout": "bhnd"},
        # two prompts of an ordinary, odd length on a model with four query heads per kv head, in the layout the
        # projections leave
        {"name": "prefill_b2_gqa_n1501_d128", "kind": "prefill", "batch": 2, "heads": 32, "kv_heads": 8, "seq": 1501,
         "dim": 128, "mask": "causal", "layout": "bnhd"},
        # a batch of prompts of very different lengths, padded
        {"name": "padded_b16_h16_n1024_d64", "kind": "padded", "batch": 16, "heads": 16, "seq": 1024, "shortest": 128,
         "dim": 64},
        # local attention over long sequences
        {"name": "window_b4_h16_n4096_d64_w256", "kind": "window", "batch": 4, "heads": 16, "kv_heads": 16, "seq": 4096,
         "dim": 64, "window": 256, "layout": "bnhd"},
        # an encoder or decoder block with a mask tensor
        {"name": "masked_b4_h16_n1024_d64", "kind": "masked", "batch": 4, "heads": 16, "t_q": 1024, "t_kv": 1024,
         "dim": 64, "per_head": False},
        # the preparation of four long prompts
        {"name": "prompt_b4_gqa_n4096_d128", "kind": "prompt", "batch": 4, "heads": 32, "kv_heads": 8, "seq": 4096,
         "max_seq": 8192, "dim": 128, "norm": True},
        # one token of one conversation: the smallest call, and the one made most often
        {"name": "token_gqa_ctx2048_d128", "kind": "token", "heads": 32, "kv_heads": 8, "context": 2048, "max_seq": 4096,
         "dim": 128, "norm": True},
        # a serving batch of 64 sequences of 512 to 8192 tokens
        {"name": "decode_b64_gqa_ctx8192_d128", "kind": "decode", "batch": 64, "heads": 32, "kv_heads": 8,
         "shortest": 512, "context": 8192, "max_seq": 8192, "dim": 128},
        # sixteen new positions of one sequence over a long cache
        {"name": "chunk_b1_gqa_new16_ctx8192_d128", "kind": "chunk", "batch": 1, "heads": 32, "kv_heads": 8, "new": 16,
         "context": 8192, "max_seq": 8192, "dim": 128},
        # the f32 causal forward of a small model
        {"name": "forward_f32_b1_h8_n2048_d64", "kind": "forward", "batch": 1, "heads": 8, "seq": 2048, "dim": 64,
         "mask": "causal"},
        # one attention layer of a training step
        {"name": "train_f32_b4_h16_n1024_d64", "kind": "train", "batch": 4, "heads": 16, "seq": 1024, "dim": 64},
        # the host-slice call of a program whose tensors live on the host
        {"name": "host_f32_b1_h4_n1024_d64", "kind": "host", "batch": 1, "heads": 4, "seq": 1024, "dim": 64,
         "mask": "none"},
    ]


# ---- drawn cases ------------------------------------------------------------------------------------------------


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm; odd ones as likely as even ones."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _shrink(case, names, most):
    """Halves `names` in turn until the case costs no more than `most` (flops, and bytes at 1/300 of it)."""
    n = 0
    while max(work(case)["flops"], 300.0 * work(case)["bytes"]) > most and any(case[x] > 1 for x in names):
        x = names[n % len(names)]
        case[x] = max(1, case[x] // 2)
        n += 1
    return case


_BF16_DIMS = (64, 64, 64, 128, 128, 128, 128, 32, 80, 96, 256)
_F32_DIMS = (64, 64, 64, 128, 128, 32, 80, 96)
_MOST_BF16 = 2.5e11  # flops of a drawn bf16 case: half of the largest listed one, for the head dims that take longer
_MOST_F32 = 3e10


def _heads(rng):
    """(query heads, kv heads)"""
    return rng.choice(((8, 8), (16, 16), (32, 32), (12, 12), (32, 8), (16, 2), (40, 8), (28, 4), (8, 2)))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "padded", "window", "masked", "prompt", "token", "decode", "chunk", "forward",
                       "train", "host"))
    heads, kv_heads = _heads(rng)
    if kind == "prefill":
        case = {"kind": kind, "batch": _log(rng, 1, 8), "heads": heads, "kv_heads": kv_heads, "seq": _log(rng, 16, 16384),
                "dim": rng.choice(_BF16_DIMS), "mask": rng.choice(("causal", "causal", "causal", "none", "padding")),
                "layout": rng.choice(("bhnd", "bnhd"))}
        return _shrink(case, ("batch", "seq"), _MOST_BF16)
    if kind == "padded":
        seq = _log(rng, 64, 4096)
        case = {"kind": kind, "batch": _log(rng, 2, 32), "heads": heads, "seq": seq, "shortest": max(1, seq // rng.randint(2, 8)),
                "dim": rng.choice(_BF16_DIMS)}
        return _shrink(case, ("batch",), _MOST_BF16)
    if kind == "window":
        seq = _log(rng, 256, 16384)
        case = {"kind": kind, "batch": _log(rng, 1, 8), "heads": heads, "kv_heads": kv_heads, "seq": seq,
                "dim": rng.choice(_BF16_DIMS), "window": _log(rng, 64, max(64, seq // 4)),
                "layout": rng.choice(("bhnd", "bnhd"))}
        return _shrink(case, ("batch", "seq"), _MOST_BF16)
    if kind == "masked":
        t_q = _log(rng, 16, 4096)
        t_kv = t_q if rng.random() < 0.6 else _log(rng, 16, 4096)
        case = {"kind": kind, "batch": _log(rng, 1, 16), "heads": rng.choice((8, 12, 16)), "t_q": t_q, "t_kv": t_kv,
                "dim": rng.choice((32, 64, 64, 80, 96, 128)), "per_head": rng.random() < 0.2}
        return _shrink(case, ("batch", "t_q"), _MOST_BF16 / 4)
    if kind == "prompt":
        seq = _log(rng, 2, 8192)
        case = {"kind": kind, "batch": _log(rng, 1, 8), "heads": heads, "kv_heads": kv_heads, "seq": seq,
                "max_seq": seq + _log(rng, 1, 4096), "dim": rng.choice((64, 128, 128, 256)), "norm": rng.random() < 0.5}
        return _shrink(case, ("batch", "seq"), _MOST_BF16 / 2)
    if kind == "token":
        context = _log(rng, 1, 16384)
        return {"kind": kind, "heads": heads, "kv_heads": kv_heads, "context": context,
                "max_seq": max(context, rng.choice((2048, 4096, 8192))), "dim": rng.choice((64, 128, 128, 128, 256)),
                "norm": rng.random() < 0.5}
    if kind == "decode":
        context = _log(rng, 32, 8192)
        case = {"kind": kind, "batch": _log(rng, 1, 128), "heads": heads, "kv_heads": kv_heads,
                "shortest": max(1, context // rng.randint(1, 16)), "context": context,
                "max_seq": context + _log(rng, 1, 512), "dim": rng.choice((64, 128, 128, 128, 256))}
        return _shrink(case, ("batch",), _MOST_BF16)
    if kind == "chunk":
        new = _log(rng, 2, 512)
        context = new + _log(rng, 1, 8192)
        case = {"kind": kind, "batch": _log(rng, 1, 16), "heads": heads, "kv_heads": kv_heads, "new": new,
                "context": context, "max_seq": context + _log(rng, 1, 512), "dim": rng.choice((64, 128, 128, 128, 256))}
        return _shrink(case, ("batch",), _MOST_BF16)
    case = {"kind": kind, "batch": _log(rng, 1, 8), "heads": rng.choice((4, 8, 12, 16)), "seq": _log(rng, 16, 4096),
            "dim": rng.choice(_F32_DIMS)}
    if kind != "train":
        case["mask"] = rng.choice(("none", "causal"))
    return _shrink(case, ("batch", "seq"), _MOST_F32 if kind != "host" else _MOST_F32 / 8)


# ---- inputs -----------------------------------------------------------------------------------------------------


def _lengths(case):
    """The batch's lengths, evenly spread from the shortest to the longest."""
    b, lo, hi = case["batch"], case["shortest"], case.get("context", case["seq"] if "seq" in case else 0)
    return [hi] if b == 1 else [lo + (hi - lo) * i // (b - 1) for i in range(b)]


class _Rand:
    """Tensors of N(0, 1) values, as normalised activations have, from the seed."""

    def __init__(self, seed, device="cuda"):
        self.gen = torch.Generator(device=device)
        self.gen.manual_seed(seed)
        self.device = device

    def bf16(self, *shape):
        return torch.randn(shape, generator=self.gen, device=self.device, dtype=torch.bfloat16)

    def f32(self, *shape):
        return torch.randn(shape, generator=self.gen, device=self.device)


def _visible(case, n):
    """Keys that a padding mask leaves of n."""
    return max(1, n - n // 8)


def prepare(case, seed):
    kind, d = case["kind"], case["dim"]
    s = {"kind": kind, "case": case, "stream": torch.cuda.current_stream().cuda_stream}
    b = case.get("batch", 1)
    if kind == "host":
        r = _Rand(seed, "cpu")
        n = b * case["heads"] * case["seq"] * d
        s["shape"] = ra.AttentionShape.new(b, case["heads"], case["seq"], d)
        s["mask"] = ra.Mask.causal() if case["mask"] == "causal" else ra.Mask.none()
        s["q"], s["k"], s["v"] = (r.f32(n).numpy() for _ in range(3))
        s["out"] = torch.empty(n).numpy()
        return s
    r = _Rand(seed)
    h, hkv = case["heads"], case.get("kv_heads", case["heads"])
    if kind in ("prefill", "window"):
        n = case["seq"]
        if case["layout"] == "bnhd":
            s["q"], s["k"], s["v"] = r.bf16(b, n, h, d), r.bf16(b, n, hkv, d), r.bf16(b, n, hkv, d)
        else:
            s["q"], s["k"], s["v"] = r.bf16(b, h, n, d), r.bf16(b, hkv, n, d), r.bf16(b, hkv, n, d)
        s["out"] = torch.empty_like(s["q"])
        s["shape"] = ra.AttentionShape.new(b, h, n, d)
        if kind == "prefill":
            keep = torch.arange(n) < _visible(case, n)
            s["mask"] = {"none": ra.Mask.none, "causal": ra.Mask.causal, "padding": lambda: ra.Mask.padding(keep.numpy())}[case["mask"]]()
            s["keep"] = keep.to(torch.uint8).cuda() if case["mask"] == "padding" else None
            s["call"] = ra.flash_forward_bnhd_bf16_dev if case["layout"] == "bnhd" else ra.flash_forward_bf16_dev
    elif kind == "padded":
        s["q"], s["k"], s["v"] = (r.bf16(b, h, case["seq"], d) for _ in range(3))
        s["out"] = torch.empty_like(s["q"])
        lens = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
        s["lens"] = lens[torch.randperm(b, generator=r.gen, device="cuda")].contiguous()
        s["shape"] = ra.AttentionShape.new(b, h, case["seq"], d)
    elif kind == "masked":
        tq, tk = case["t_q"], case["t_kv"]
        s["q"], s["k"], s["v"] = r.bf16(b, tq, h * d), r.bf16(b, tk, h * d), r.bf16(b, tk, h * d)
        s["out"] = torch.empty_like(s["q"])
        # an additive mask: a band around the diagonal keeps its scores (plus a small position bias), the rest gets the
        # library's masking value
        i, j = torch.arange(tq, device="cuda")[:, None] * tk // tq, torch.arange(tk, device="cuda")[None, :]
        far = (i - j).abs() > max(16, tk // 4)
        bias = 0.1 * r.f32(*((b * h, tq, tk) if case["per_head"] else (tq, tk)))
        s["bias"] = torch.where(far, torch.full_like(bias, float(ra.MASK_NEG)), bias).contiguous()
    elif kind in ("prompt", "token"):
        new = case["seq"] if kind == "prompt" else 1
        s["q"], s["k_in"], s["v_in"] = r.bf16(b, h, new, d), r.bf16(b, hkv, new, d), r.bf16(b, hkv, new, d)
        s["k"], s["v"] = r.bf16(b, hkv, case["max_seq"], d), r.bf16(b, hkv, case["max_seq"], d)
        s["rope"] = ra.RoPE(d, case["max_seq"])
        s["rope"].device_tables()
        s["q_gamma"] = 1 + 0.1 * r.f32(d) if case["norm"] else None
        s["k_gamma"] = 1 + 0.1 * r.f32(d) if case["norm"] else None
        s["out"] = torch.empty_like(s["q"])
    elif kind in ("decode", "chunk"):
        new = case.get("new", 1)
        s["q"] = r.bf16(b, new, h, d)
        s["k"], s["v"] = r.bf16(b, hkv, case["max_seq"], d), r.bf16(b, hkv, case["max_seq"], d)
        s["out"] = torch.empty_like(s["q"])
        if kind == "decode":
            lens = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
            s["lens"] = lens[torch.randperm(b, generator=r.gen, device="cuda")].contiguous()
            s["ws_bytes"] = max(256, K.gqa_decode_workspace_bytes(b, h, hkv, d, case["max_seq"]))
            s["ws"] = torch.empty(s["ws_bytes"], dtype=torch.uint8, device="cuda")
    else:  # forward, train
        n = case["seq"]
        s["shape"] = ra.AttentionShape.new(b, h, n, d)
        s["q"], s["k"], s["v"] = (r.f32(b, h, n, d) for _ in range(3))
        s["out"] = torch.empty_like(s["q"])
        if kind == "forward":
            s["mask"] = ra.Mask.causal() if case["mask"] == "causal" else ra.Mask.none()
        else:
            s["d_out"] = r.f32(b, h, n, d)
            s["lse"] = torch.empty(b, h, n, device="cuda")
            s["dq"], s["dk"], s["dv"] = (torch.empty_like(s["q"]) for _ in range(3))
            s["ws_bytes"] = 4 * b * h * n
            s["ws"] = torch.empty(b * h * n, device="cuda")
    return s


# ---- one pass -----------------------------------------------------------------------------------------------------


def run(s):
    kind, c, stream = s["kind"], s["case"], s["stream"]
    if kind == "prefill":
        s["call"](s["shape"], s["q"], s["k"], s["v"], s["out"], s["mask"], s["keep"], c["kv_heads"], stream)
        return s["out"]
    if kind == "window":
        ra.flash_forward_window_bf16_dev(s["shape"], s["q"], s["k"], s["v"], s["out"], c["window"], c["kv_heads"],
                                         c["layout"] == "bnhd", stream)
        return s["out"]
    if kind == "padded":
        ra.flash_forward_varlen_bf16_dev(s["shape"], s["q"], s["k"], s["v"], s["lens"], s["out"], stream=stream)
        return s["out"]
    if kind == "masked":
        ra.mha_forward_masked_bf16_dev(s["q"], s["k"], s["v"], s["out"], c["batch"], c["t_q"], c["t_kv"], c["heads"],
                                       c["dim"], s["bias"], s["bias"].numel(), stream)
        return s["out"]
    if kind == "prompt":
        K.qk_norm_rope_kv_append_bf16(stream, s["q"], s["k_in"], s["v_in"], s["k"], s["v"], 0, s["rope"], c["batch"],
                                      c["heads"], c["kv_heads"], c["dim"], c["max_seq"], s["q_gamma"], s["k_gamma"],
                                      seq=c["seq"])
        return {"q": s["q"], "k_cache": s["k"], "v_cache": s["v"]}
    if kind == "token":
        K.qk_norm_rope_kv_append_bf16(stream, s["q"], s["k_in"], s["v_in"], s["k"], s["v"], c["context"] - 1, s["rope"], 1,
                                      c["heads"], c["kv_heads"], c["dim"], c["max_seq"], s["q_gamma"], s["k_gamma"])
        K.gqa_decode_online_bf16(stream, s["q"], s["k"], s["v"], s["out"], c["heads"], c["kv_heads"], c["context"],
                                 c["dim"], c["max_seq"])
        return {"out": s["out"], "q": s["q"], "k_cache": s["k"], "v_cache": s["v"]}
    if kind == "decode":
        K.gqa_decode_batched_bf16(stream, s["q"], s["k"], s["v"], s["out"], s["lens"], c["batch"], c["heads"],
                                  c["kv_heads"], c["dim"], c["max_seq"], s["ws"], s["ws_bytes"])
        return s["out"]
    if kind == "chunk":
        K.gqa_decode_chunk_bf16(stream, s["q"], s["k"], s["v"], s["out"], c["context"], c["batch"], c["new"], c["heads"],
                                c["kv_heads"], c["dim"], c["max_seq"])
        return s["out"]
    if kind == "forward":
        ra.flash_forward_f32_dev(s["shape"], s["q"], s["k"], s["v"], s["out"], s["mask"], stream=stream)
        return s["out"]
    if kind == "train":
        ra.flash_forward_stats_f32_dev(s["shape"], s["q"], s["k"], s["v"], s["out"], s["lse"], stream=stream)
        ra.flash_backward_saved_f32_dev(s["shape"], s["q"], s["k"], s["v"], s["out"], s["lse"], s["d_out"], s["dq"], s["dk"],
                                        s["dv"], s["ws"], s["ws_bytes"], stream=stream)
        return {"out": s["out"], "lse": s["lse"], "dq": s["dq"], "dk": s["dk"], "dv": s["dv"]}
    return ra.flash_forward_masked(s["shape"], s["q"], s["k"], s["v"], s["mask"], s["out"])


# ---- what a pass cannot do without --------------------------------------------------------------------------------


def _causal_pairs(queries, keys):
    """(query, key) pairs when the last query sees every key and each one before it one key less."""
    first = max(0, keys - queries)
    n = min(queries, keys)
    return n * first + n * (n + 1) // 2


def work(case):
    kind, d, h, b = case["kind"], case["dim"], case["heads"], case.get("batch", 1)
    hkv = case.get("kv_heads", h)
    if kind in ("prefill", "forward", "host"):
        n, e = case["seq"], 2 if kind == "prefill" else 4
        pairs = {"none": n * n, "causal": n * (n + 1) // 2, "padding": n * _visible(case, n)}[case["mask"]]
        return {"bytes": e * b * n * d * (2 * h + 2 * hkv), "flops": 4 * b * h * d * pairs}
    if kind == "window":
        n, w = case["seq"], min(case["window"], case["seq"])
        return {"bytes": 2 * b * n * d * (2 * h + 2 * hkv), "flops": 4 * b * h * d * (w * (w + 1) // 2 + (n - w) * w)}
    if kind == "padded":  # valid rows in, every row out
        lens = _lengths(case)
        return {"bytes": 2 * h * d * (3 * sum(lens) + b * case["seq"]), "flops": 4 * h * d * sum(x * (x + 1) // 2 for x in lens)}
    if kind == "masked":  # the mask is a bias: every pair is scored
        tq, tk = case["t_q"], case["t_kv"]
        bias = 4 * tq * tk * (b * h if case["per_head"] else 1)
        return {"bytes": 2 * b * h * d * (2 * tq + 2 * tk) + bias, "flops": 4 * b * h * d * tq * tk}
    if kind == "prompt":  # q in and out, k and v in, their cache rows out, the table rows
        n = case["seq"]
        return {"bytes": 2 * b * n * d * (2 * h + 4 * hkv) + 4 * n * d, "flops": 12 * b * n * d * (h + hkv)}
    if kind == "token":
        n = case["context"]
        return {"bytes": 4 * hkv * n * d + 2 * d * (4 * h + 4 * hkv), "flops": 4 * h * d * n}
    if kind == "decode":
        n = sum(_lengths(case))
        return {"bytes": 4 * hkv * d * n + 4 * b * h * d, "flops": 4 * h * d * n}
    if kind == "chunk":
        n, new = case["context"], case["new"]
        return {"bytes": b * (4 * hkv * d * n + 4 * new * h * d), "flops": 4 * b * h * d * _causal_pairs(new, n)}
    n = case["seq"]  # train: two products forward, five backward; q, k, v, d_out in, out, lse and three gradients out
    return {"bytes": 4 * b * h * n * (8 * d + 1), "flops": 14 * b * h * d * n * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "prompt":  # every rounding of the preparation is laid down
        return "exact"
    if kind in ("forward", "host", "train"):
        return {"rel": 1e-5}
    return {"rel": 1e-2}
