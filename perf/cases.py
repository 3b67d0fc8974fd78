"""Workloads of the attention and quantised-linear path of a diffusion transformer, through this package's public
entry points: ``listed()`` names twelve of them, ``draw(rng)`` gives further ones from the same ranges, ``prepare``
makes a workload's inputs and layers on the GPU, ``run`` is one pass, ``work`` what such a pass cannot do without
and ``tolerance`` how far two correct implementations of the same precision may be apart."""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(1, os.path.join(os.getcwd(), "mindie-sd_amd"))

import mindiesd  # noqa: E402
from mindiesd.layers.quant import mx_quantize  # noqa: E402
from mindiesd.quantization.layer import FP8RotateQuantFA, W8A8MXFP8QuantLinear  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

# the most a drawn case may cost: dense attention of the 720p video (4 N S^2 D)
MOST_FLOPS = 4.0 * 40 * 75600 ** 2 * 128


def _dense(batch, heads, q_len, kv_len, dim, dtype="bf16", layout="BSND", text_pad=0):
    """``text_pad``: that many keys at the end are text of which each batch entry uses a prefix; 0: no mask."""
    return {"path": "dense", "batch": batch, "heads": heads, "q_len": q_len, "kv_len": kv_len, "dim": dim,
            "dtype": dtype, "layout": layout, "text_pad": text_pad}


def _packed(heads, tokens, sequences, causal, lengths_on_gpu):
    return {"path": "packed", "heads": heads, "tokens": tokens, "sequences": sequences, "causal": causal,
            "lengths_on_gpu": lengths_on_gpu}


def _sparse(kind, heads, grid, sparsity, layout="BNSD"):
    return {"path": "sparse", "kind": kind, "heads": heads, "t": grid[0], "h": grid[1], "w": grid[2],
            "sparsity": sparsity, "layout": layout}


def _fp8(heads, length, layout="BNSD"):
    return {"path": "fp8", "heads": heads, "length": length, "layout": layout}


def _linear(tokens, inner, outer, swiglu, bias):
    """``outer``: output features of the layer; with ``swiglu`` the weight has twice as many rows."""
    return {"path": "linear", "tokens": tokens, "inner": inner, "outer": outer, "swiglu": swiglu, "bias": bias}


def listed():
    return [
        # a small picture (32 x 32 latent tokens) with 77 text tokens in one sequence: the launch and the host count
        dict(_dense(1, 24, 1101, 1101, 128), name="small_image_joint"),
        # picture of 64 x 64 latent tokens with up to 226 text tokens, both guidance branches in one batch, the
        # text padding masked out of the keys
        dict(_dense(2, 24, 4322, 4322, 128, layout="BNSD", text_pad=226), name="image_joint_padded"),
        # self attention of a 480p video clip (21 x 30 x 52 latent tokens) in the small video model
        dict(_dense(1, 12, 32760, 32760, 128), name="video_480p"),
        # the same of a 720p clip (21 x 45 x 80) in the large one: the largest call
        dict(_dense(1, 40, 75600, 75600, 128, layout="BNSD"), name="video_720p"),
        # a video model with 64-wide heads (13 x 30 x 45 latent and 226 text tokens), run in fp16
        dict(_dense(1, 48, 17776, 17776, 64, dtype="fp16", layout="BNSD"), name="video_head_dim_64"),
        # the video tokens' attention over the encoded prompt
        dict(_dense(1, 40, 32760, 512, 128), name="cross_attention_text"),
        # pictures of different sizes packed into one call, lengths on the host
        dict(_packed(24, 16380, 7, False, False), name="packed_images"),
        # RainFusion block-sparse attention of the 720p clip, three quarters of the key blocks dropped
        dict(_sparse("rf_v3", 40, (21, 45, 80), 0.75), name="rainfusion_720p"),
        # adaptive block-sparse attention of the 480p clip: mask estimate and attention
        dict(_sparse("ada_bsa", 12, (21, 30, 52), 0.75), name="adaptive_sparse_480p"),
        # FP8 attention module (rotation, quantisation, attention) of the 480p clip in the large model
        dict(_fp8(40, 32760), name="fp8_attention_480p"),
        # MXFP8 projection of the encoded prompt (key or value of the cross attention)
        dict(_linear(512, 5120, 5120, False, True), name="mxfp8_text_projection"),
        # MXFP8 gated feed-forward input layer on all tokens of the 480p clip
        dict(_linear(32760, 5120, 13824, True, False), name="mxfp8_ffn_480p"),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _draw_grid(rng):
    """A latent grid of 2000 to 75600 tokens."""
    while True:
        t, h, w = rng.randint(1, 21), rng.randint(16, 60), rng.randint(16, 104)
        if 2000 <= t * h * w <= 75600:
            return t, h, w


def draw(rng):
    path = rng.choice(("self", "self", "padded", "cross", "packed", "sparse", "fp8", "linear", "linear"))
    layout = rng.choice(("BNSD", "BSND"))
    heads = rng.choice((8, 12, 16, 20, 24, 30, 40, 48))
    if path in ("self", "padded"):
        dim = rng.choice((64, 128, 128))
        batch = rng.randint(1, 2)
        longest = 75600 if path == "self" else 20000
        length = _log_int(rng, 512, longest)
        while 4.0 * batch * heads * length ** 2 * dim > MOST_FLOPS:
            length = _log_int(rng, 512, longest)
        return _dense(batch, heads, length, length, dim, rng.choice(("bf16", "bf16", "fp16")), layout,
                      0 if path == "self" else rng.randint(32, 512))
    if path == "cross":
        return _dense(rng.randint(1, 2), min(heads, 40), _log_int(rng, 1024, 75600), _log_int(rng, 64, 1024), 128,
                      "bf16", layout)
    if path == "packed":
        return _packed(heads, _log_int(rng, 2048, 32760), rng.randint(2, 16), rng.random() < 0.25, rng.random() < 0.5)
    if path == "sparse":
        return _sparse(rng.choice(("rf_v3", "ada_bsa")), min(heads, 40), _draw_grid(rng),
                       rng.choice((0.5, 0.6, 0.7, 0.75, 0.8, 0.85, 0.9)), layout)
    if path == "fp8":
        return _fp8(min(heads, 40), _log_int(rng, 1024, 75600), layout)
    inner = rng.choice((1536, 3072, 5120))
    swiglu = rng.random() < 0.4
    outer = inner * rng.choice((2, 3, 4)) if swiglu else inner * rng.choice((1, 1, 3, 4))
    return _linear(_log_int(rng, 64, 75600), inner, outer, swiglu, rng.random() < 0.6)


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _normal(g, *shape, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def _latent_field(g, heads, grid, layout):
    """Queries or keys of a video: per head and channel a field that varies slowly over the frames, rows and columns
    of the latent grid, plus a third of noise (block-sparse attention lives on that structure)."""
    t, h, w = grid
    coarse = torch.randn((heads, 128, max(2, t // 2), max(2, h // 5), max(2, w // 5)), generator=g, device="cuda")
    x = F.interpolate(coarse, size=(t, h, w), mode="trilinear", align_corners=True)
    x = x / x.std()
    x = x.add_(torch.randn(x.shape, generator=g, device="cuda"), alpha=0.3).flatten(2)     # [heads, 128, tokens]
    return (x.transpose(1, 2) if layout == "BNSD" else x.permute(2, 0, 1)).to(torch.bfloat16).unsqueeze(0).contiguous()


def _cuts(g, tokens, sequences):
    """Cumulative lengths of ``sequences`` sequences of unequal lengths that sum to ``tokens``."""
    share = torch.rand(sequences, generator=g, dtype=torch.float64) + 0.1
    ends = (share.cumsum(0) / share.sum() * tokens).round().to(torch.int64).tolist()
    return [0] + [int(e) for e in ends[:-1]] + [tokens]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    path = case["path"]
    if path == "dense":
        dtype, bnsd = DTYPES[case["dtype"]], case["layout"] == "BNSD"
        def tensor(length):
            b, n, d = case["batch"], case["heads"], case["dim"]
            return _normal(g, *((b, n, length, d) if bnsd else (b, length, n, d)), dtype=dtype)
        q, k, v = tensor(case["q_len"]), tensor(case["kv_len"]), tensor(case["kv_len"])
        mask = None
        if case["text_pad"]:
            used = torch.randint(1, case["text_pad"] + 1, (case["batch"], 1), generator=g, device="cuda")
            keys = torch.arange(case["kv_len"], device="cuda").unsqueeze(0)
            mask = (keys < case["kv_len"] - case["text_pad"] + used).view(case["batch"], 1, 1, case["kv_len"])
        return {"path": path, "qkv": (q, k, v), "mask": mask, "head_first": bnsd}
    if path == "packed":
        qkv = tuple(_normal(g, case["tokens"], case["heads"], 128) for _ in range(3))
        cu = _cuts(torch.Generator().manual_seed(seed), case["tokens"], case["sequences"])
        if case["lengths_on_gpu"]:
            cu = torch.tensor(cu, dtype=torch.int32, device="cuda")
        return {"path": path, "qkv": qkv, "cu": cu, "causal": case["causal"]}
    if path == "sparse":
        grid = (case["t"], case["h"], case["w"])
        q, k = (_latent_field(g, case["heads"], grid, case["layout"]) for _ in range(2))
        options = {"sparse_type": case["kind"], "head_num": case["heads"], "input_layout": case["layout"],
                   "sparsity": case["sparsity"]}
        if case["kind"] == "rf_v3":
            options["latent_shape_q"] = list(grid)
        else:
            options["cdf_threshold"] = 0.9
        return {"path": path, "qkv": (q, k, _normal(g, *k.shape)), "options": options}
    if path == "fp8":
        n, s = case["heads"], case["length"]
        shape = (1, n, s, 128) if case["layout"] == "BNSD" else (1, s, n, 128)
        def with_outliers():                                  # one element in a hundred eight times as large
            x = torch.randn(shape, generator=g, device="cuda")
            return torch.where(torch.rand(shape, generator=g, device="cuda") < 0.01, x * 8, x).to(torch.bfloat16)
        qkv = tuple(with_outliers() for _ in range(3))
        had = torch.ones((1, 1), device="cuda")
        while had.shape[0] < 128:
            had = torch.cat([torch.cat([had, had], 1), torch.cat([had, -had], 1)], 0)
        rot = (had / 128 ** 0.5).to(torch.bfloat16)
        return {"path": path, "qkv": qkv, "module": FP8RotateQuantFA("attn", {"attn.q_rot": rot, "attn.k_rot": rot}),
                "layout": case["layout"]}
    rows = case["outer"] * (2 if case["swiglu"] else 1)
    w_q, w_scale = mx_quantize(_normal(g, rows, case["inner"]) * 0.02)
    weights = {"fc.weight": w_q, "fc.weight_scale": w_scale}
    if case["bias"]:
        weights["fc.bias"] = torch.randn(rows, generator=g, device="cuda") * 0.1
    layer = W8A8MXFP8QuantLinear(case["inner"], rows, bias=case["bias"], weights=weights, prefix="fc",
                                 swiglu=case["swiglu"])
    return {"path": path, "x": _normal(g, 1, case["tokens"], case["inner"]), "module": layer}


# ---- one pass -------------------------------------------------------------------------------------------------------
def run(state):
    path = state["path"]
    if path == "linear":
        return state["module"](state["x"])
    q, k, v = state["qkv"]
    if path == "dense":
        return mindiesd.attention_forward(q, k, v, attn_mask=state["mask"], head_first=state["head_first"])
    if path == "packed":
        return mindiesd.attention_forward_varlen(q, k, v, state["cu"], state["cu"], causal=state["causal"])
    if path == "sparse":
        return mindiesd.sparse_attention(q, k, v, **state["options"])
    return state["module"](q, k, v, layout=state["layout"])


def work(case):
    path = case["path"]
    if path == "dense":
        rows = case["batch"] * case["heads"] * case["dim"]
        keys = case["kv_len"] - case["text_pad"] / 2          # on average half of the padded text is there
        return {"bytes": 4.0 * rows * (case["q_len"] + keys), "flops": 4.0 * rows * case["q_len"] * keys}
    if path == "packed":
        # unequal shares (0.1 + U(0,1)): the mean square of a length is 1.23 times the square of the mean
        n, t = case["heads"], case["tokens"]
        return {"bytes": 8.0 * n * t * 128,
                "flops": 4.0 * n * 128 * 1.23 * t * t / case["sequences"] * (0.5 if case["causal"] else 1.0)}
    if path == "sparse":
        s, n = case["t"] * case["h"] * case["w"], case["heads"]
        keep, products = 1.0 - case["sparsity"], 0.0
        if case["kind"] == "rf_v3":
            first = 1.0 / case["t"]                           # first-frame rows see all keys, all rows the first frame
            keep = first + (1.0 - first) * max(first, keep)
        else:
            products = 2.0 * n * (s / 8.0) ** 2 * 8 * 128     # strided scores behind the estimated mask
        return {"bytes": 8.0 * n * s * 128, "flops": 4.0 * n * s * s * 128 * keep + products}
    if path == "fp8":
        n, s = case["heads"], case["length"]
        return {"bytes": 8.0 * n * s * 128, "flops": 4.0 * n * s * s * 128}
    rows = case["outer"] * (2 if case["swiglu"] else 1)
    m, k = case["tokens"], case["inner"]
    return {"bytes": 2.0 * m * k + rows * k * (1 + 1 / 32) + 2.0 * m * case["outer"], "flops": 2.0 * m * k * rows}


def tolerance(case):
    """About four times the relative error that the path shows against the same operands in 64-bit arithmetic
    (FP8 attention: that its two rules for rounding a probability show against each other)."""
    if case["path"] == "fp8":
        return {"rel": 0.03, "max": 0.9}      # 0.012 and 0.39: probabilities carry 3-bit mantissas
    if case["path"] == "linear":
        return {"rel": 7e-3, "max": 0.02}     # 0.0017 and 0.004: exact products, one rounding to bf16
    if case["path"] == "dense" and case["dtype"] == "fp16":
        return {"rel": 1.5e-3, "max": 6e-3}   # 0.00037 and 0.0015
    if case["path"] == "sparse":
        return {"rel": 1.3e-2, "max": 0.17}   # 0.0033 and 0.042
    return {"rel": 1.2e-2, "max": 0.07}       # 0.0029 and 0.017: 16-bit probabilities and output
