"""GPU parity of the MXFP8 path vs the CPU oracle: MX quantisation bit-exact against the OCP MX
definition; GEMM (+ bias) and GEMM + SwiGLU against the dequantise -> exact GEMM oracle.  Stated
tolerance: cosine >= 0.999; since both sides multiply the same quantised numbers the match is in
fact limited only by fp32 accumulation and the 16-bit output rounding, which is asserted too."""
import pytest
import torch

from oracle import quant as oq
from oracle.attention import cosine

pytestmark = pytest.mark.gpu


def _rand(shape, seed, scale=1.0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mx_quant_bit_exact(cuda, dtype):
    from mindiesd.layers.quant import mx_quantize
    x = _rand((300, 512), 1, dtype=dtype) * torch.logspace(-2, 2, 300)[:, None].to(dtype)
    x[7, 64:96] = 0
    q, e = mx_quantize(x.to(cuda))
    codes, e8 = oq.mx_quant(x)
    assert q.dtype == torch.float8_e4m3fn and e.dtype == torch.float8_e8m0fnu and e.shape == (300, 16)
    assert torch.equal(e.view(torch.uint8).cpu(), e8)
    assert torch.equal(q.view(torch.uint8).cpu() & 0x7f, codes & 0x7f)
    assert torch.equal((q.view(torch.uint8).cpu() >> 7)[codes & 0x7f != 0], (codes >> 7)[codes & 0x7f != 0])


@pytest.mark.parametrize("m,k,f", [(256, 512, 128), (300, 1024, 136), (1000, 256, 520)])
def test_gemm_swiglu_vs_oracle(cuda, m, k, f):
    from mindiesd.layers.quant import mx_quantize, mxfp8_gemm_swiglu
    x = _rand((m, k), 2)
    w = _rand((2 * f, k), 3, scale=0.05)
    wq, ws = mx_quantize(w.to(cuda))
    out = mxfp8_gemm_swiglu(x.to(cuda), wq, ws).cpu()
    want = oq.mxfp8_gemm_swiglu(x, w, torch.float32)
    assert out.shape == (m, f) and out.dtype == torch.bfloat16
    assert cosine(out, want) >= 0.999
    err = (out.float() - want).abs()
    assert (err <= 2.0 ** -7 * want.abs() + 1e-3).all(), f"max err {err.max()}"


def test_plain_gemm_with_bias_and_linear_module(cuda):
    from mindiesd.layers.quant import mx_quantize, mxfp8_matmul
    from mindiesd.quantization import W8A8MXFP8QuantLinear
    m, k, n = 520, 384, 264
    x = _rand((2, m // 2, k), 4)
    w = _rand((n, k), 5, scale=0.05)
    bias = _rand((n,), 6, dtype=torch.float32)
    wq, ws = mx_quantize(w.to(cuda))
    want = oq.mxfp8_gemm(x.reshape(m, k), w, bias).float()
    xq, xs = mx_quantize(x.reshape(m, k).to(cuda))
    out = mxfp8_matmul(xq, xs, wq, ws, bias.to(cuda), torch.bfloat16).cpu()
    assert out.shape == (m, n)
    assert ((out.float() - want).abs() <= 2.0 ** -7 * want.abs() + 1e-3).all()
    # reference-shaped module: weight_scale stored as [N, K/64, 2]
    weights = {"ffn.up.weight": wq, "ffn.up.weight_scale": ws.view(torch.uint8).reshape(n, k // 64, 2),
               "ffn.up.bias": bias.to(cuda)}
    lin = W8A8MXFP8QuantLinear(k, n, bias=True, weights=weights, prefix="ffn.up")
    y = lin(x.to(cuda))
    assert y.shape == (2, m // 2, n) and torch.equal(y.reshape(m, n).cpu(), out)


def tile(m, nw, swiglu):
    """The tile the GEMM takes, as its dispatch has it: the smallest whose grid is one round over 256 compute units, 128 x 128
    also in two rounds against one of 256 x 256; SwiGLU halves the columns a tile covers."""
    def count(tm, tn):
        return -(-m // tm) * -(-(nw // 2 if swiglu else nw) // (tn // 2 if swiglu else tn))
    if not swiglu and count(64, 64) <= 256:
        return 64, 64
    if count(64, 128) <= 256:
        return 64, 128
    return (128, 128) if count(128, 128) <= (512 if count(256, 256) <= 256 else 256) else (256, 256)


# shapes of every tile, plain and SwiGLU, 128 x 128 in one and in two rounds; rows and columns past a tile's edge; K of one block,
# of a few, and of 9, 11 or 13 (more than two chunks of scales, a number four does not divide)
@pytest.mark.parametrize("m,k,nw,swiglu,want_tile", [
    (1, 128, 8, False, (64, 64)), (65, 640, 1032, False, (64, 64)), (200, 1152, 1000, False, (64, 64)),
    (320, 640, 3600, False, (64, 128)), (130, 1152, 6000, False, (64, 128)),
    (64, 512, 16, True, (64, 128)), (130, 384, 2064, True, (64, 128)), (70, 1664, 1040, True, (64, 128)),
    (700, 128, 3080, False, (128, 128)), (1000, 896, 2056, False, (128, 128)), (700, 1152, 3080, False, (128, 128)),
    (1536, 1408, 5000, False, (128, 128)),
    (300, 256, 9232, True, (128, 128)), (300, 1408, 9232, True, (128, 128)), (1100, 640, 6160, True, (128, 128)),
    (2100, 128, 4104, False, (256, 256)), (4500, 128, 4104, False, (256, 256)), (2100, 640, 4104, False, (256, 256)),
    (2305, 1152, 4616, False, (256, 256)), (2100, 384, 8208, True, (256, 256)), (2100, 1664, 8208, True, (256, 256))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_tiles_vs_oracle(cuda, m, k, nw, swiglu, want_tile, dtype):
    """Against the exact product of the quantised operands on sampled rows (all of the first and last tile's edges):
    the matrix instruction aligns its 64 products to the largest and drops what falls below (measured with the bias set to
    minus the exact result: 2^-13 of the largest product and instruction at K 128, less at larger K; twice that is allowed),
    fp32 sums of K products deviate by at most K 2^-24 sum |x w|, the output rounds by 2^-9 (bf16, half an ulp) or 2^-12
    (fp16), and silu * up carries the error of two sums."""
    from mindiesd.layers.quant import mx_quantize, mxfp8_matmul
    assert tile(m, nw, swiglu) == want_tile
    x, w, bias = _rand((m, k), 11), _rand((nw, k), 12, scale=0.05), _rand((nw,), 13, dtype=torch.float32)
    xq, xs = mx_quantize(x.to(cuda))
    wq, ws = mx_quantize(w.to(cuda))
    got = mxfp8_matmul(xq, xs, wq, ws, bias.to(cuda), dtype, swiglu).double().cpu()
    assert got.shape == (m, nw // 2 if swiglu else nw)
    rows = torch.cat([torch.arange(0, m, max(1, m // 37)), torch.arange(max(0, m - 70), m)]).unique()
    deq = lambda q, e: (q.float().cpu().view(q.shape[0], -1, 32) * e.float().cpu().unsqueeze(-1)).view(q.shape).double()
    xd, wd = deq(xq, xs)[rows], deq(wq, ws)
    want, slack = xd @ wd.T + bias.double(), k * 2.0 ** -24 * (xd.abs() @ wd.abs().T + bias.double().abs())
    slack += k / 64 * 2.0 ** -12 * xd.abs().amax(1, keepdim=True) * wd.abs().amax(1)
    if swiglu:
        g, u = want.chunk(2, -1)
        sg, su = slack.chunk(2, -1)
        want = torch.nn.functional.silu(g) * u
        # |silu'| <= 1.1; exp2, reciprocal and the products add a few fp32 roundings
        slack = 1.1 * sg * (u.abs() + su) + g.abs() * su + 2.0 ** -18 * (g * u).abs()
    err = (got[rows] - want).abs()
    half_ulp = (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12) * 2 * want.abs()
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0
    assert (err <= half_ulp * (1 + 2.0 ** -6) + slack + tiny).all(), float((err - half_ulp - slack).max())


# Plain products that the rule above gives 128 x 128 tiles in one round: where 96 columns to a tile are still one round they run
# as 128 x 96, the others do not.  Columns past a tile's edge by 8, 40 and 88, exactly 256 workgroups of either.
@pytest.mark.parametrize("m,k,nw,columns", [(385, 1408, 5000, 96), (129, 640, 12200, 96), (512, 128, 5128, 96), (1000, 1152, 2056, 96),
                                            (900, 640, 3080, 128), (1000, 128, 4088, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_tiles_of_96_columns(cuda, m, k, nw, columns, dtype):
    assert columns == (96 if -(-m // 128) * -(-nw // 96) <= 256 else 128)
    test_gemm_tiles_vs_oracle(cuda, m, k, nw, False, (128, 128), dtype)


def test_gemm_errors(cuda):
    from mindiesd import ParametersInvalid
    from mindiesd.layers.quant import mx_quantize, mxfp8_matmul
    x = _rand((64, 96), 7)
    xq, xs = mx_quantize(x.to(cuda))
    with pytest.raises(ParametersInvalid):
        mxfp8_matmul(xq, xs, xq, xs)            # K not a multiple of 128
    with pytest.raises(ParametersInvalid):
        mx_quantize(_rand((4, 40), 8).to(cuda))  # K not a multiple of 32


def test_quantize_injected_layers_match_direct_calls(cuda, tmp_path):
    """quantize() on a toy block (descriptor + safetensors written here): the swapped-in linear equals the direct
    MXFP8 GEMM on the same tensors, the attached fa_quant equals the direct FP8 attention call."""
    import json
    import os
    from safetensors.torch import save_file
    from torch import nn
    from mindiesd import quantize
    from mindiesd.layers.quant import fp8_attention_forward, mx_quantize, mxfp8_matmul

    class Block(nn.Module):
        def __init__(self):
            super().__init__()
            self.up = nn.Linear(256, 512)
            self.attn = nn.Identity()

    g = torch.Generator().manual_seed(0)
    w = (torch.randn(512, 256, generator=g) * 0.05).to(torch.bfloat16).to(cuda)
    wq, ws = mx_quantize(w)
    bias = torch.randn(512, generator=g)
    rot = torch.linalg.qr(torch.randn(128, 128, generator=g))[0].to(torch.bfloat16).contiguous()
    weights = {"up.weight": wq.cpu(), "up.weight_scale": ws.view(torch.uint8).cpu().reshape(512, -1, 2).contiguous(),
               "up.bias": bias, "attn.q_rot": rot, "attn.k_rot": rot.clone()}
    des = {"model_quant_type": "W8A8_MXFP8", "up.weight": "W8A8_MXFP8", "attn.fa_q.scale": "FP8_DYNAMIC"}
    with open(os.path.join(tmp_path, "d.json"), "w") as f:
        json.dump(des, f)
    save_file(weights, os.path.join(tmp_path, "quant_model_weight_w8a8_mxfp8.safetensors"))
    model = quantize(Block(), os.path.join(str(tmp_path), "d.json")).to(cuda)
    x = torch.randn(3, 40, 256, generator=g).to(torch.bfloat16).to(cuda)
    got = model.up(x)
    xq, xs = mx_quantize(x.reshape(-1, 256))
    want = mxfp8_matmul(xq, xs, wq, ws, bias.to(cuda), torch.bfloat16, False).view(3, 40, 512)
    assert got.shape == (3, 40, 512) and torch.equal(got, want)
    q, k, v = (torch.randn(1, 2, 300, 128, generator=g).to(torch.bfloat16).to(cuda) for _ in range(3))
    a = model.attn.fa_quant(q, k, v, layout="BNSD")
    b = fp8_attention_forward(q, k, v, layout="BNSD", q_rot=rot.to(cuda), k_rot=rot.to(cuda))
    assert torch.equal(a, b)


@pytest.mark.parametrize("form", ["2d", "4d", "1d", "row_stride", "column_stride", "transposed"])
def test_linear_in_one_call_equals_quantise_then_multiply(cuda, form):
    """``mxfp8_linear`` on every form of x that needs another way to its rows, with and without SwiGLU and bias: the bits of
    ``mx_quantize`` followed by ``mxfp8_matmul``."""
    from mindiesd.layers.quant.mxfp8 import mx_quantize, mxfp8_linear, mxfp8_matmul
    g = torch.Generator().manual_seed(5)
    rnd = lambda *shape: torch.randn(shape, generator=g).to(torch.bfloat16).to(cuda)
    x = {"2d": lambda: rnd(70, 256), "4d": lambda: rnd(2, 5, 7, 256), "1d": lambda: rnd(256),
         "row_stride": lambda: rnd(70, 264)[:, :256], "column_stride": lambda: rnd(70, 512)[:, ::2],
         "transposed": lambda: rnd(7, 10, 256).transpose(0, 1)}[form]()
    wq, ws = mx_quantize(rnd(528, 256))
    bias = torch.randn(528, generator=g).to(torch.float16).to(cuda)
    xq, xs = mx_quantize(x.reshape(-1, 256))
    for swiglu in (False, True):
        for b in (None, bias):
            want = mxfp8_matmul(xq, xs, wq, ws, b, torch.float16, swiglu)
            got = mxfp8_linear(x, wq, ws.reshape(528, -1, 2), b, torch.float16, swiglu)
            assert got.shape == (*x.shape[:-1], want.shape[1]) and torch.equal(got.view(want.shape), want)


def test_linear_in_one_call_refuses_what_its_parts_refuse(cuda):
    import mindiesd
    from mindiesd.layers.quant.mxfp8 import mx_quantize, mxfp8_linear
    x = torch.ones(4, 256, dtype=torch.bfloat16, device=cuda)
    wq, ws = mx_quantize(x.repeat(2, 1))
    refused = mindiesd.ParametersInvalid
    for bad in (lambda: mxfp8_linear(x.cpu(), wq, ws), lambda: mxfp8_linear(x.float(), wq, ws),
                lambda: mxfp8_linear(x[:, :40], wq[:, :40], ws), lambda: mxfp8_linear(x[:, :160], wq[:, :160], ws),
                lambda: mxfp8_linear(x, wq[:, :128], ws), lambda: mxfp8_linear(x, wq[:4], ws[:4]),
                lambda: mxfp8_linear(x, wq, ws, out_dtype=torch.float32), lambda: mxfp8_linear(x, wq, ws, swiglu=True),
                lambda: mxfp8_linear(x, wq.cpu(), ws), lambda: mxfp8_linear(x, wq, ws, torch.ones(7, device=cuda))):
        with pytest.raises(refused):
            bad()
    with pytest.raises(RuntimeError):
        mxfp8_linear(x, wq, ws[:, :4])       # fewer scales than the weight has blocks
    for bad in (x[:0], torch.ones(1028, dtype=torch.bfloat16, device=cuda)[4:].view(4, 256)):     # empty; not 16-byte aligned
        for call in (lambda: mxfp8_linear(bad, wq, ws), lambda: mx_quantize(bad)):
            with pytest.raises(RuntimeError):
                call()
