"""Causal attention whose last key tiles some waves of a workgroup do not see (fa_fwd16_kernel, general mode): the diagonal on
either side of a 128-key tile and of a wave's 32 rows, more queries than keys and fewer, dense and packed, against the softmax in
float64.  Tolerance: relative error of the tensor within 2^-8 (outputs, probabilities and scaled queries are rounded to bf16
once each)."""
import pytest
import torch

import mindiesd
from mindiesd.layers.flash_attn.hip_flash_attn import flash_attention

pytestmark = pytest.mark.gpu


def _exact(q, k, v, scale):
    """q [N,S,D], k / v [N,K,D], causal aligned to the bottom-right corner; rows that see no key are zero."""
    sq, skv = q.shape[1], k.shape[1]
    seen = torch.ones(sq, skv, dtype=torch.bool, device=q.device).tril(skv - sq)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * scale
    p = torch.softmax(s.masked_fill(~seen, float("-inf")), -1)
    return torch.matmul(torch.where(seen.any(-1)[:, None], p, torch.zeros_like(p)), v.double())


SHAPES = [(256, 385), (256, 512), (300, 427), (300, 428), (513, 513), (513, 514), (700, 669), (700, 668), (640, 512), (900, 401),
          (512, 640), (512, 607), (512, 609), (1024, 1024)]


@pytest.mark.parametrize("sq, skv", SHAPES)
def test_dense(cuda, sq, skv):
    g = torch.Generator(device=cuda).manual_seed(sq + skv)
    # (enough heads for the 8-wave kernel: grids of 129 to 256 workgroups of 256 rows)
    n = -(-160 // -(-sq // 256))
    q, k, v = (torch.randn(1, n, s, 128, generator=g, device=cuda).to(torch.bfloat16) for s in (sq, skv, skv))
    out = flash_attention(q, k, v, 0.09, causal=True)[0]
    want = _exact(q[0], k[0], v[0], 0.09)
    assert ((out.double() - want).norm() / want.norm()).item() <= 2.0 ** -8
    if sq > skv:
        assert not out[:, :sq - skv].any()


@pytest.mark.parametrize("on_gpu", [False, True])
def test_packed(cuda, on_gpu):
    g = torch.Generator(device=cuda).manual_seed(3)
    cu = [[0], [0]]
    for shape in SHAPES:
        for c, s in zip(cu, shape):
            c.append(c[-1] + s)
    q, k, v = (torch.randn(c[-1], 3, 128, generator=g, device=cuda).to(torch.bfloat16) for c in (cu[0], cu[1], cu[1]))
    tables = [torch.tensor(c, dtype=torch.int32, device=cuda) if on_gpu else c for c in cu]
    out = mindiesd.attention_forward_varlen(q, k, v, *tables, softmax_scale=0.09, causal=True)
    for i in range(len(SHAPES)):
        rows, keys = slice(cu[0][i], cu[0][i + 1]), slice(cu[1][i], cu[1][i + 1])
        want = _exact(*(x.transpose(0, 1).contiguous() for x in (q[rows], k[keys], v[keys])), 0.09)
        assert ((out[rows].transpose(0, 1).double() - want).norm() / want.norm()).item() <= 2.0 ** -8
