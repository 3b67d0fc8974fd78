"""Dense attention over at most 256 keys that stay in LDS (flash_attn_keys.hip), against the softmax in float64 on the same
inputs.  Tolerance: outputs and probabilities are rounded to 16 bits once each, the query after scaling once: relative error of
the whole tensor within 2 * 2^-9 (bf16; 2^-12 fp16) of it, and equal rows give equal bits wherever they lie."""
import pytest
import torch

pytestmark = pytest.mark.gpu

REL = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _exact(q, k, v, scale):
    """q [B,N,S,D], k / v [B,Nkv,K,D] -> output and log-sum-exp in float64 on the GPU."""
    rep = q.shape[1] // k.shape[1]
    k, v = (t.double().repeat_interleave(rep, 1).contiguous() for t in (k, v))
    s = torch.matmul(q.double(), k.transpose(-1, -2).contiguous()) * scale
    return torch.matmul(torch.softmax(s, -1), v), torch.logsumexp(s, -1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b, n, nkv, sq, skv, layout", [
    (1, 8, 8, 8192, 1, "BNSD"), (1, 8, 8, 8200, 31, "BSND"), (2, 12, 3, 2731, 32, "BNSD"), (1, 8, 2, 8161, 33, "BNSD"),
    (1, 16, 16, 4096, 64, "BSND"), (1, 24, 24, 2817, 65, "BNSD"), (2, 40, 40, 1025, 96, "BSND"), (1, 8, 8, 9000, 127, "BNSD"),
    (1, 8, 8, 8192, 128, "BNSD"), (1, 20, 4, 3300, 160, "BSND"), (1, 8, 8, 8193, 192, "BNSD"), (1, 8, 8, 8193, 193, "BSND"),
    (4, 33, 11, 512, 224, "BNSD"), (1, 8, 8, 8500, 225, "BNSD"), (1, 10, 10, 7001, 255, "BSND"), (8, 40, 8, 530, 256, "BNSD")])
def test_keys_in_lds_against_exact_softmax(cuda, b, n, nkv, sq, skv, layout, dtype):
    """Every number of 32-key blocks, whole and ragged; rows that end inside a wave's 32; workgroups that go from head to head."""
    from mindiesd.layers.flash_attn.hip_flash_attn import flash_attention
    assert b * n * ((sq + 31) // 32) >= 2048 and sq >= 512 and skv <= 256          # (the rule of the dispatch)
    g = torch.Generator(device=cuda).manual_seed(sq + skv)
    q, k, v = (torch.randn(b, h, s, 128, generator=g, device=cuda).to(dtype) for h, s in ((n, sq), (nkv, skv), (nkv, skv)))
    q[:, :, 100:200] = q[:, :, :100]
    view = (lambda t: t) if layout == "BNSD" else (lambda t: t.transpose(1, 2))
    inner = (lambda t: t) if layout == "BNSD" else (lambda t: t.transpose(1, 2).contiguous().transpose(1, 2))
    q, k, v = inner(q), inner(k), inner(v)
    out, lse = flash_attention(view(q), view(k), view(v), 0.0883883, layout, return_lse=True)
    out = view(out)
    want, want_lse = _exact(q, k, v, 0.0883883)
    assert ((out.double() - want).norm() / want.norm()).item() <= REL[dtype]
    # A score's error is the sum of 128 rounding errors of q * scale, each uniform within u of a product (u = REL / 2): standard
    # deviation u / sqrt(3) times the root of the products' squares, which for N(0, 1) inputs is 1 and at most 1.5; eight of them,
    # as a single key averages nothing out: 8 * 1.5 / sqrt(3) * REL / 2 = 3.5 * REL.
    assert (lse.double() - want_lse).abs().max().item() <= 3.5 * REL[dtype]
    assert torch.equal(out[:, :, 100:200], out[:, :, :100])


def test_scores_far_from_zero_and_no_finite_score(cuda):
    """Rows whose scores all lie hundreds below zero, keys that dominate, and a row of NaN that stays by itself."""
    from mindiesd.layers.flash_attn.hip_flash_attn import flash_attention
    g = torch.Generator(device=cuda).manual_seed(1)
    q, k, v = (torch.randn(1, 8, s, 128, generator=g, device=cuda).to(torch.bfloat16) for s in (8192, 77, 77))
    q[:, :, :64], k[:, :4] = 8.0, (k[:, :4].float() * 0.5 - 8.0).to(torch.bfloat16)
    k[:, 4:, 5] = 6.0
    nan_row = q.clone()
    nan_row[:, :, 70] = float("nan")
    out, got = (flash_attention(t, k, v, 128 ** -0.5) for t in (q, nan_row))
    want, _ = _exact(q, k, v, 128 ** -0.5)
    # (a score near 700 carries the query's rounding, 2^-9 of it, where the queries are not constant)
    assert ((out.double() - want)[:, :, :64].norm() / want[:, :, :64].norm()).item() <= 2.0 ** -6
    assert torch.isfinite(out.float()).all()
    assert torch.isnan(got[:, :, 70].float()).all()
    keep = torch.arange(8192, device=cuda) != 70
    assert torch.equal(got[:, :, keep], out[:, :, keep])
