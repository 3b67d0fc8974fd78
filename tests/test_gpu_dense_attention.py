"""GPU parity: the HIP flash-attention kernel behind attention_forward vs the CPU oracle
(restatement of the reference's attention_math).  Tolerance (bf16): max-abs <= 2e-2 and
cosine >= 0.9999; the reference's own fused-vs-fallback rule (data_compare) is checked as well."""
import pytest
import torch

from oracle.attention import attention_math, attention_math_rows, cosine, data_compare

pytestmark = pytest.mark.gpu

MAX_ABS = 2e-2
MIN_COS = 0.9999


@pytest.fixture(autouse=True, params=["auto", "256", "128"])
def dense_tile_rows(request, monkeypatch):
    """Every test of this file under the library's own choice between its 256-row (8 waves) and 128-row (4 waves)
    kernels at head_dim 128 - made from how the grid fills the chip - and with either forced."""
    if request.param == "auto":
        monkeypatch.delenv("MINDIESD_DENSE_TILE_ROWS", raising=False)
    else:
        monkeypatch.setenv("MINDIESD_DENSE_TILE_ROWS", request.param)


def _qkv(shape, seed, dtype=torch.bfloat16, mul=1.0, kv_shape=None):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(shape, generator=g) * mul).to(dtype)
    k = (torch.randn(kv_shape or shape, generator=g) * mul).to(dtype)
    v = (torch.randn(kv_shape or shape, generator=g) * mul).to(dtype)
    return q, k, v


def _check(out, ref, max_abs=MAX_ABS, min_cos=MIN_COS):
    err = (out.float() - ref.float()).abs().max().item()
    cos = cosine(out, ref)
    assert err <= max_abs, f"max-abs {err}"
    assert cos >= min_cos, f"cosine {cos}"


@pytest.mark.parametrize("head_first", [True, False])
@pytest.mark.parametrize("s", [1, 31, 128, 300, 1024, 1153])
def test_small_shapes_both_layouts(cuda, head_first, s):
    import mindiesd
    shape = (2, 3, s, 128) if head_first else (2, s, 3, 128)
    q, k, v = _qkv(shape, seed=s)
    ref = attention_math(q, k, v, None, 128 ** -0.5, head_first=head_first)
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), head_first=head_first)
    assert out.shape == q.shape and out.dtype == q.dtype
    _check(out.cpu(), ref)


def test_config1_full(cuda):
    """B1 N12 S4096 D128 bf16 N(0,1), scale 1/sqrt(128): oracle evaluated whole."""
    import mindiesd
    q, k, v = _qkv((1, 12, 4096, 128), seed=1)
    ref = attention_math(q, k, v, None, 128 ** -0.5, head_first=True)
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), head_first=True).cpu()
    _check(out, ref)
    # the reference's own rule at its own thresholds (tests/utils/utils/precision_compare.py:89: relative to
    # max(1, |golden|) within 1e-3 for 99.9 % of the elements, never above 0.1); the share that passes is printed
    assert data_compare(out, ref), "reference's data_compare rule"
    diff = (out.float() - ref.float()).abs() / ref.float().abs().clamp(min=1.0)
    print(f"config 1: data_compare pass fraction at the reference's threshold 1e-3: {float((diff <= 1e-3).float().mean()):.5f}, "
          f"largest relative difference {float(diff.max()):.4f}")


def test_fp16(cuda):
    import mindiesd
    q, k, v = _qkv((1, 777, 4, 128), seed=5, dtype=torch.float16)
    ref = attention_math(q, k, v, None, 0.11, head_first=False)
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), scale=0.11).cpu()
    _check(out, ref, max_abs=2e-3, min_cos=0.99999)
    assert data_compare(out, ref), "reference's data_compare rule"


def test_cross_attention_and_gqa(cuda):
    from mindiesd.layers.flash_attn.hip_flash_attn import flash_attention
    q, k, v = _qkv((1, 8, 500, 128), seed=7, kv_shape=(1, 2, 1300, 128))
    ref = attention_math(q, k.repeat_interleave(4, dim=1), v.repeat_interleave(4, dim=1), None, 128 ** -0.5, True)
    out, lse = flash_attention(q.to(cuda), k.to(cuda), v.to(cuda), 128 ** -0.5, "BNSD", return_lse=True)
    _check(out.cpu(), ref)
    s = (q.float() @ k.repeat_interleave(4, dim=1).float().transpose(-1, -2)) * 128 ** -0.5
    # the kernel folds scale*log2(e) into Q in bf16, which moves the scores by ~2^-9 relative
    assert (lse.cpu() - torch.logsumexp(s, dim=-1)).abs().max() < 5e-3


def test_strided_views_run_in_place(cuda):
    """BSND tensors viewed as BNSD (and the reverse) must give the same result without a copy."""
    import mindiesd
    q, k, v = _qkv((1, 640, 5, 128), seed=9)
    qc, kc, vc = q.to(cuda), k.to(cuda), v.to(cuda)
    a = mindiesd.attention_forward(qc, kc, vc, head_first=False)
    b = mindiesd.attention_forward(qc.transpose(1, 2), kc.transpose(1, 2), vc.transpose(1, 2), head_first=True)
    assert torch.equal(a, b.transpose(1, 2))
    for mode in ("static", "manual"):
        c = mindiesd.attention_forward(qc, kc, vc, opt_mode=mode, op_type="ascend_laser_attention", layout="BSH")
        assert torch.equal(a, c)


def test_rising_row_maxima_vs_fp64(cuda):
    """Late keys raise the row maxima far above what the first tiles saw, so the lazily updated
    softmax reference maximum has to move several times.  Checked against an fp64 evaluation: in
    this regime the bf16-rounded scores of the reference's unfused path are themselves too coarse
    to serve as the yardstick."""
    import mindiesd
    from oracle.attention import attention_fp64
    q, k, v = _qkv((1, 2, 2048, 128), seed=11, mul=1.5)
    k[:, :, 700:1400] *= 2.0
    k[:, :, 1400:] *= 3.0
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), head_first=True).cpu()
    for n in range(2):
        ref = attention_fp64(q[0, n], k[0, n], v[0, n], 128 ** -0.5)
        # scores reach |s| ~ 40 here; the kernel (like the reference, attention_func.py:40) rounds the
        # scaled queries to bf16, i.e. moves such scores by up to ~0.1, hence the wider max-abs bound
        _check(out[0, n], ref, max_abs=1e-1)


def _far_below_zero(shape, seed, dtype=torch.bfloat16):
    """q near +8, k near -8 in every component: every score of a row lies hundreds of units below zero, so the first
    key tile already moves the running maximum far down (2^-delta overflows there); v is N(0, 1)."""
    g = torch.Generator().manual_seed(seed)
    q = (8.0 + 0.5 * torch.randn(shape, generator=g)).to(dtype)
    k = (-8.0 + 0.5 * torch.randn(shape, generator=g)).to(dtype)
    v = torch.randn(shape, generator=g).to(dtype)
    return q, k, v


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("s", [300, 1153])
def test_scores_far_below_zero(cuda, s, d):
    """Checked against an fp64 evaluation on the queries as the kernel uses them (scaled by scale * log2(e) and
    rounded to bf16, the reference rounds q * scale as well, attention_func.py:40): at |s| ~ 700 the bf16-rounded
    scores of the reference's unfused path are too coarse to serve as the yardstick."""
    import math
    import mindiesd
    from oracle.attention import attention_fp64
    q, k, v = _far_below_zero((1, 2, s, d), seed=s + d)
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), head_first=True).cpu()
    assert not torch.isnan(out.float()).any()
    qs = (q.float() * (d ** -0.5 * math.log2(math.e))).to(torch.bfloat16)
    for n in range(2):
        _check(out[0, n], attention_fp64(qs[0, n], k[0, n], v[0, n], math.log(2.0)))


def test_config2_head_subset(cuda):
    """Wan2.1-1.3B shape (S=32760): full GPU run, oracle on a row sample of two heads."""
    import mindiesd
    q, k, v = _qkv((1, 12, 32760, 128), seed=2, mul=0.5)
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), head_first=True).cpu()
    for head in (0, 11):
        for rows in (slice(0, 512), slice(32248, 32760)):
            ref = attention_math_rows(q[:, head:head + 1], k[:, head:head + 1], v[:, head:head + 1], 128 ** -0.5,
                                      row_chunk=512, q_rows=rows)
            _check(out[:, head:head + 1, rows], ref)


def test_unfused_path_matches_oracle(cuda):
    import mindiesd
    q, k, v = _qkv((1, 200, 2, 128), seed=13)
    mask = torch.rand(200, 200) > 0.3
    mask[:, 0] = True
    ref = attention_math(q, k, v, mask, 0.09, head_first=False)
    out = mindiesd.attention_forward(q.to(cuda), k.to(cuda), v.to(cuda), attn_mask=mask.to(cuda), scale=0.09, fused=False)
    _check(out.cpu(), ref)


def test_errors(cuda):
    import mindiesd
    from mindiesd import ParametersInvalid
    q = torch.randn(1, 64, 2, 128, dtype=torch.bfloat16, device=cuda)
    with pytest.raises(ParametersInvalid):
        mindiesd.attention_forward(q, q, q, opt_mode="fastest")
    with pytest.raises(ParametersInvalid):
        mindiesd.attention_forward(q, q, q, scale=1)
    with pytest.raises(ParametersInvalid):
        mindiesd.attention_forward(q[0], q, q)
    with pytest.raises(ParametersInvalid):
        mindiesd.attention_forward(q.float(), q.float(), q.float())
    with pytest.raises(ParametersInvalid):
        mindiesd.attention_forward(q[..., :68], q[..., :68], q[..., :68])   # head_dim must be a multiple of 8
    with pytest.raises(ParametersInvalid):
        mindiesd.attention_forward(q, q, q, opt_mode="manual", op_type="nope")


@pytest.mark.parametrize("s", [128, 300, 1153])
def test_tail_tile_reads_nothing_past_the_sequence(cuda, s):
    """K and V are views into slabs whose rows past the sequence hold NaN: the last key tile must take those rows
    as zeros (the kernels rely on the range check of their buffer descriptors for that), otherwise 0 * NaN from
    the second product shows up in the output."""
    import mindiesd
    q, k, v = _qkv((1, 2, s, 128), seed=s + 7)
    slabs = []
    for t in (k, v):
        slab = torch.full((1, 2, s + 256, 128), float("nan"), dtype=torch.bfloat16, device=cuda)
        slab[:, :, :s] = t.to(cuda)
        slabs.append(slab[:, :, :s])
    ref = attention_math(q, k, v, None, 128 ** -0.5, head_first=True)
    out = mindiesd.attention_forward(q.to(cuda), slabs[0], slabs[1], head_first=True).cpu()
    assert not out.isnan().any()
    _check(out, ref)
    keep = torch.ones(s, s, dtype=torch.bool)
    keep[:, s // 2] = False
    ref = attention_math(q, k, v, keep, 128 ** -0.5, head_first=True)
    out = mindiesd.attention_forward(q.to(cuda), slabs[0], slabs[1], attn_mask=keep.to(cuda), head_first=True).cpu()
    assert not out.isnan().any()
    _check(out, ref)


class _Tokens(torch.Tensor):
    pass


@pytest.mark.parametrize("layout", ["BNSD", "BSND"])
@pytest.mark.parametrize("strided", [False, True])
def test_a_query_of_a_tensor_subclass_gives_a_plain_output(cuda, layout, strided):
    """Dense and FP8 attention: the type of the output does not follow the query's class, its bits are those of a plain query."""
    from mindiesd.layers.flash_attn.hip_flash_attn import flash_attention
    from mindiesd.layers.quant.fp8_attention import fp8_attention_forward
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(1, 130, 2, 256, generator=g).to(torch.bfloat16).to(cuda) for _ in range(3))
    q, k, v = (x[..., ::2] if strided else x[..., :128] for x in (q, k, v))
    for attend in (lambda t: flash_attention(t, k, v, 0.1, layout), lambda t: fp8_attention_forward(t, k, v, 0.1, layout)):
        got = attend(q.as_subclass(_Tokens))
        assert type(got) is torch.Tensor and got.is_contiguous() and torch.equal(got, attend(q))
