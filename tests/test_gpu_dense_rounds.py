"""Dense attention at head dims 128 and 64 where the last round of workgroups is cut into half or quarter tiles
(fa16_split) or, over a few key tiles, workgroups keep their CU (fa16_loop_kernel): whole rounds before it or none, tiles per XCD at the edges of the rule, ragged query and key
lengths around the 64-, 128- and 256-row and the 128-key tiles, both layouts and types, and the key-padding mask.

Bounds against the float64 softmax of the same 16-bit operands: the query is rounded to 16 bits after scaling and a
probability before the second product (a relative u = 2^-9 for bf16, 2^-12 for fp16, each), the output once more; in the
2-norm 3 u covers their sum, an element lies within 16 u of the largest absolute value of v."""
import pytest
import torch

import mindiesd
from mindiesd.layers.flash_attn.hip_flash_attn import flash_attention

pytestmark = pytest.mark.gpu
U = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def reference(q, k, v, mask=None):
    out = []
    for b in range(q.shape[0]):
        for n in range(q.shape[1]):
            s = q[b, n].double() @ k[b, n].double().t() * q.shape[-1] ** -0.5
            if mask is not None:
                s = s.masked_fill(~mask[b].view(1, -1), float("-inf"))
            out.append(torch.softmax(s, -1) @ v[b, n].double())
    return torch.stack(out).reshape(q.shape)


def check(got, want, v, dtype):
    err = got.double() - want
    assert torch.isfinite(got).all()
    assert (err.norm() / want.norm()).item() <= 3 * U[dtype]
    assert err.abs().max().item() <= 16 * U[dtype] * v.abs().max().item()


# (batch, heads, q_len, kv_len), 2 to 9 rounds: even and odd numbers of key tiles, ragged rows, heads that change inside
# a workgroup's run, and the last key count of the rule
LOOP_CASES = [(1, 40, 4200, 385), (2, 20, 3328, 513), (1, 264, 600, 640), (3, 11, 8200, 767), (1, 536, 256, 768), (1, 523, 257, 500)]


@pytest.mark.parametrize("batch,heads,q_len,kv_len", LOOP_CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masked", [False, True])
def test_rows_in_a_loop(batch, heads, q_len, kv_len, dtype, masked):
    print("case", batch, heads, q_len, kv_len, dtype, masked, flush=True)
    g = torch.Generator(device="cuda").manual_seed(heads + q_len)
    q, k, v = (torch.randn((batch, s, heads, 128), generator=g, device="cuda").to(dtype) for s in (q_len, kv_len, kv_len))
    mask = torch.rand((batch, kv_len), generator=g, device="cuda") < 0.5 if masked else None
    m4 = None if mask is None else mask.view(batch, 1, 1, kv_len)
    want = reference(*(x.transpose(1, 2) for x in (q, k, v)), mask)
    got = mindiesd.attention_forward(q, k, v, attn_mask=m4, head_first=False)
    check(got.transpose(1, 2), want, v, dtype)


# heads x ceil(q_len / 256) tiles over 8 XCDs: tiles per XCD 1, 1, 8, 9, 16, 17 (no round before the last),
# 32 + 1, 32 + 8, 32 + 9, 32 + 16, 64 + 3
CASES = [(1, 1, 385), (3, 257, 512), (64, 129, 1000), (72, 200, 513), (43, 700, 641), (136, 256, 400), (8, 2300, 2100), (264, 300, 2050),
         (264, 193, 400), (160, 300, 577), (164, 511, 390), (128, 641, 700), (536, 65, 450)]


@pytest.mark.parametrize("heads,q_len,kv_len", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("d", [128, 64])
def test_cut_rounds(heads, q_len, kv_len, dtype, masked, d):
    if masked and q_len < 256:
        q_len += 256                      # key masks run on this kernel from 256 query rows on
    print("case", heads, q_len, kv_len, dtype, masked, d, flush=True)
    g = torch.Generator(device="cuda").manual_seed(heads + q_len)
    q, k, v = (torch.randn((1, heads, s, d), generator=g, device="cuda").to(dtype) for s in (q_len, kv_len, kv_len))
    mask = None
    if masked:
        mask = torch.rand((1, kv_len), generator=g, device="cuda") < 0.5
        mask[:, :70] = False              # the first groups of keys and all of a group's keys in the last tile hidden
        mask[:, kv_len - kv_len % 128 - 20:] = False
        mask[:, 200] = True
    want = reference(q, k, v, mask)
    m4 = None if mask is None else mask.view(1, 1, 1, kv_len)
    check(mindiesd.attention_forward(q, k, v, attn_mask=m4, head_first=True), want, v, dtype)
    t = [x.transpose(1, 2).contiguous() for x in (q, k, v)]
    check(mindiesd.attention_forward(*t, attn_mask=m4, head_first=False).transpose(1, 2), want, v, dtype)


# equal problems side by side: 32 + 1 and 32 + 12 tiles per XCD, 32 + 19, 64 + 2 with ragged rows, 64 without a rest and few keys
EQUAL = [(8, 8448, 640), (8, 11264, 1536), (8, 12800, 900), (264, 300, 450), (8, 16384, 512), (24, 1101, 1101)]


@pytest.mark.parametrize("heads,q_len,kv_len", EQUAL)
@pytest.mark.parametrize("d,dtype", [(128, torch.bfloat16), (128, torch.float16), (64, torch.float16)])
@pytest.mark.parametrize("masked", [False, True])
def test_equal_problems_have_equal_bits(monkeypatch, heads, q_len, kv_len, d, dtype, masked):
    """The heads of a call hold the same problem: whichever kind of tile computes a row, its output and log-sum-exp have the
    same bits, those of a launch in whole tiles of 256 rows."""
    g = torch.Generator(device="cuda").manual_seed(kv_len)
    q, k, v = (torch.randn((1, 1, s, d), generator=g, device="cuda").to(dtype).expand(1, heads, s, d).contiguous()
               for s in (q_len, kv_len, kv_len))
    mask = (torch.rand((1, 1, 1, kv_len), generator=g, device="cuda") < 0.5) if masked else None
    out, lse = flash_attention(q, k, v, d ** -0.5, return_lse=True, attn_mask=mask)
    assert torch.equal(out, out[:, :1].expand_as(out)) and torch.equal(lse, lse[:, :1].expand_as(lse))
    assert torch.equal(out, flash_attention(q, k, v, d ** -0.5, attn_mask=mask))
    monkeypatch.setenv("MINDIESD_DENSE_TILE_ROWS", "256")
    whole, whole_lse = flash_attention(q, k, v, d ** -0.5, return_lse=True, attn_mask=mask)
    assert torch.equal(out, whole) and torch.equal(lse, whole_lse)


# one whole round and a rest per XCD (1, 8, 9, 16 tiles, B x N 8) on few keys: the 4-wave kernel where the last 128-key tile is at
# most half full, below 449 keys for rests up to 8 and below 833 above; a second whole round, a full last tile: never
@pytest.mark.parametrize("q_len,kv_len,four_waves", [
    (8448, 385, True), (10240, 448, True), (10240, 449, False), (10496, 448, True), (12288, 448, True), (12288, 449, False),
    (10240, 576, False), (10496, 520, True), (12288, 832, True), (12288, 833, False), (12288, 900, False), (12544, 448, False),
    (8192, 448, False), (16640, 448, False)])
def test_kernel_of_one_round_and_a_rest(monkeypatch, q_len, kv_len, four_waves):
    """The two kernels add a row up in different orders, so their bits tell which one ran."""
    g = torch.Generator(device="cuda").manual_seed(q_len + kv_len)
    q, k, v = (torch.randn((1, 8, s, 128), generator=g, device="cuda").bfloat16() for s in (q_len, kv_len, kv_len))
    out = {}
    for rows in (None, "256", "128"):
        if rows:
            monkeypatch.setenv("MINDIESD_DENSE_TILE_ROWS", rows)
        out[rows] = mindiesd.attention_forward(q, k, v, head_first=True)
    assert not torch.equal(out["128"], out["256"])
    assert torch.equal(out[None], out["128" if four_waves else "256"])


@pytest.mark.parametrize("d", [128, 64])
def test_very_different_maxima(d):
    """Scores that differ by hundreds between the halves of every key tile, rows whose scores all lie far below zero, and a
    NaN and an infinity that stay in their rows."""
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((1, 4, s, d), generator=g, device="cuda").bfloat16() for s in (512, 640, 640))
    q[:, :, :, 0] = 4.0
    k[:, :, :, 0] = torch.where(torch.arange(640, device="cuda") % 128 < 64, -900.0, -300.0).view(1, 1, -1).bfloat16()
    q[:, 1, :, 0] = -4.0
    q[:, 2, :, 0] = torch.where(torch.arange(512, device="cuda") % 2 == 0, 4.0, -0.5).bfloat16()
    check(mindiesd.attention_forward(q, k, v, head_first=True), reference(q, k, v), v, torch.bfloat16)
    clean = mindiesd.attention_forward(q, k, v, head_first=True)
    q[0, 3, 17, 5] = float("nan")
    q[0, 3, 300, 5] = float("inf")
    out = mindiesd.attention_forward(q, k, v, head_first=True)
    bad = torch.zeros_like(out, dtype=torch.bool)
    bad[0, 3, 17] = bad[0, 3, 300] = True
    assert torch.isnan(out[bad]).all()
    assert torch.equal(out[~bad], clean[~bad])
