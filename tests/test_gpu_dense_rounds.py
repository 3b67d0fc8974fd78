"""Dense attention at head dims 128 and 64 where the last round of workgroups is cut into half or quarter tiles (fa16_split) or,
over a few key tiles, workgroups keep their CU (fa16_loop_kernel): whole rounds before it or none, tiles per XCD at the edges of
the rules, ragged query and key lengths around the 64-, 128- and 256-row and the 128-key tiles, both layouts and types, the
key-padding mask, and the bits of equal rows.

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


def kind(problems, q_len, kv_len, d=128, masked=False):
    """What runs a dense call without or with a key mask, as the library's dispatch has it: "loop", "4 waves", or the number of
    parts a tile of the last round is cut into (0: whole tiles)."""
    per_xcd = -(-problems * -(-q_len // 256) // 8)
    rounds, rest = divmod(per_xcd, 32)
    parts = 0 if rest == 0 or rest > 16 or rounds >= 16 else 2 if rest > 8 else 4
    keys64 = -(-kv_len // 64)
    if d == 128 and kv_len <= 768 and rounds >= (8 if parts else 2):
        return "loop"
    if not masked and rounds == 1 and parts and (kv_len < 1280 and parts == 2 if d == 64 else
                                                 keys64 % 2 and keys64 <= (13 if parts == 2 else 7)):
        return "4 waves"
    return parts


# (batch, heads, heads of k and v, q_len, kv_len), 2 to 8 rounds: 4, 5 and 6 key tiles, ragged rows, batch entries and (shared)
# heads that change inside a workgroup's run, the first and the last key count of the rule, eight rounds and a rest
LOOP_CASES = [(1, 40, 40, 4200, 385), (2, 21, 7, 4097, 513), (1, 225, 45, 600, 640), (3, 11, 11, 5400, 767), (1, 680, 68, 250, 768),
              (1, 350, 350, 257, 500), (1, 2100, 210, 256, 600)]


@pytest.mark.parametrize("batch,heads,kv_heads,q_len,kv_len", LOOP_CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masked", [False, True])
def test_rows_in_a_loop(batch, heads, kv_heads, q_len, kv_len, dtype, masked):
    """Output and log-sum-exp.  Bound of the latter: a score moves by at most u times the sum of its products' absolute values
    (the query's second rounding), the log-sum-exp by at most the largest of these, plus the 32-bit sums."""
    if masked and q_len < 256:
        q_len = 256                       # key masks run on this kernel from 256 query rows on
    assert kind(batch * heads, q_len, kv_len, masked=masked) == "loop"
    g = torch.Generator(device="cuda").manual_seed(heads + q_len)
    q, k, v = (torch.randn((batch, s, h, 128), generator=g, device="cuda").to(dtype)
               for s, h in ((q_len, heads), (kv_len, kv_heads), (kv_len, kv_heads)))
    mask = torch.rand((batch, kv_len), generator=g, device="cuda") < 0.5 if masked else None
    got, lse = flash_attention(q, k, v, 128 ** -0.5, layout="BSND", return_lse=True,
                               attn_mask=None if mask is None else mask.view(batch, 1, 1, kv_len))
    qt, kt, vt = (x.transpose(1, 2).repeat_interleave(heads // x.shape[2], 1) for x in (q, k, v))
    check(got.transpose(1, 2), reference(qt, kt, vt, mask), v, dtype)
    for b, n in {(0, 0), (batch - 1, heads // 2), (batch - 1, heads - 1)}:
        qd, kd = qt[b, n].double(), kt[b, n].double()
        s, slack = qd @ kd.t() * 128 ** -0.5, (qd.abs() @ kd.abs().t() * 128 ** -0.5).amax(-1) * U[dtype] + 1e-5
        want = torch.logsumexp(s if mask is None else s.masked_fill(~mask[b].view(1, -1), float("-inf")), -1)
        assert ((lse[b, n].double() - want).abs() <= slack).all()


# heads, q_len, kv_len, parts; heads x ceil(q_len / 256) tiles over 8 XCDs: tiles per XCD 1, 1, 8, 9, 16, 16, 17, 9 (no round
# before the last), 64 + 2, 32 + 1, 32 + 8, 32 + 9, 32 + 16, 64 + 3
CASES = [(1, 1, 385, 4), (3, 257, 512, 4), (64, 129, 1000, 4), (72, 200, 513, 2), (42, 700, 641, 2), (128, 250, 400, 2),
         (136, 256, 400, 0), (8, 2300, 2100, 2), (264, 300, 2050, 4), (264, 193, 500, 4), (160, 300, 577, 4), (164, 511, 1300, 2),
         (128, 641, 1400, 2), (536, 65, 450, 4)]


@pytest.mark.parametrize("heads,q_len,kv_len,parts", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("d", [128, 64])
def test_cut_rounds(heads, q_len, kv_len, parts, dtype, masked, d):
    if masked and q_len < 256:
        q_len = 256                       # key masks run on this kernel from 256 query rows on
    assert kind(heads, q_len, kv_len, d, masked) == parts
    g = torch.Generator(device="cuda").manual_seed(heads + q_len)
    q, k, v = (torch.randn((1, heads, s, d), generator=g, device="cuda").to(dtype) for s in (q_len, kv_len, kv_len))
    mask = None
    if masked:
        mask = torch.rand((1, kv_len), generator=g, device="cuda") < 0.5
        mask[:, :70] = False              # the first half of the first key tile and the last keys hidden
        mask[:, kv_len - kv_len % 128 - 20:] = False
        mask[:, 200] = True
    want = reference(q, k, v, mask)
    m4 = None if mask is None else mask.view(1, 1, 1, kv_len)
    check(mindiesd.attention_forward(q, k, v, attn_mask=m4, head_first=True), want, v, dtype)
    t = [x.transpose(1, 2).contiguous() for x in (q, k, v)]
    check(mindiesd.attention_forward(*t, attn_mask=m4, head_first=False).transpose(1, 2), want, v, dtype)


# the cut ends at 16 whole rounds: 15 rounds and 16 tiles per XCD, 16 rounds and one (key heads shared by 128 and 152 heads)
@pytest.mark.parametrize("heads,kv_heads,parts", [(3968, 31, 2), (4104, 27, 0)])
@pytest.mark.parametrize("d", [128, 64])
def test_last_cut_round(heads, kv_heads, parts, d):
    assert kind(heads, 70, 900, d) == parts
    g = torch.Generator(device="cuda").manual_seed(heads)
    q, k, v = (torch.randn((1, n, s, d), generator=g, device="cuda").bfloat16()
               for n, s in ((heads, 70), (kv_heads, 900), (kv_heads, 900)))
    got = flash_attention(q, k, v, d ** -0.5)
    some = torch.arange(0, heads, 31, device="cuda")
    kv = some // (heads // kv_heads)
    check(got[:, some], reference(q[:, some], k[:, kv], v[:, kv]), v, torch.bfloat16)


# equal problems side by side: 32 + 1 and 32 + 12 tiles per XCD, 32 + 18, 64 + 2 with ragged rows, 64 without a rest and few keys
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
