"""Packed sequences of unequal length, taken longest first by at most 64 of them and in descending tile order beyond
(fa16_find_work): equal lengths among them, sequences without queries or keys, key counts in another order than the query
counts, each kernel width, host lists and device tables.  Every row is compared with dense attention over its own sequence in
float64; bound as in test_gpu_dense_rounds.py."""
import pytest
import torch

import mindiesd
from test_gpu_dense_rounds import check, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [128, 64, 96, 256])
@pytest.mark.parametrize("nseq", [2, 7, 64, 65])
@pytest.mark.parametrize("on_gpu", [False, True])
def test_longest_first(nseq, d, on_gpu):
    lens_q = [(257, 900, 1300, 256, 900, 511, 1)[i % 7] for i in range(nseq)]
    lens_k = [(700, 400, 513, 1500, 400, 0, 640)[i % 7] for i in range(nseq)]
    if nseq > 8:
        lens_q[8], lens_q[nseq - 1] = 0, 3000
    cu_q, cu_k = [0], [0]
    for a, b in zip(lens_q, lens_k):
        cu_q.append(cu_q[-1] + a)
        cu_k.append(cu_k[-1] + b)
    g = torch.Generator(device="cuda").manual_seed(nseq)
    q, k, v = (torch.randn((s, 2, d), generator=g, device="cuda").bfloat16() for s in (cu_q[-1], cu_k[-1], cu_k[-1]))
    cus = [torch.tensor(c, dtype=torch.int32, device="cuda") if on_gpu else c for c in (cu_q, cu_k)]
    out = mindiesd.attention_forward_varlen(q, k, v, *cus)
    for i in range(nseq):
        part = out[cu_q[i]:cu_q[i + 1]]
        ks = slice(cu_k[i], cu_k[i + 1])
        if lens_k[i] == 0:
            assert not part.any()
        elif lens_q[i]:
            want = reference(*(x.transpose(0, 1).unsqueeze(0) for x in (q[cu_q[i]:cu_q[i + 1]], k[ks], v[ks])))
            check(part.transpose(0, 1).unsqueeze(0), want, v[ks], torch.bfloat16)


@pytest.mark.parametrize("table, total, max_q, covered", [
    ([0, 40, 100], 100, None, (0, 100)),             # all rows
    ([0, 40, 97], 100, None, (0, 97)),               # a rest, inside a workgroup's rows
    ([33, 33, 64, 64], 97, None, (33, 64)),          # a gap on either side, empty sequences
    ([0, 0], 70, None, (0, 0)),                      # nothing
    ([0, 60, 40, 100], 100, None, (0, 0)),           # decreasing: sequences overlap
    ([-5, 40, 100], 100, None, (0, 0)),              # outside of the tensor
    ([0, 40, 101], 100, None, (0, 0)),
    ([0, 40, 100], 100, 59, (0, 0)),                 # a sequence longer than the longest one named
    ([0, 40, 100], 100, 60, (0, 100)),
    (list(range(0, 2001, 4)), 2003, None, (0, 2000)),  # more sequences than a workgroup has threads
])
def test_rows_outside_of_a_device_table_are_cleared(cuda, table, total, max_q, covered):
    """The launch that builds the table clears exactly the rows that no sequence covers, and every row when the table is not one
    that the attention kernels cover whole; the table itself is that of mindiesd_varlen_meta."""
    from mindiesd.layers.flash_attn.hip_flash_attn import _varlen_meta
    cu = torch.tensor(table, dtype=torch.int32, device=cuda)
    out = torch.ones(total, 3, 24, dtype=torch.float16, device=cuda)
    meta, *_ = _varlen_meta(cu, cu, total, total, cu.device, max_q, None, out)
    want, *_ = _varlen_meta(cu, cu, total, total, cu.device, max_q, None)
    assert torch.equal(meta, want)
    assert (out[covered[0]:covered[1]] == 1).all()
    assert not out[:covered[0]].any() and not out[covered[1]:].any()


@pytest.mark.parametrize("heads, d, total", [(1, 8, 12290), (1, 128, 769), (3, 24, 1400), (24, 128, 40), (300, 128, 9)])
@pytest.mark.parametrize("where", ["none", "all", "tail", "head", "inside", "backwards"])
def test_rows_outside_of_a_device_table_in_every_share(cuda, heads, d, total, where):
    """The same over several workgroups' shares of the output: 4096, 256, 456 and 11 rows, one row; covered rows that end at a
    share's edge and one row beside it."""
    from mindiesd.layers.flash_attn.hip_flash_attn import _varlen_meta
    share = -(-65536 // (2 * heads * d))
    table = {"none": [0, 0], "all": [0, total // 2, total], "tail": [share, total], "head": [0, 1, total - 1],
             "inside": [share - 1, share + 1, 2 * share], "backwards": [0, total, total - 1]}[where]
    first, last = (0, 0) if where == "backwards" else (table[0], table[-1])
    cu = torch.tensor(table, dtype=torch.int32, device=cuda)
    guard = torch.ones(total + 8, heads, d, dtype=torch.bfloat16, device=cuda)
    _varlen_meta(cu, cu, total, total, cu.device, None, None, guard[4:total + 4])
    assert 2 * share < total and (guard[:4] == 1).all() and (guard[total + 4:] == 1).all()
    out = guard[4:total + 4]
    assert (out[first:last] == 1).all() and not out[:first].any() and not out[last:].any()
