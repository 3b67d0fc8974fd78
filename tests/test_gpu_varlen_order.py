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
