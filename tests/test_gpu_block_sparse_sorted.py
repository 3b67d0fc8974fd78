"""Block-sparse attention of small masks: one workgroup per mask row, the longest lists of each XCD first
(bsa_sorted_lists_kernel).  The order in which workgroups start changes no bit of a row, so the result equals the list
kernel's on lists built by mask_to_index; the paired kernel, which such masks no longer reach through the Python
functions, runs the cases of its own file again with the dispatch replaced."""
import pytest
import torch

import test_gpu_block_sparse_paired as paired_cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, qb, kb", [
    (1, 1, 1),            # one row: seven of eight runs are empty
    (1, 7, 64), (3, 3, 65), (2, 8, 127), (1, 17, 128), (1, 9, 129), (2, 5, 300),   # words and pairs of words of a mask row
    (5, 67, 70),          # rows that do not divide by the XCDs, four rows of a wave at a time with a remainder
    (8, 96, 40),          # the most rows that take this way: runs of 96
])
def test_equals_the_lists_in_natural_order(cuda, n, qb, kb):
    from mindiesd.layers.flash_attn import rainfusion as rf
    g = torch.Generator().manual_seed(1000 * n + 10 * qb + kb)
    sq, skv = 128 * qb - 37, 128 * kb - 100
    q, k, v = (torch.randn(1, n, s, 128, generator=g).to(torch.bfloat16).to(cuda) for s in (sq, skv, skv))
    mask = torch.rand(1, n, qb, kb, generator=g) < torch.rand(1, n, qb, 1, generator=g)     # rows of every length
    mask[:, :, qb // 2] = False
    mask[:, :, 0] = True
    out, lse = rf.block_sparse_attention_mask(q, k, v, mask.to(cuda), 0.09, return_lse=True)
    idx, cnt = rf.mask_to_lists(mask.to(cuda))
    want, want_lse = rf.block_sparse_attention_lists(q, k, v, idx, cnt, 0.09, return_lse=True)
    assert torch.equal(out, want) and torch.equal(lse, want_lse)


class _Paired:
    """The library with the mask entry point answered by the paired one."""

    def __init__(self, lib):
        self._lib = lib

    def __getattr__(self, name):
        return getattr(self._lib, name.replace("attention_mask_fwd", "attention_paired_fwd"))


@pytest.mark.parametrize("case, args", [
    ("test_paired_vs_oracle_and_lists", (1100, 2, 2, torch.bfloat16)), ("test_paired_vs_oracle_and_lists", (2048, 4, 2, torch.float16)),
    ("test_paired_vs_oracle_and_lists", (1500, 1, 1, torch.float16)), ("test_paired_vs_oracle_and_lists", (130, 2, 1, torch.bfloat16)),
    ("test_paired_scores_far_below_zero", ()), ("test_paired_bsnd_cross_lengths_and_full_mask", ()),
    ("test_paired_with_token_order_matches_explicit_permutation", ())])
def test_paired_kernel_on_small_masks(cuda, monkeypatch, case, args):
    from mindiesd import _native
    monkeypatch.setattr(_native, "_lib", _Paired(_native.lib()))
    getattr(paired_cases, case)(cuda, *args)


@pytest.mark.parametrize("n, qb, kb, lists", [
    (8, 96, 64, True), (8, 97, 64, False),            # keys that stay in the L2: by the rows
    (8, 64, 64, True), (8, 64, 65, False),            # 256 pairs, one whole round
    (4, 96, 65, True), (4, 97, 65, False),            # 192 pairs, and 196
    (6, 85, 65, True), (8, 80, 96, True), (8, 81, 96, False),   # odd rows: 258 pairs; 320; 328
    (4, 96, 96, True), (4, 96, 97, False),
    (2, 128, 97, True), (1, 255, 130, True), (2, 129, 97, False),   # 128 pairs; 130
])
def test_which_kernel_a_mask_takes(cuda, monkeypatch, n, qb, kb, lists):
    """The lines of the dispatch, told by the bits: the two kernels add a row's key blocks up in different orders."""
    from mindiesd import _native
    from mindiesd.layers.flash_attn import rainfusion as rf
    g = torch.Generator(device="cuda").manual_seed(100 * qb + kb)
    q, k, v = (torch.randn(1, n, s, 128, generator=g, device=cuda).to(torch.bfloat16) for s in (128 * qb, 128 * kb, 128 * kb))
    mask = torch.rand(1, n, qb, kb, generator=g, device=cuda) < 0.3
    got = rf.block_sparse_attention_mask(q, k, v, mask, 0.09)
    listed = rf.block_sparse_attention_lists(q, k, v, *rf.mask_to_lists(mask), 0.09)
    monkeypatch.setattr(_native, "_lib", _Paired(_native.lib()))
    paired = rf.block_sparse_attention_mask(q, k, v, mask, 0.09)
    assert not torch.equal(listed, paired)
    assert torch.equal(got, listed if lists else paired)
