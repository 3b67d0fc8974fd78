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
