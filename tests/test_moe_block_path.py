"""Which launches an expert block is made of (lk_moe_block_path): a rule on the host, no GPU."""
import pytest

from loken_amd import lib

GROUPED, TILES = lib.MOE_GROUPED, lib.MOE_TILES


def path(gu, dn, tokens, topk, n_experts, hidden, ffn):
    return lib.load().lk_moe_block_path(gu, dn, tokens, topk, n_experts, hidden, ffn)


@pytest.mark.parametrize("gu,dn", [(lib.TYPE_Q4_0, lib.TYPE_Q4_0), (lib.TYPE_Q4_1, lib.TYPE_Q4_1), (lib.TYPE_Q8_0, lib.TYPE_Q4_0),
                                   (lib.TYPE_Q4_0, lib.TYPE_Q4_K), (lib.TYPE_Q4_1, lib.TYPE_Q5_K)])
@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn", [(12, 2, 8, 256, 256), (16, 2, 8, 1024, 512), (24, 2, 8, 1024, 512), (20, 2, 8, 2048, 512),
                                                              (6, 4, 8, 512, 256), (25, 8, 60, 512, 256)])
def test_formats_without_a_mat_vec_per_pair_are_batched_from_three_rows_an_expert(gu, dn, tokens, topk, n_experts, hidden, ffn):
    assert path(gu, dn, tokens, topk, n_experts, hidden, ffn) & GROUPED
    assert not path(gu, dn, tokens // 4, topk, n_experts, hidden, ffn) & GROUPED   # fewer rows: refused, as ever
