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


# both sides of the lines in pairs, at weights of a few MB: Q4_K to Q6_K and Q8_0 together, Q8_0 alone, the other formats
@pytest.mark.parametrize("gu,dn,few", [(lib.TYPE_Q4_K, lib.TYPE_Q4_K, 40), (lib.TYPE_Q4_K, lib.TYPE_Q6_K, 40), (lib.TYPE_Q5_K, lib.TYPE_Q5_K, 40),
                                       (lib.TYPE_Q6_K, lib.TYPE_Q6_K, 40), (lib.TYPE_Q8_0, lib.TYPE_Q4_K, 40), (lib.TYPE_Q8_0, lib.TYPE_Q8_0, 64),
                                       (lib.TYPE_MXFP4, lib.TYPE_MXFP4, 20), (lib.TYPE_MXFP4, lib.TYPE_Q8_0, 20), (lib.TYPE_IQ3_S, lib.TYPE_IQ3_S, 20),
                                       (lib.TYPE_Q2_0, lib.TYPE_Q2_0, 20), (lib.TYPE_Q3_K, lib.TYPE_Q3_K, 20), (lib.TYPE_Q5_1, lib.TYPE_IQ4_XS, 20)])
def test_many_pairs_of_small_matrices_are_batched(gu, dn, few):
    n_experts = few // 4   # four rows an expert: past the line of lk_moe_grouped_pays in every format
    assert not path(gu, dn, few, 1, n_experts, 256, 256) & GROUPED
    assert path(gu, dn, few + 1, 1, n_experts, 256, 256) & GROUPED
    assert path(gu, dn, 6 * 128 // 2, 2, 128, 256, 256) & GROUPED


@pytest.mark.parametrize("wtype,tokens,topk,n_experts,hidden,ffn,grouped", [
    (lib.TYPE_Q5_K, 10, 8, 64, 2048, 1536, False), (lib.TYPE_Q5_K, 10, 8, 64, 2048, 2048, True), (lib.TYPE_Q5_K, 5, 8, 32, 2048, 1792, False),
    (lib.TYPE_Q5_K, 14, 8, 64, 1024, 1536, True), (lib.TYPE_Q5_K, 13, 8, 64, 1024, 1536, False), (lib.TYPE_Q5_K, 14, 8, 64, 1024, 1024, False),
    (lib.TYPE_Q8_0, 9, 8, 32, 2560, 1280, False), (lib.TYPE_Q8_0, 20, 8, 64, 2048, 768, True), (lib.TYPE_Q8_0, 19, 8, 64, 2048, 768, False),
    (lib.TYPE_Q8_0, 36, 8, 128, 512, 768, False)])
def test_large_matrices_are_batched_sooner_where_there_are_pairs_enough(wtype, tokens, topk, n_experts, hidden, ffn, grouped):
    assert bool(path(wtype, wtype, tokens, topk, n_experts, hidden, ffn) & GROUPED) == grouped


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,tiles", [
    (11, 2, 4, 3072, 1536, False), (22, 2, 8, 3072, 1536, True), (39, 2, 16, 3072, 256, False), (39, 2, 16, 1280, 256, True),
    (60, 4, 64, 1792, 1792, False), (105, 4, 64, 1792, 1792, True), (60, 4, 64, 1792, 1536, True), (107, 4, 128, 256, 1792, False),
    (107, 4, 128, 256, 1280, True), (88, 8, 128, 1536, 512, False), (110, 8, 128, 1536, 512, True)])
def test_short_q4k_runs_go_on_the_tiles_where_these_are_ahead(tokens, topk, n_experts, hidden, ffn, tiles):
    assert 9 <= lib.load().lk_moe_longest_run(tokens, topk, n_experts) < 20
    assert bool(path(lib.TYPE_Q4_K, lib.TYPE_Q4_K, tokens, topk, n_experts, hidden, ffn) & TILES) == tiles
