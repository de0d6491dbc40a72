"""Where the lines between kernels lie: answers of the library's rules at both sides of each, without a GPU."""
import pytest

from imparo_amd.kernels import library


@pytest.mark.parametrize("streams,width,top,pays", [
    (1, 4096, 0, 1), (2, 4096, 0, 1), (3, 1024, 0, 1), (3, 1280, 0, 0), (4, 1024, 0, 1), (4, 1280, 0, 0), (4, 4096, 0, 0),
    (1, 2048, 1, 1), (1, 2304, 1, 0), (2, 2048, 8, 1), (2, 2304, 8, 0), (4, 1024, 8, 1), (3, 1280, 2, 0)])
def test_a_step_norm_without_a_router(streams, width, top, pays):
    assert library().imparo_stream_step_takes(8, streams, width, 0 if top else 1, top)
    assert library().imparo_stream_step_pays(streams, width, top) == pays


@pytest.mark.parametrize("tokens,outputs,top,k,pays", [
    (129, 8, 1, 128, 1), (12288, 9, 1, 8192, 1), (12289, 9, 1, 4096, 1), (12289, 9, 1, 4224, 0), (16384, 8, 2, 8192, 1),
    (4096, 16, 1, 8192, 1), (8192, 16, 1, 4096, 1), (8192, 16, 1, 8192, 0), (8192, 16, 4, 8192, 1), (8193, 21, 1, 1280, 1), (8193, 21, 1, 1408, 0),
    (8193, 21, 2, 3072, 0), (129, 24, 4, 128, 1), (129, 32, 4, 128, 0), (1023, 32, 4, 384, 0), (1024, 32, 4, 384, 1), (512, 32, 4, 512, 1), (2048, 32, 4, 128, 1),
    (2048, 32, 2, 3072, 1), (2048, 32, 2, 4096, 0), (2048, 32, 4, 4096, 1), (2048, 32, 4, 8192, 0), (4096, 32, 8, 8192, 1),
    (4097, 32, 1, 128, 0), (8192, 22, 2, 1024, 1), (8192, 22, 2, 2048, 0), (8192, 32, 4, 2048, 1), (16384, 32, 4, 4096, 0)])
def test_a_prompts_router_with_choice_and_plan(tokens, outputs, top, k, pays):
    assert library().imparo_moe_router_takes(tokens, outputs, outputs, top, 1, 0, k)
    assert library().imparo_moe_router_pays(tokens, outputs, top, k) == pays


@pytest.mark.parametrize("tokens,used,experts,width,hidden,pays", [
    (8, 5, 9, 1024, 768, 1), (16, 4, 16, 1024, 2048, 1), (16, 4, 16, 1024, 2080, 0), (16, 2, 8, 1024, 4096, 1), (4, 2, 12, 512, 5632, 0),
    (1, 4, 8, 2048, 1408, 1), (1, 4, 12, 2048, 1024, 0), (1, 2, 16, 2048, 4096, 1), (2, 1, 16, 2048, 4096, 1), (1, 3, 16, 2048, 4096, 0)])
def test_products_by_the_tokens_choices(tokens, used, experts, width, hidden, pays):
    assert library().imparo_moe_direct_takes(tokens, used, experts)
    assert library().imparo_moe_direct_pays(tokens, used, experts, width, hidden) == pays


@pytest.mark.parametrize("rows,splits,heads,kv_heads,brings,whole,far_first,pays", [
    (16, 8, 16, 8, 1, 1, 1, 1), (16, 9, 16, 8, 1, 1, 1, 0), (16, 8, 32, 8, 1, 1, 1, 1), (8, 4, 32, 16, 1, 1, 1, 1), (8, 5, 32, 16, 1, 1, 1, 0),
    (8, 8, 32, 16, 0, 1, 1, 1), (1, 64, 32, 16, 1, 1, 1, 1), (17, 1, 16, 8, 0, 0, 0, 0), (16, 64, 16, 8, 1, 0, 0, 1), (16, 65, 16, 8, 1, 0, 0, 0),
    (16, 8, 32, 16, 1, 0, 0, 1), (16, 9, 32, 16, 1, 0, 0, 0), (16, 64, 32, 16, 0, 0, 0, 1), (8, 64, 32, 16, 1, 0, 0, 1),
    (16, 12, 8, 8, 1, 0, 1, 1), (16, 13, 8, 8, 1, 0, 1, 0), (8, 64, 8, 8, 1, 0, 1, 1)])
def test_attention_under_a_rule_from_the_projections_rows(rows, splits, heads, kv_heads, brings, whole, far_first, pays):
    assert library().imparo_attention_decode_qkv_ruled_takes(heads, kv_heads, 64, 32, whole)
    assert library().imparo_attention_decode_qkv_ruled_pays(rows, splits, heads, kv_heads, brings, whole, far_first) == pays


@pytest.mark.parametrize("tokens,heads,kv_heads,dim,window,keep,pays", [
    (1, 16, 4, 128, 0, 0, 1), (64, 16, 4, 128, 0, 0, 1), (65, 16, 4, 128, 0, 0, 0), (1, 20, 4, 64, 0, 0, 0), (1, 16, 8, 96, 0, 0, 0),
    (1, 16, 4, 128, 79, 0, 0), (1, 16, 4, 128, 80, 0, 1), (1, 32, 8, 64, 20, 0, 0), (1, 32, 8, 64, 20, 4, 1), (1, 32, 8, 64, -20, 0, 0), (1, 32, 8, 64, -64, 0, 1),
    (1, 32, 8, 64, -100, 0, 0), (1, 32, 8, 64, -200, 0, 1), (1, 12, 4, 128, 31, 0, 0), (1, 12, 4, 128, 32, 0, 1), (1, 12, 4, 128, -20, 0, 0), (1, 24, 8, 64, 8, 0, 1),
    (1, 16, 8, 128, 1, 0, 1), (1, 8, 8, 64, -20, 0, 1)])
def test_float32_attention_of_few_tokens(tokens, heads, kv_heads, dim, window, keep, pays):
    assert library().imparo_attention_f32_split_pays(tokens, heads, kv_heads, dim, window, keep) == pays
