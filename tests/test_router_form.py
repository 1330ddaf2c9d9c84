"""The rule by which a block of a mixture gets from its rows to their experts, host side: each line of the rule at both of its ends."""
import pytest

from helpers.device import cai
from helpers.oracle_lib import Q4_0, Q4_K, Q6_K, Q8_0

LAUNCHES, FUSED, IN_BANK, ROWS = range(4)


@pytest.mark.parametrize("router,bank,experts,top_k,width,n_tok,want", [
    # one token: up to 24 places (20 of 4-bit banks), 64 experts and 4096 columns of a type whose gated launch takes a bank
    (Q8_0, Q8_0, 64, 8, 2048, 1, IN_BANK), (Q8_0, Q4_0, 64, 20, 512, 1, IN_BANK), (Q8_0, Q4_0, 64, 21, 512, 1, FUSED), (Q8_0, Q8_0, 64, 24, 512, 1, IN_BANK), (Q8_0, Q8_0, 64, 25, 512, 1, FUSED), (Q8_0, Q8_0, 64, 64, 2048, 1, FUSED), (Q8_0, Q8_0, 20, 20, 4096, 1, IN_BANK),
    (Q8_0, Q8_0, 64, 8, 4128, 1, FUSED), (Q8_0, Q6_K, 64, 8, 2048, 1, FUSED), (Q8_0, Q8_0, 65, 8, 2048, 1, LAUNCHES), (Q4_K, Q4_K, 64, 8, 2048, 1, IN_BANK), (Q4_K, Q4_K, 64, 21, 2048, 1, LAUNCHES),
    # several
    (Q8_0, Q8_0, 64, 8, 2048, 2, FUSED), (Q8_0, Q8_0, 64, 64, 2048, 8, FUSED), (Q4_0, Q4_0, 64, 8, 2048, 2, LAUNCHES)])
def test_how_a_step_finds_its_experts(router, bank, experts, top_k, width, n_tok, want):
    assert cai.load().cai_router_form(router, bank, experts, top_k, width, 1024, n_tok, 0) == want


@pytest.mark.parametrize("router,experts,top_k,width,n_tok,want", [
    # rows whose planes the launch leaves; longer ones of up to 32 experts, or of up to 256 tokens
    (Q8_0, 64, 8, 2048, 2048, ROWS), (Q8_0, 64, 64, 512, 2048, ROWS), (Q8_0, 32, 8, 4096, 2048, ROWS), (Q8_0, 33, 8, 4096, 256, ROWS), (Q8_0, 33, 8, 4096, 257, LAUNCHES), (Q8_0, 64, 8, 2080, 2048, LAUNCHES),
    (Q8_0, 65, 8, 2048, 100, LAUNCHES), (Q4_0, 64, 8, 2048, 100, LAUNCHES)])
def test_how_a_prompt_finds_its_experts(router, experts, top_k, width, n_tok, want):
    assert cai.load().cai_router_form(router, router, experts, top_k, width, 1024, n_tok, 1) == want
