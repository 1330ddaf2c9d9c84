"""The rule by which a prompt's product over bfloat16 weights takes its tiles, host side: each line of the rule at both of its ends, by depth."""
import pytest

from helpers.device import cai

T32, T64, T128_16, T128_8, T256_128, T256 = range(6)


@pytest.mark.parametrize("rows,cols,n_tok,want,gated", [(*c, 0) for c in [
    # small tiles
    (2048, 2048, 32, T32), (512, 64, 2048, T64), (512, 64, 1900, T32), (18720, 256, 64, T64), (2048, 2048, 1024, T64),
    # one round of 128 x 128 against up to three tiles of 64 x 64 a CU, by depth
    (3072, 256, 700, T64), (3072, 1024, 700, T64), (3072, 2048, 700, T64), (3072, 4096, 768, T64), (3072, 4097, 700, T128_16), (2816, 4096, 768, T64), (11264, 256, 200, T64), (2816, 1024, 1024, T64),
    (4096, 1024, 768, T64), (4096, 1025, 768, T128_16), (4096, 1024, 770, T128_16), (4096, 256, 770, T128_16), (3072, 1088, 769, T128_16), (2048, 2048, 2048, T128_16), (18720, 2048, 70, T128_16),
    # one round of 256 x 256 against two of 256 x 128, by how full it is, by depth and by how full the second of the others is
    (6200, 2048, 1536, T256_128), (6200, 2048, 1537, T256), (11264, 2048, 768, T256_128), (11264, 2048, 769, T256), (6200, 513, 1540, T256), (6200, 512, 1537, T256_128), (11264, 256, 700, T256_128),
    (8192, 256, 1792, T256_128), (8192, 256, 1793, T256), (6200, 256, 2304, T256_128), (6200, 256, 2305, T256),
    # by rounds otherwise
    (11264, 2048, 300, T256_128), (11264, 2048, 640, T128_8), (32800, 2048, 128, T128_8), (11264, 2048, 2048, T256_128), (11264, 2048, 1024, T256)]] + [
    # gated products: 256 x 256 at every depth
    (6208, 256, 1536, T256_128, 1), (6208, 256, 1537, T256, 1), (12800, 256, 900, T256, 1), (3072, 256, 700, T64, 1), (4096, 256, 770, T128_16, 1), (6208, 256, 1280, T256_128, 1)])
def test_which_tiles_a_product_takes(rows, cols, n_tok, want, gated):
    assert cai.load().cai_bf16_tiles(rows, cols, n_tok, gated) == want
