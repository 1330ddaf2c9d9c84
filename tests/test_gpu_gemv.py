"""Block-fused GEMV / small-batch kernels against the oracle's dequantize-then-dot definition.

Tolerance: max |y - y_ref| / max |y_ref| <= 1e-3 (north-star bar for fp32 logits); measured values are ~1e-6.
y_ref accumulates in double over the bit-exact dequantized weights.
"""
import numpy as np
import pytest

from helpers import oracle_lib as O

pytestmark = pytest.mark.gpu
TOL = 1e-3
TIGHT = 2e-5


def make(qt, rows, cols, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    return O.quantize(qt, w), rng


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,cols", [(2048, 2048), (5632, 2048), (2048, 5632), (3, 256), (1, 9728), (1000, 3584), (64, 18944), (40000, 512),
                                       (1001, 4352), (77, 6144), (3, 5120), (4099, 5120)])   # 17..24 super-blocks: four rows packed per wave
@pytest.mark.parametrize("nb", [1, 4])
def test_gemv_matches_oracle(qt, rows, cols, nb):
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(qt, rows, cols, rows * 7 + cols)
    x = rng.standard_normal((nb, cols)).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw, bias)
    got = w.gemv(x)
    want = O.gemv(qt, raw, rows, cols, x, bias, 0, 1)
    assert got.shape == want.shape
    assert rel_err(got, want, floor=0.02 * cols ** 0.5) < TIGHT


@pytest.mark.parametrize("qt,rows,cols", [(O.Q8_0, 576, 576), (O.Q8_0, 192, 576), (O.Q8_0, 576, 1536), (O.Q4_0, 96, 160), (O.Q8_0, 5, 32)])
def test_gemv_non_256_multiple_widths(qt, rows, cols):
    # SmolLM2-135M widths: 576 = 18 blocks of 32 (not a multiple of 256)
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(qt, rows, cols, 5)
    for nb in (1, 2, 3, 5, 8):
        x = rng.standard_normal((nb, cols)).astype(np.float32)
        got = cai.QWeight(qt, rows, cols, raw).gemv(x)
        assert rel_err(got, O.gemv(qt, raw, rows, cols, x, None, 0, 1)) < TIGHT


@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 6, 7, 8])
def test_all_batch_widths_q4k(nb):
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(O.Q4_K, 777, 1024, nb)
    x = rng.standard_normal((nb, 1024)).astype(np.float32)
    got = cai.QWeight(O.Q4_K, 777, 1024, raw).gemv(x)
    assert rel_err(got, O.gemv(O.Q4_K, raw, 777, 1024, x, None, 0, 1)) < TIGHT


@pytest.mark.parametrize("act", [0, 1, 2, 3])
def test_fused_bias_and_activation_order(act):
    # y = act(dot + bias): bias before activation (neural.cl:111-146)
    from helpers.device import dev
    cai = dev()
    raw, rng = make(O.Q8_0, 300, 512, 77)
    x = rng.standard_normal((2, 512)).astype(np.float32) * 3
    bias = rng.standard_normal(300).astype(np.float32)
    got = cai.QWeight(O.Q8_0, 300, 512, raw, bias).gemv(x, act)
    want = O.gemv(O.Q8_0, raw, 300, 512, x, bias, act, 1)
    assert np.max(np.abs(got - want)) < 1e-5


@pytest.mark.parametrize("qt", [O.F32, O.F16])
@pytest.mark.parametrize("rows,cols", [(11, 8), (8, 12), (8, 5), (300, 1000)])
def test_float_weight_types_any_width(qt, rows, cols):
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(qt, rows, cols, 3)
    x = rng.standard_normal((3, cols)).astype(np.float32)
    got = cai.QWeight(qt, rows, cols, raw).gemv(x)
    assert rel_err(got, O.gemv(qt, raw, rows, cols, x, None, 0, 1)) < TIGHT


@pytest.mark.parametrize("rows,cols,nb", [(37, 256, 1), (512, 3584, 1), (300, 2048, 3), (9001, 512, 1), (33001, 256, 1), (70, 18944, 1),
                                          (66, 18944, 2), (41, 1024, 8), (18000, 256, 5)])
def test_q6_k_gemv_matches_oracle(rows, cols, nb):
    """Q6_K (the type real Q4_K_M files use for output.weight and part of ffn_down) on the vector kernel: 16 lanes per
    210-byte super-block, unaligned dword requests; 1, 2 and 4 rows per wave, several activation panels, batches."""
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(O.Q6_K, rows, cols, rows + cols)
    x = rng.standard_normal((nb, cols)).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    got = cai.QWeight(O.Q6_K, rows, cols, raw, bias).gemv(x)
    want = O.gemv(O.Q6_K, raw, rows, cols, x, bias, 0, 1)
    assert rel_err(got, want, floor=0.02 * cols ** 0.5) < TIGHT


def test_q6_k_largest_codes_on_equal_activations_do_not_overflow_the_integer_sums():
    """16 codes of 63 against 16 activations at the top of the 23-bit range: 16 * 63 * (2^22 - 1) exceeds 32 bits, so the
    batch-1 kernel combines its three digit sums in floating point."""
    from helpers.device import dev, rel_err
    cai = dev()
    rows, cols = 6, 512
    blk = np.zeros(210, np.uint8)
    blk[:192] = 0xFF                                   # every code 63
    blk[192:208] = np.array([1, 2, 3, 127, 1, 1, 5, 1, 9, 1, 1, 1, 77, 1, 1, 1], np.int8).view(np.uint8)
    blk[208:210] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    raw = np.tile(blk, rows * cols // 256)
    for x in (np.ones((1, cols), np.float32), -np.ones((1, cols), np.float32), np.full((1, cols), 3.0e4, np.float32)):
        got = cai.QWeight(O.Q6_K, rows, cols, raw).gemv(x)
        want = O.gemv(O.Q6_K, raw, rows, cols, x, None, 0, 1)
        assert rel_err(got, want) < TIGHT


def test_int8_row_path_scale_then_bias():
    # the reference's own fused-quant format: y = scale_a * sum(code*x) + bias_a (neuralvolume.pas:12693-12745)
    from helpers.device import dev, rel_err
    cai = dev()
    rng = np.random.default_rng(9)
    wf = (rng.standard_normal((128, 515)) * 0.05).astype(np.float32)
    codes, scales = O.quant_int8_rows(wf)
    bias = rng.standard_normal(128).astype(np.float32)
    x = rng.standard_normal((2, 515)).astype(np.float32)
    got = cai.QWeight(cai.I8ROW, 128, 515, codes, bias, scales).gemv(x)
    want = O.gemv(O.I8ROW, codes.view(np.uint8), 128, 515, x, bias, 0, 1, scales)
    assert rel_err(got, want) < TIGHT


@pytest.mark.parametrize("rows,cols", [(128, 512), (1000, 3584), (3, 32), (577, 576), (4096, 18944), (37, 2080)])
@pytest.mark.parametrize("nb", [1, 3, 8])
def test_int8_row_widths_of_whole_32_blocks_take_the_vector_kernel(rows, cols, nb):
    """Per-row int8 matrices whose width is a multiple of 32 run the 16-byte-per-lane kernel of the block types (the row scale
    applied to the finished sum, then the bias: neuralvolume.pas:12693-12745); same contract and tolerance as other widths."""
    from helpers.device import dev, rel_err
    cai = dev()
    rng = np.random.default_rng(rows + cols)
    wf = (rng.standard_normal((rows, cols)) * 0.05).astype(np.float32)
    codes, scales = O.quant_int8_rows(wf)
    bias = rng.standard_normal(rows).astype(np.float32)
    x = rng.standard_normal((nb, cols)).astype(np.float32)
    got = cai.QWeight(cai.I8ROW, rows, cols, codes, bias, scales).gemv(x)
    want = O.gemv(O.I8ROW, codes.view(np.uint8), rows, cols, x, bias, 0, 1, scales)
    assert rel_err(got, want, floor=0.05 * cols ** 0.5) < TIGHT


def test_linearity_and_zero_input():
    # size-independent properties at a full-size shape (18944 x 3584 Q4_K)
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(O.Q4_K, 18944, 3584, 42)
    w = cai.QWeight(O.Q4_K, 18944, 3584, raw)
    a = rng.standard_normal(3584).astype(np.float32); b = rng.standard_normal(3584).astype(np.float32)
    ya, yb, yab = w.gemv(a)[0], w.gemv(b)[0], w.gemv(a + b)[0]
    assert rel_err(yab, ya + yb) < 1e-5
    assert np.all(w.gemv(np.zeros(3584, np.float32)) == 0)
    # one-hot input reads one dequantized column exactly
    e = np.zeros(3584, np.float32); e[1234] = 1
    col = O.dequant(O.Q4_K, raw, 18944 * 3584).reshape(18944, 3584)[:, 1234]
    assert rel_err(w.gemv(e)[0], col) < 1e-6


def test_lm_head_shape_q8_0():
    # 152064 x 3584 Q8_0 (Qwen2.5-7B head) at batch 1
    from helpers.device import dev, rel_err
    cai = dev()
    rows, cols = 152064, 3584
    rng = np.random.default_rng(1)
    raw = np.empty(rows * O.row_bytes(O.Q8_0, cols), np.uint8)
    step = 19008
    for r0 in range(0, rows, step):
        blk = (rng.standard_normal((step, cols)) * 0.02).astype(np.float32)
        raw[r0 * O.row_bytes(O.Q8_0, cols):(r0 + step) * O.row_bytes(O.Q8_0, cols)] = O.quantize(O.Q8_0, blk)
    x = rng.standard_normal(cols).astype(np.float32)
    got = cai.QWeight(O.Q8_0, rows, cols, raw).gemv(x)
    want = O.gemv(O.Q8_0, raw, rows, cols, x, None, 0, 1)
    assert rel_err(got, want) < TIGHT
    assert int(np.argmax(got)) == int(np.argmax(want))


@pytest.mark.parametrize("rows,cols,T", [(128, 256, 1), (1000, 1024, 5), (300, 3584, 128), (777, 2048, 200), (4608, 3584, 64)])
def test_multi_token_gemm_on_matrix_cores_equals_gemv(rows, cols, T):
    """cai_qgemm (Q4_K: MFMA with exact integer blocks and hi/lo-split activations) == T single-token layers."""
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(O.Q4_K, rows, cols, T)
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)   # very different scales per token
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(O.Q4_K, rows, cols, raw, bias)
    got = w.gemm(x)
    want = O.gemv(O.Q4_K, raw, rows, cols, x, bias, 0, 1)
    for t in range(T):
        assert rel_err(got[t], want[t], floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < TIGHT, t


@pytest.mark.parametrize("rows,cols,T", [(128, 256, 2), (33, 512, 3), (1000, 1024, 8), (3584, 3584, 8), (512, 18944, 4), (40000, 2048, 16), (5000, 768, 13)])
def test_small_batch_gemm_on_matrix_cores_equals_gemv(rows, cols, T):
    """2..16 tokens: the streaming matrix-core kernel (scales folded exactly into the f16 weight operand, block sums fed as one
    more reduction step, 1/2/4 super-block slices per row tile) == T single-token layers, bias included."""
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(O.Q4_K, rows, cols, T + 100)
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    x[0, : cols // 2] = 0.0                          # all-zero blocks
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(O.Q4_K, rows, cols, raw, bias)
    got = w.gemm(x)
    want = O.gemv(O.Q4_K, raw, rows, cols, x, bias, 0, 1)
    for t in range(T):
        assert rel_err(got[t], want[t], floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < TIGHT, t


def test_multi_token_gemm_other_types_and_tokens_not_multiple_of_eight():
    from helpers.device import dev, rel_err
    cai = dev()
    for qt in (O.Q8_0, O.Q4_0):
        raw, rng = make(qt, 200, 576, 9)
        x = rng.standard_normal((13, 576)).astype(np.float32)
        got = cai.QWeight(qt, 200, 576, raw).gemm(x)
        assert rel_err(got, O.gemv(qt, raw, 200, 576, x, None, 0, 1)) < TIGHT


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,cols,T", [(128, 256, 2), (33, 512, 3), (1000, 1024, 8), (3584, 3584, 8), (512, 18944, 4), (40000, 2048, 16),
                                         (5000, 768, 13), (577, 576, 8), (192, 576, 40), (96, 160, 5), (5, 32, 2), (70, 1536, 7)])
def test_small_batch_gemm_q8_0_q4_0_on_matrix_cores(qt, rows, cols, T):
    """32-weight block types on the matrix cores: signed codes as exact f16 (activations the A operand, 16 weight rows the B
    operand, one MFMA per block, the block scale applied to its result) == T single-token layers, bias included.  Widths that
    are not a multiple of 256 end in a short group of blocks."""
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(qt, rows, cols, T + 200)
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    x[0, : cols // 2] = 0.0
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw, bias)
    got = w.gemm(x, matrix_cores=True)               # small matrices would otherwise stay on the vector-unit kernel
    want = O.gemv(qt, raw, rows, cols, x, bias, 0, 1)
    for t in range(T):
        assert rel_err(got[t], want[t], floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < TIGHT, t
    assert rel_err(w.gemm(x), want, floor=0.02 * cols ** 0.5 * float(np.abs(x).mean())) < TIGHT   # the dispatcher's own choice


@pytest.mark.parametrize("rows,cols,T", [(128, 256, 2), (33, 512, 3), (1000, 1024, 8), (3584, 3584, 8), (512, 18944, 4), (20000, 2048, 16), (5000, 768, 13), (70, 1536, 7),
                                         (1000, 1024, 40), (3584, 3584, 77), (512, 18944, 33), (130, 512, 64), (4099, 256, 129)])
def test_small_batch_gemm_q6_k_on_matrix_cores(rows, cols, T):
    """Q6_K on the matrix cores: one 16-deep MFMA per 16-weight scale group (codes q - 32 exact in f16, d * scale applied to
    the result by the lane that owns the weight row), 16-byte requests transposed over the four k lanes
    == T single-token layers, bias included.  More than 16 tokens take the prompt kernel: the scale split into
    16 * (s >> 4) and s & 15, two exact f16 operand slots per weight."""
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(O.Q6_K, rows, cols, T + 300)
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    x[0, : cols // 2] = 0.0
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(O.Q6_K, rows, cols, raw, bias)
    got = w.gemm(x, matrix_cores=True)
    want = O.gemv(O.Q6_K, raw, rows, cols, x, bias, 0, 1)
    for t in range(T):
        assert rel_err(got[t], want[t], floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < TIGHT, t
    assert rel_err(w.gemm(x), want, floor=0.02 * cols ** 0.5 * float(np.abs(x).mean())) < TIGHT   # the dispatcher's own choice


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0, O.I8ROW])
@pytest.mark.parametrize("rows,cols", [(1, 32), (3, 1024), (5, 1056), (7, 2048), (6, 2080), (9, 4064), (5, 4096), (5, 4128), (8195, 96), (8195, 2080), (32771, 160), (32771, 1056), (8195, 4128), (32771, 5152), (5, 18912)])
def test_one_row_of_activations_at_the_edges_of_what_a_launch_holds(qt, rows, cols):
    """Widths around one, two and four activations a thread and past them (another kernel, up to three panels), one to nine steps of 64 units, rows that end
    inside a group of one, two and four."""
    from helpers.device import dev, rel_err
    cai = dev()
    scales = None
    rng = np.random.default_rng(rows + cols)
    if qt == O.I8ROW:
        raw, scales = O.quant_int8_rows((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    else:
        raw, rng = make(qt, rows, cols, 1)
    x = rng.standard_normal((1, cols)).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw, bias, scales)
    want = O.gemv(qt, raw.view(np.uint8), rows, cols, x, bias, 0, 1, scales) if qt == O.I8ROW else O.gemv(qt, raw, rows, cols, x, bias, 0, 1)
    assert rel_err(w.gemv(x), want, floor=0.02 * cols ** 0.5) < TIGHT


@pytest.mark.parametrize("qt,rows,cols", [(O.Q8_0, 4101, 4096), (O.Q4_0, 8203, 4096), (O.Q4_K, 8203, 4096), (O.Q6_K, 5003, 4096), (O.I8ROW, 4101, 4096), (O.I8ROW, 7001, 2400)])
@pytest.mark.parametrize("nb", [2, 4, 8])
def test_gemv_batch_on_large_matrix_goes_to_matrix_cores(qt, rows, cols, nb):
    """cai_qgemv with a batch on a matrix of 16 MiB or more takes the matrix-core small-batch path; same contract as batch 1."""
    from helpers.device import dev, rel_err
    cai = dev()
    scales = None
    if qt == O.I8ROW:      # the reference's own per-row int8 format (width 2400: a short last block group)
        rng = np.random.default_rng(nb)
        raw, scales = O.quant_int8_rows((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    else:
        raw, rng = make(qt, rows, cols, nb)
    x = rng.standard_normal((nb, cols)).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw, bias, scales)
    got = w.gemv(x)
    want = O.gemv(qt, raw.view(np.uint8) if qt == O.I8ROW else raw, rows, cols, x, bias, 0, 1, scales) if qt == O.I8ROW else O.gemv(qt, raw, rows, cols, x, bias, 0, 1)
    assert rel_err(got, want, floor=0.02 * cols ** 0.5) < TIGHT
    one = w.gemv(x[:1])
    assert rel_err(got[:1], one, floor=0.02 * cols ** 0.5) < TIGHT


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,cols,T", [(200, 576, 17), (577, 576, 40), (192, 576, 255), (1000, 1024, 33), (3584, 3584, 77), (512, 18944, 64), (130, 512, 129),
                                         (4099, 256, 96), (96, 160, 31), (5, 32, 100), (9000, 2048, 300), (64, 2048, 255)])
def test_prompt_gemm_q8_0_q4_0_on_matrix_cores(qt, rows, cols, T):
    """More than 16 tokens of a 32-weight block type go to the prompt kernel (weights as the B operand of 32x32x16 tiles, the
    block scale applied to each block's sums): == T single-token layers of the oracle, bias included; widths that end inside a
    256-column step, row counts that end inside a tile, token counts that end inside a token tile."""
    from helpers.device import dev, rel_err
    cai = dev()
    raw, rng = make(qt, rows, cols, T + 300)
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    x[0, : cols // 2] = 0.0
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw, bias)
    got = w.gemm(x)
    want = O.gemv(qt, raw, rows, cols, x, bias, 0, 1)
    for t in range(T):
        assert rel_err(got[t], want[t], floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < TIGHT, t
    w.close()


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q8_0, O.Q4_0, O.Q6_K])
@pytest.mark.parametrize("cols", [3584, 5120])
def test_a_nan_or_inf_activation_reaches_every_output(qt, cols):
    """The integer-dot kernels hold the activation in block-float form (a maximum and integers): a NaN or an infinity in x
    must still poison every output row, as it does in the float dot product of the reference (0 * inf = NaN, x + NaN = NaN),
    and must not leak into rows of a clean batch neighbour."""
    from helpers.device import dev
    cai = dev()
    rows = 300
    raw, rng = make(qt, rows, cols, cols + qt)
    w = cai.QWeight(qt, rows, cols, raw)
    for bad in (np.nan, np.inf, -np.inf):
        for at in (0, 7, cols - 1, cols // 2 + 33):
            x = rng.standard_normal((1, cols)).astype(np.float32)
            x[0, at] = bad
            got = w.gemv(x)
            assert not np.isfinite(got).any(), (bad, at, int(np.isfinite(got).sum()))
    x = rng.standard_normal((3, cols)).astype(np.float32)
    x[1, 100] = np.nan
    got = w.gemv(x)
    assert np.isfinite(got[0]).all() and np.isfinite(got[2]).all() and not np.isfinite(got[1]).any()
    w.close()


@pytest.mark.parametrize("qt,rows,cols", [(O.Q4_K, 8203, 4096), (O.Q8_0, 4101, 4096)])
def test_a_nan_token_poisons_only_its_own_row_on_the_matrix_cores(qt, rows, cols):
    """The same through the matrix-core kernels (a batch of 8 on a matrix of 16 MiB or more, and a 40-token prompt product):
    the poisoned token's outputs are all non-finite, every other token's outputs are finite."""
    from helpers.device import dev
    cai = dev()
    raw, rng = make(qt, rows, cols, 31)
    w = cai.QWeight(qt, rows, cols, raw)
    x = rng.standard_normal((8, cols)).astype(np.float32)
    x[5, 77] = np.nan; x[2, 4000] = np.inf
    got = w.gemv(x)
    for t in range(8):
        assert np.isfinite(got[t]).all() == (t not in (2, 5)), t
        if t in (2, 5):
            assert not np.isfinite(got[t]).any(), t
    x = rng.standard_normal((40, cols)).astype(np.float32)
    x[33, 1] = np.nan
    got = w.gemm(x)
    assert not np.isfinite(got[33]).any()
    assert np.isfinite(np.delete(got, 33, axis=0)).all()
    w.close()


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q4_0, O.Q6_K])
def test_blocks_of_denormal_and_huge_activations(qt):
    """Block-float corner cases of the integer-dot kernels: a 32-block holding only denormals (its scale underflows: the block
    must count as zero, not as NaN), a block of values near 1e30, and a block with one huge and otherwise tiny values (the
    tiny ones round to zero integers, as 2^-23 of the maximum allows).  The kernels sum quant x activation over a 32-block
    BEFORE the block's scale (about 1e-3) multiplies it, so their range ends about four decades below the float maximum:
    activations beyond 1e33 may overflow where a dequantise-first product would not."""
    from helpers.device import dev, rel_err
    cai = dev()
    rows, cols = 200, 3584
    raw, rng = make(qt, rows, cols, 5 + qt)
    w = cai.QWeight(qt, rows, cols, raw)
    x = rng.standard_normal((1, cols)).astype(np.float32)
    x[0, 64:96] = np.float32(1e-40); x[0, 70] = 0.0; x[0, 71] = np.float32(-3e-41)
    x[0, 512:544] *= np.float32(1e30)
    x[0, 1024:1056] = np.float32(1e-12); x[0, 1030] = np.float32(5e6)
    got = w.gemv(x)
    want = O.gemv(qt, raw, rows, cols, x, None, 0, 1)
    assert np.isfinite(got).all()
    assert rel_err(got, want) < TIGHT
    w.close()


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q5_K])
@pytest.mark.parametrize("rows,cols,T", [(255, 2560, 17), (256, 2560, 64), (257, 2048, 65), (700, 2816, 129), (33000, 2048, 130)])
def test_prompt_products_on_wide_tiles(qt, rows, cols, T):
    """tiles of 256 rows x 64 or 128 tokens: one row short of a tile, exactly one, one more; widths of 8, 10 and 11 super-blocks cut into
    slices of unequal length; 258 tiles, of which two are left over from a round of 256 and cut"""
    from helpers.device import dev, rel_err
    cai = dev()
    rng = np.random.default_rng(rows + cols + T)
    base = O.quantize(qt, (rng.standard_normal((min(rows, 700), cols)) * 0.02).astype(np.float32)).reshape(min(rows, 700), -1)
    raw = np.ascontiguousarray(base[np.arange(rows) % 700])
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    x[0, : cols // 2] = 0.0
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw.reshape(-1), bias)
    got = w.gemm(x)
    for t in sorted({0, 1, 15, 31, 32, T // 2, 63, 64, T - 2, T - 1} & set(range(T))):
        want = O.gemv(qt, base.reshape(-1), base.shape[0], cols, x[t:t + 1], None, 0, 1)[0][np.arange(rows) % 700] + bias
        assert rel_err(got[t], want, floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < 2e-5, t
    w.close()


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,cols,T", [(40, 96, 17), (300, 544, 9), (3584, 3584, 8), (2048, 8192, 16), (8192, 64, 33), (8193, 544, 65), (9000, 128, 255), (40000, 96, 31), (40000, 128, 32), (40000, 96, 64),
                                         (40000, 128, 63), (40000, 96, 129), (39937, 192, 128), (66000, 32, 100)])
def test_prompt_products_on_block_tiles(qt, rows, cols, T):
    """each form of the block product at its edges: cut tiles of 32 and 64 rows (one and two work-groups a CU), tiles of 256 rows x 64 tokens
    (half empty, full, one token short) and x 128; rows of an odd and an even number of blocks, one block, one chunk"""
    from helpers.device import dev, rel_err
    cai = dev()
    rng = np.random.default_rng(rows + cols + T)
    base = O.quantize(qt, (rng.standard_normal((min(rows, 700), cols)) * 0.02).astype(np.float32)).reshape(min(rows, 700), -1)
    raw = np.ascontiguousarray(base[np.arange(rows) % 700])
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw.reshape(-1), bias)
    got = w.gemm(x)
    for t in sorted({0, 1, 15, 31, 32, T // 2, 63, 64, T - 2, T - 1} & set(range(T))):
        want = O.gemv(qt, base.reshape(-1), base.shape[0], cols, x[t:t + 1], None, 0, 1)[0][np.arange(rows) % 700] + bias
        assert rel_err(got[t], want, floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < 2e-5, t
    w.close()


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0, O.Q2_K, O.Q3_K, O.Q4_1, O.Q5_0, O.Q5_1])
@pytest.mark.parametrize("T", [9, 70])
def test_prompt_rows_at_the_ends_of_the_number_range(qt, T):
    """the largest finite values, very small ones, denormals, an infinity (which takes the sign of its weight) and a NaN, each in a token of its own"""
    from helpers.device import dev
    cai = dev()
    rows, cols = 300, 768
    raw, rng = make(qt, rows, cols, qt)
    w, full = cai.QWeight(qt, rows, cols, raw), O.dequant(qt, raw, rows * cols).reshape(rows, cols)
    x = rng.standard_normal((T, cols)).astype(np.float32)
    x[0, 100] = 3.3e38
    for t, scale in ((1, 1e36), (2, 1e-20), (3, 1e-33), (4, 1e-36), (5, 1e-40)):
        x[t] *= np.float32(scale)
    x[6, 37], x[7, 37], x[8, 37] = np.inf, -np.inf, np.nan
    got = w.gemm(x)
    for t in (0, 1, 2, 3, 4, 5, T - 1):
        if t == 8:
            continue
        want = full.astype(np.float64) @ x[t].astype(np.float64)
        slack = cols * 2.0 ** -149 if t == 5 else TIGHT * np.abs(want).max()        # (denormals: whole multiples of 2^-149)
        assert np.abs(got[t].astype(np.float64) - want).max() <= slack, t
    clear = np.abs(full[:, 37]) > 1e-4
    np.testing.assert_array_equal(got[6, clear], np.sign(full[clear, 37]) * np.inf)
    np.testing.assert_array_equal(got[7, clear], np.sign(full[clear, 37]) * -np.inf)
    assert np.isnan(got[8]).all()
    w.close()


@pytest.mark.parametrize("qt", [O.Q4_K, O.Q5_K])
def test_prompt_of_a_decoder_on_wide_tiles(qt):
    """q | k | v in one launch of three row groups, gate | up with SwiGLU in the epilogue and behind the slices, residual on a cut product:
    a prompt of 70 tokens equals its tokens one by one"""
    from helpers.device import dev, rel_err
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=2, d_model=2048, n_q_heads=4, n_kv_heads=1, head_dim=128, ffn=2304, vocab=500, max_ctx=128, eps=1e-5, rope_theta=1e4)
    spec = synthetic_spec(cfg, qt, head_qtype=O.Q8_0, seed=5, std=0.03, qkv_bias=True)
    dec = cai.Decoder(spec, max_batch=2)
    tok = np.random.default_rng(2).integers(0, 500, 70).astype(np.int32)
    _, got = dec.prefill(tok)
    for p_, t in enumerate(tok):
        _, want = dec.step_window([t], p_, seq=1)
    assert rel_err(got, want[0]) < 1e-4
    dec.close()


# one block of width and of ffn, odd numbers of blocks, k and v rows that are no whole 32, tiles of 16 tokens (whole, one token over), one work-group a CU
# (the last but one refills its rings of four chunks a wave), two (the last two: gate | up alone, all but the ends, rings refilled)
@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("d,ffn,hq,hkv,hd,T", [(32, 32, 1, 1, 32, 9), (64, 96, 2, 1, 32, 17), (96, 160, 6, 3, 16, 16), (96, 1120, 6, 3, 16, 33), (1056, 2144, 8, 2, 64, 12), (1600, 320, 8, 2, 64, 9),
                                             (576, 1536, 9, 3, 64, 90), (1088, 1120, 9, 3, 128, 125)])
def test_short_prompts_whose_activations_stay_planes(qt, d, ffn, hq, hkv, hd, T):
    """A prompt equals its tokens one by one, with gains and biases everywhere.  Both sides are 32-bit sums over activations of 22 bits: 4e-7 from 64 bits a layer
    (2e-6 of the largest logit where a layer's rounding is carried on), so 1e-5 apart at most."""
    from helpers.device import dev, rel_err
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=3, d_model=d, n_q_heads=hq, n_kv_heads=hkv, head_dim=hd, ffn=ffn, vocab=300, max_ctx=128, eps=1e-5, rope_theta=1e4)
    spec = synthetic_spec(cfg, qt, head_qtype=O.Q8_0, seed=d + T, std=0.05, qkv_bias=True)
    rng = np.random.default_rng(T)
    for key in spec["vecs"]:
        spec["vecs"][key] = (1.0 + 0.3 * rng.standard_normal(spec["vecs"][key].size)).astype(np.float32)
    for l in range(cfg["n_layers"]):
        for slot, n in ((O.W_O, d), (O.W_GATEUP, 2 * ffn), (O.W_DOWN, d)):
            spec["tensors"][(l, slot)]["bias"] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    dec = cai.Decoder(spec, max_batch=2)
    tok = rng.integers(0, 300, T).astype(np.int32)
    _, got = dec.prefill(tok)
    for p_, t in enumerate(tok):
        _, want = dec.step_window([t], p_, seq=1)
    assert rel_err(got, want[0]) < 1e-5
    after = dec.step(np.array([7, 7], np.int32), np.array([T, T], np.int32))[1]      # (from the cached rows of either)
    assert rel_err(after[0], after[1]) < 1e-5
    dec.close()


# heads whose results become planes in the attention (64, 32, 128 on the matrix cores) and not (16, 48); rows appended by the product (float, half) and not (int8, a rolling cache);
# one slice, slices that a merge adds, a window that leaves out the first of them; a prompt behind cached rows
@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("hq,hkv,hd", [(3, 1, 64), (4, 2, 32), (6, 6, 16), (2, 1, 48), (3, 1, 128)])
@pytest.mark.parametrize("kv,ctx,window,rolling", [("f32", 40, 0, 0), ("f16", 96, 20, 0), ("f16", 700, 0, 0), ("f32", 2000, 50, 0), ("i8", 96, 0, 0), ("f32", 200, 0, 90)])
def test_short_prompts_append_their_rows_and_leave_planes(qt, hq, hkv, hd, kv, ctx, window, rolling):
    """Two portions of a prompt equal its tokens one by one, and so does a step from the rows they left (a half on the edge between two may land one
    apart, 2^-11 of a cached element, a code of an int8 cache too)"""
    from helpers.device import dev, rel_err
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=2, d_model=96, n_q_heads=hq, n_kv_heads=hkv, head_dim=hd, ffn=160, vocab=300, max_ctx=ctx, eps=1e-5, rope_theta=1e4, window=window)
    spec = synthetic_spec(cfg, qt, head_qtype=O.Q8_0, seed=hd, std=0.05, qkv_bias=True)
    dec = cai.Decoder(spec, max_batch=2, kv_dtype={"f32": cai.KV_F32, "f16": cai.KV_F16, "i8": cai.KV_I8}[kv])
    if rolling:
        dec.set_eviction(8, rolling - 8)
    tok = np.random.default_rng(ctx).integers(0, 300, 39).astype(np.int32)
    tol = {"f32": 1e-5, "f16": 1e-3, "i8": 5e-3}[kv]
    for p_, t in enumerate(tok[:38]):
        _, want = dec.step_window([t], p_, seq=1)
        if p_ == 20:
            first = want[0].copy()
    _, got = dec.prefill(tok[:21])
    assert rel_err(got, first) < tol
    _, got = dec.prefill(tok[21:38], 21)
    assert rel_err(got, want[0]) < tol
    after = dec.step(np.array([tok[38]] * 2, np.int32), np.array([38, 38], np.int32))[1]
    assert rel_err(after[0], after[1]) < tol
    dec.close()


# rows that fill a part of the work-group, one, two and four pieces a thread, and rows past what it holds; one expert, and more than are requested at once
@pytest.mark.parametrize("d,experts,top", [(96, 4, 1), (1056, 12, 9), (2080, 3, 2), (4128, 2, 2)])
def test_prompt_of_a_mixture_whose_rows_become_planes(d, experts, top):
    """The experts' rows are added where the next layer's planes are made: a prompt equals its tokens one by one (32-bit sums over activations of 22 bits, 1e-5
    apart at most where a layer's rounding is carried on)"""
    from helpers.device import dev, rel_err
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=3, d_model=d, n_q_heads=2, n_kv_heads=1, head_dim=32, ffn=64, vocab=300, max_ctx=64, eps=1e-5, rope_theta=1e4, n_experts=experts, top_k=top, norm_topk=1)
    dec = cai.Decoder(synthetic_spec(cfg, O.Q8_0, head_qtype=O.Q8_0, seed=d, std=0.05), max_batch=2)
    tok = np.random.default_rng(d).integers(0, 300, 33).astype(np.int32)
    _, got = dec.prefill(tok)
    for p_, t in enumerate(tok):
        _, want = dec.step_window([t], p_, seq=1)
    assert rel_err(got, want[0]) < 1e-5
    dec.close()


@pytest.mark.parametrize("qt,ffn,T", [(O.Q8_0, 352, 100), (O.Q4_0, 64, 40), (O.Q8_0, 320, 150)])
def test_prompt_of_a_mixture_on_tiles_of_64_slots(qt, ffn, T):
    """banks of four experts, two a token: runs of about T / 2 slots in tiles of 64 (full, half empty, a remainder), widths of an odd and an
    even number of blocks, windows of 704, 128 and 640 rows: a prompt equals its tokens one by one"""
    from helpers.device import dev, rel_err
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=2, d_model=256, n_q_heads=4, n_kv_heads=2, head_dim=64, ffn=ffn, vocab=300, max_ctx=256, eps=1e-5, rope_theta=1e4,
               n_experts=4, top_k=2, norm_topk=1)
    spec = synthetic_spec(cfg, qt, head_qtype=O.Q8_0, seed=T, std=0.05, qkv_bias=False)
    dec = cai.Decoder(spec, max_batch=2)
    tok = np.random.default_rng(3).integers(0, 300, T).astype(np.int32)
    _, got = dec.prefill(tok)
    for p_, t in enumerate(tok):
        _, want = dec.step_window([t], p_, seq=1)
    assert rel_err(got, want[0]) < 1e-4
    dec.close()


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,cols,T", [(39937, 544, 128), (39937, 576, 100)])
def test_large_block_tiles_of_many_chunks(qt, rows, cols, T):
    """tiles of 256 rows x 128 tokens nine chunks of 64 columns deep, whose ring of three is filled three times; an odd and an even number of blocks"""
    from helpers.device import dev, rel_err
    cai = dev()
    rng = np.random.default_rng(cols + qt)
    base = O.quantize(qt, (rng.standard_normal((700, cols)) * 0.02).astype(np.float32)).reshape(700, -1)
    raw = np.ascontiguousarray(base[np.arange(rows) % 700])
    x = rng.standard_normal((T, cols)).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw.reshape(-1))
    got = w.gemm(x)
    want = x.astype(np.float64) @ O.dequant(qt, base.reshape(-1), 700 * cols).reshape(700, cols).astype(np.float64).T
    assert rel_err(got, want[:, np.arange(rows) % 700]) < TIGHT
    w.close()


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("rows,cols,T", [(16380, 544, 97), (10600, 576, 140), (10600, 544, 150)])
def test_block_tiles_of_128_rows(qt, rows, cols, T):
    """tiles of 128 rows x 64 tokens, one a CU: a last tile of 33, 12 and 22 tokens, rows that are no whole tile, an odd and an even number of blocks"""
    from helpers.device import dev, rel_err
    cai = dev()
    rng = np.random.default_rng(cols + qt + T)
    base = O.quantize(qt, (rng.standard_normal((700, cols)) * 0.02).astype(np.float32)).reshape(700, -1)
    raw = np.ascontiguousarray(base[np.arange(rows) % 700])
    x = rng.standard_normal((T, cols)).astype(np.float32)
    w = cai.QWeight(qt, rows, cols, raw.reshape(-1))
    got = w.gemm(x)
    want = x.astype(np.float64) @ O.dequant(qt, base.reshape(-1), 700 * cols).reshape(700, cols).astype(np.float64).T
    assert rel_err(got, want[:, np.arange(rows) % 700]) < TIGHT
    w.close()


@pytest.mark.parametrize("experts,T", [(130, 40), (500, 70)])
def test_prompt_of_a_mixture_of_more_experts_than_a_wave(experts, T):
    """slots grouped by expert where the sums over the experts before one run over several waves: a prompt equals its tokens one by one"""
    from helpers.device import dev, rel_err
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=2, d_model=128, n_q_heads=4, n_kv_heads=2, head_dim=32, ffn=64, vocab=300, max_ctx=128, eps=1e-5, rope_theta=1e4,
               n_experts=experts, top_k=2, norm_topk=1)
    spec = synthetic_spec(cfg, O.Q8_0, head_qtype=O.Q8_0, seed=T, std=0.05, qkv_bias=False)
    dec = cai.Decoder(spec, max_batch=2)
    tok = np.random.default_rng(3).integers(0, 300, T).astype(np.int32)
    _, got = dec.prefill(tok)
    for p_, t in enumerate(tok):
        _, want = dec.step_window([t], p_, seq=1)
    assert rel_err(got, want[0]) < 1e-4
    dec.close()


@pytest.mark.parametrize("qt", [O.Q8_0, O.Q4_0])
@pytest.mark.parametrize("cols", [512, 3584])
@pytest.mark.parametrize("spread", [0.0, 1.5])
def test_products_of_nine_tokens_are_as_near_as_the_walk_of_eight(qt, cols, spread):
    """activations of even and of widely differing sizes: nine tokens at once are as close to 64 bits as the same tokens in a pass of eight (relative
    errors of 64 tokens of 3000 results each, squares averaged: a hundredth apart at most by chance)"""
    from helpers.device import dev
    cai = dev()
    rng = np.random.default_rng(cols + qt)
    raw = O.quantize(qt, (rng.standard_normal((3000, cols)) * 0.02).astype(np.float32))
    w, full = cai.QWeight(qt, 3000, cols, raw), O.dequant(qt, raw, 3000 * cols).reshape(3000, cols).astype(np.float64)
    err = np.zeros(2)
    for _ in range(8):
        x = (rng.standard_normal((9, cols)) * np.exp(spread * rng.standard_normal((9, cols)))).astype(np.float32)
        want = x[:8].astype(np.float64) @ full.T
        for i, got in enumerate((w.gemm(x)[:8], w.gemv(x[:8]))):
            err[i] += np.sum(np.linalg.norm(got - want, axis=1) ** 2 / np.linalg.norm(want, axis=1) ** 2)
    assert err[0] <= 1.02 * err[1], np.sqrt(err / 64)
    w.close()


def test_short_prompt_of_a_mixture_sums_its_width_in_steps():
    """12 tokens through experts whose weights and activations are all positive, so that a chain over the width rounds at the size of the whole
    sum: the last of 128 blocks in one chain is added at 128 times its own size, in steps of sixteen at 16 times.  What the two add to the other
    roundings of the block (1.6e-7, the walks of the tokens one by one) is 2.0e-7 and 0.3e-7: the bound lies between their sums.
    The reference is the same block in 64 bits; the attention is switched off by a zero output projection"""
    from helpers.device import dev
    from helpers.model_build import _t, synthetic_spec
    cai = dev()
    d, I, E, V = 4096, 32, 4, 256
    cfg = dict(n_layers=1, d_model=d, n_q_heads=2, n_kv_heads=1, head_dim=64, ffn=I, vocab=V, max_ctx=64, eps=1e-5, rope_theta=1e4, n_experts=E, top_k=2, norm_topk=1)
    spec = synthetic_spec(cfg, O.Q8_0, head_qtype=O.Q8_0, seed=1, std=0.02)
    rng = np.random.default_rng(2)
    T = spec["tensors"]
    put = lambda key, w: T.__setitem__(key, _t(w.astype(np.float32), O.Q8_0))
    put((-1, O.W_EMBED), rng.uniform(0.5, 1.5, (V, d))); put((0, O.W_O), np.zeros((d, 128)))
    put((0, O.W_GATEUP), rng.uniform(0.0, 2.0 / d, (2 * I * E, d))); put((0, O.W_DOWN), rng.standard_normal((E * d, I)))
    w = {k: O.dequant(O.Q8_0, np.asarray(t["raw"]).reshape(-1), t["rows"] * t["cols"]).reshape(t["rows"], t["cols"]).astype(np.float64) for k, t in T.items()}
    dec = cai.Decoder(spec)
    rms = lambda x: x / np.sqrt(np.mean(x * x) + np.float64(np.float32(1e-5)))
    err = size = 0.0
    for seed in range(8):
        tok = np.random.default_rng(10 + seed).integers(0, V, 12).astype(np.int32)
        dec.reset()
        _, got = dec.prefill(tok)
        x = w[(-1, O.W_EMBED)][tok[-1]]
        u = rms(x)
        s = w[(0, O.W_ROUTER)] @ u
        top = np.argsort(-s)[:2]
        g = np.exp(s[top] - s[top].max()); g /= g.sum()
        for e, ge in zip(top, g):
            gu = w[(0, O.W_GATEUP)][e * 2 * I:(e + 1) * 2 * I] @ u
            x = x + ge * (w[(0, O.W_DOWN)][e * d:(e + 1) * d] @ (gu[:I] * gu[I:] / (1.0 + np.exp(-gu[I:]))))
        want = w[(-1, O.W_HEAD)] @ rms(x)
        err += np.sum((got - want) ** 2); size += np.sum(want ** 2)
    dec.close()
    assert np.sqrt(err / size) < 2.1e-7


@pytest.mark.parametrize("cols", [32, 1024, 1056, 2048, 2080, 4096, 4128, 8192, 8224, 24576, 24608])
def test_prompt_rows_at_the_widths_of_the_pre_pass(cols):
    """the last and the first width of each number of values a thread keeps, and rows that start one float off alignment"""
    import torch
    from helpers.device import dev, rel_err
    cai = dev()
    rows, T = 40, 18
    raw, rng = make(O.Q8_0, rows, cols, cols)
    x = (rng.standard_normal((T, cols)) * rng.uniform(0.01, 30.0, (T, 1))).astype(np.float32)
    w = cai.QWeight(O.Q8_0, rows, cols, raw)
    want = O.gemv(O.Q8_0, raw, rows, cols, x, None, 0, 1)
    buf, y = torch.zeros(T * cols + 1, device="cuda"), torch.zeros((T, rows), device="cuda")
    for shift in (0, 1):
        buf[shift:shift + T * cols].copy_(torch.from_numpy(x).reshape(-1))
        torch.cuda.synchronize()
        cai.check(cai.load().cai_qgemm(w.h, cai.C.c_void_p(buf.data_ptr() + 4 * shift), T, cai.C.c_void_p(y.data_ptr()), cai.X_DEVICE | cai.Y_DEVICE))
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        for t in range(T):
            assert rel_err(got[t], want[t], floor=0.02 * cols ** 0.5 * float(np.abs(x[t]).mean())) < TIGHT, (shift, t)
    w.close()
