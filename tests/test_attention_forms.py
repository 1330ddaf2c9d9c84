"""The rule by which a decoding step's attention takes its kernel, host side: each line of the rule at both of its ends."""
import pytest

from helpers.device import cai

F32, F16, I8 = cai.KV_F32, cai.KV_F16, cai.KV_I8
PER_HEAD, GROUPED, CORES = 0, 1, 2


@pytest.mark.parametrize("n_seq,hq,hkv,dk,rows,dtype,normed,want", [
    # a grid of KV heads x slices that does not fill the chip, widths and slices the grouped kernel does not take
    (1, 28, 4, 128, 1024, F32, 0, PER_HEAD), (1, 120, 15, 128, 1024, F16, 0, PER_HEAD), (8, 64, 64, 68, 1024, F32, 0, PER_HEAD), (8, 64, 64, 64, 512, F16, 0, PER_HEAD),
    # vector instructions: up to 512 work-groups per head, half and int8 rows of heads that share nothing up to 2048
    (1, 32, 16, 128, 1024, F32, 0, PER_HEAD), (1, 48, 16, 128, 1024, F32, 0, GROUPED), (2, 16, 16, 128, 1024, F32, 0, PER_HEAD), (3, 16, 16, 128, 1024, F32, 0, GROUPED),
    (4, 32, 32, 64, 2048, F16, 0, PER_HEAD), (5, 32, 32, 64, 2048, F16, 0, GROUPED), (4, 32, 32, 64, 2048, F32, 0, GROUPED), (1, 64, 32, 64, 2048, I8, 0, GROUPED), (1, 32, 16, 64, 2048, I8, 0, PER_HEAD),
    # matrix cores
    (1, 32, 16, 128, 1024, F16, 0, CORES), (1, 32, 16, 128, 4096, I8, 0, CORES), (4, 16, 16, 128, 1024, F16, 0, PER_HEAD), (5, 16, 16, 128, 1024, I8, 0, CORES),
    (1, 16, 16, 128, 2048, F16, 0, CORES), (1, 16, 16, 128, 2048, I8, 0, CORES), (1, 16, 16, 128, 4096, F16, 0, CORES), (1, 16, 16, 128, 4096, I8, 0, PER_HEAD), (9, 16, 16, 128, 4096, I8, 0, CORES),
    (8, 32, 32, 128, 256, F16, 0, CORES),
    # ... and normed rows of q and k, whose norm is a launch of its own in front of the grouped kernel
    (1, 32, 16, 128, 2048, F16, 1, PER_HEAD), (1, 48, 16, 128, 1024, I8, 1, CORES), (8, 16, 16, 128, 1024, F16, 1, PER_HEAD), (9, 16, 16, 128, 1024, F16, 1, CORES), (3, 16, 16, 128, 2048, F16, 1, CORES),
    # more slices than the work-group that merges takes
    (1, 16, 16, 128, 5120, F32, 0, GROUPED), (1, 16, 16, 128, 5120, I8, 1, CORES)])
def test_which_attention_kernel_a_step_takes(n_seq, hq, hkv, dk, rows, dtype, normed, want):
    assert cai.load().cai_attn_form(n_seq, hq, hkv, dk, rows, dtype, normed) == want
