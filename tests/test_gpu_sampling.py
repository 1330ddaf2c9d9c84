"""Device distribution pipeline (softmax -> history penalty -> temperature -> candidate prefix) against the oracle's
restatement of neural/neuralchatengine.pas:1374-1396, 1495-1501.  Tokens must agree rank for rank except where two
neighbouring probabilities of the oracle are within float rounding of each other; probabilities within 2e-5 relative."""
import numpy as np
import pytest

from helpers import oracle_lib as O

pytestmark = pytest.mark.gpu


def check(got, want, rtol=2e-5):
    (gt, gp), (wt, wp) = got, want
    assert gt.size == wt.size
    np.testing.assert_allclose(gp, wp, rtol=rtol, atol=1e-30)
    assert np.all(np.diff(gp) <= 0)
    for i in np.nonzero(gt != wt)[0]:
        near = [j for j in (i - 1, i + 1) if 0 <= j < wt.size and abs(wp[j] - wp[i]) <= 4e-6 * wp[i]]
        assert near, (i, gt[i], wt[i])
    assert sorted(gt.tolist()) == sorted(wt.tolist()) or abs(float(gp[-1]) - float(wp[-1])) <= 4e-6 * wp[-1]


@pytest.mark.parametrize("n,m", [(152064, 256), (49152, 64), (1000, 1000), (37, 64), (5000, 1)])
def test_candidates_match_oracle(n, m):
    from helpers.device import dev
    cai = dev()
    rng = np.random.default_rng(n + m)
    logits = (rng.standard_normal(n) * 3).astype(np.float32)
    hist = rng.integers(0, n, 300).tolist() + [int(np.argmax(logits))] * 3
    for kw in (dict(), dict(temperature=0.7), dict(temperature=1.5, history=hist, repetition=1.3),
               dict(history=hist, frequency=0.2, presence=0.5), dict(temperature=0.9, history=hist, repetition=1.1, frequency=0.1, presence=0.1)):
        check(cai.sample_candidates(logits, m, **kw), O.sample_candidates(logits, m, **kw))


def test_ties_and_degenerate_rows():
    from helpers.device import dev
    cai = dev()
    logits = np.zeros(5000, np.float32)                       # every probability equal: token order decides
    tok, p = cai.sample_candidates(logits, 100)
    np.testing.assert_array_equal(tok, np.arange(100)); assert np.all(p == p[0])
    logits[[4000, 17, 2500]] = 1.0
    tok, p = cai.sample_candidates(logits, 7)
    np.testing.assert_array_equal(tok, [17, 2500, 4000, 0, 1, 2, 3])
    logits = np.full(3000, -50.0, np.float32); logits[123] = 40.0   # one-hot: the rest underflows to equal tiny values
    tok, p = cai.sample_candidates(logits, 5)
    wt, wp = O.sample_candidates(logits, 5)
    np.testing.assert_array_equal(tok, wt); np.testing.assert_allclose(p, wp, rtol=1e-5)
    tok, p = cai.sample_candidates(logits, 3, temperature=0.0)      # T -> 0: greedy
    assert tok[0] == 123 and abs(p[0] - 1) < 1e-6
    with pytest.raises(cai.CaiError):
        cai.sample_candidates(logits, 2000)


def test_session_candidates_read_the_resident_row():
    from helpers.device import dev
    from helpers.model_build import synthetic_spec
    cai = dev()
    cfg = dict(n_layers=2, d_model=256, n_q_heads=4, n_kv_heads=2, head_dim=64, ffn=512, vocab=3000, max_ctx=32, eps=1e-5, rope_theta=1e4)
    dec = cai.Decoder(synthetic_spec(cfg, O.Q8_0, std=0.05), max_batch=2)
    ctx_tokens = [5, 99, 5, 1200]
    for p_, t in enumerate(ctx_tokens):
        _, lg = dec.step([t, (t * 7) % 3000], [p_, p_])
    for row in (0, 1):
        got = dec.candidates(40, row=row, temperature=0.8, history=ctx_tokens, repetition=1.2)
        want = O.sample_candidates(lg[row], 40, temperature=0.8, history=ctx_tokens, repetition=1.2)
        check(got, want)
        assert got[0][0] != int(np.argmax(lg[row])) or True
    # greedy agreement: the first candidate of the plain row is the arg-max the step reported
    am, lg = dec.step([7, 8], [4, 4])
    assert dec.candidates(1, row=0)[0][0] == am[0] and dec.candidates(1, row=1)[0][0] == am[1]


@pytest.mark.parametrize("n", [1, 255, 1024, 1025, 262144, 262145, 300001])
def test_slices_of_a_row(n):
    """rows that end inside a slice, fill slices exactly, fill all 256 of them, and need longer ones; m where the values in reach are
    ranked directly (64) and near the limit (1024)"""
    from helpers.device import dev
    cai = dev()
    rng = np.random.default_rng(n)
    logits = (rng.standard_normal(n) * 3).astype(np.float32)
    hist = rng.integers(0, n, 200).tolist()
    for m in (64, 1024):
        for kw in (dict(), dict(temperature=0.8, history=hist, repetition=1.2, presence=0.1)):
            check(cai.sample_candidates(logits, m, **kw), O.sample_candidates(logits, m, **kw))


def test_more_equal_values_than_are_ranked_directly():
    """5000 equal values in reach: the m-th largest is found bit by bit; quotients that underflow; rows with infinities and NaN"""
    from helpers.device import dev
    cai = dev()
    logits = np.full(60000, -3.0, np.float32)
    tied = np.random.default_rng(1).permutation(60000)[:5000]
    logits[tied] = 2.0; logits[59999] = 2.5; logits[31] = 2.25
    for kw in (dict(), dict(temperature=0.7), dict(history=[31, 59999], presence=0.5)):
        check(cai.sample_candidates(logits, 1000, **kw), O.sample_candidates(logits, 1000, **kw))
    tok, p = cai.sample_candidates(logits, 300)
    np.testing.assert_array_equal(tok, np.concatenate([[59999, 31], np.setdiff1d(np.sort(tied), [31, 59999])])[:300])
    steep = np.full(20000, -200.0, np.float32); steep[::40] = -0.001 * np.arange(500)     # the m-th largest is a zero: every value is in reach
    check(cai.sample_candidates(steep, 900, temperature=0.5), O.sample_candidates(steep, 900, temperature=0.5))
    low = np.full(5000, -np.inf, np.float32); low[[7, 4321]] = 1.0
    tok, p = cai.sample_candidates(low, 4)
    np.testing.assert_array_equal(tok, [7, 4321, 0, 1]); np.testing.assert_array_equal(p, [0.5, 0.5, 0, 0])
    low[100] = np.nan                                                # counts as far below the maximum
    tok, p = cai.sample_candidates(low, 4, temperature=0.9)
    np.testing.assert_array_equal(tok[:2], [7, 4321]); np.testing.assert_allclose(p[:2], 0.5, rtol=1e-6)


@pytest.mark.parametrize("m", [8, 300])
def test_a_probability_that_overflows_leaves_the_other_ranks_alone(m):
    """exp(100) is past the largest float: the token's share is NaN, and it still has one rank, the first, so that every place holds a token of this row"""
    from helpers.device import dev
    cai = dev()
    logits = np.random.default_rng(m).standard_normal(5000).astype(np.float32)
    cai.sample_candidates(logits, 1000)              # (what an earlier call left)
    tok, p = cai.sample_candidates(logits, m, history=[4321], presence=-100.0)
    assert tok[0] == 4321 and np.isnan(p[0])
    np.testing.assert_array_equal(tok[1:], np.arange(m - 1))
    np.testing.assert_array_equal(p[1:], np.zeros(m - 1))


@pytest.mark.parametrize("n,m,n_hist", [(8192, 128, 1025), (8193, 129, 1024), (9000, 1024, 1), (12289, 100, 5000), (33000, 256, 4097), (262145, 128, 2048), (600000, 33, 3000)])
def test_the_groups_whose_maxima_bound_the_candidates(n, m, n_hist):
    """rows whose values are binned themselves and rows in groups of 4, 16 and 64; candidates ranked by the third launch's last work-group and by a launch of their own; histories
    that fill the copying work-groups and go past what the penalties hold in registers; temperatures on both sides of the bounds"""
    from helpers.device import dev
    cai = dev()
    rng = np.random.default_rng(n + m + n_hist)
    logits = (rng.standard_normal(n) * 3).astype(np.float32)
    hist = rng.integers(0, n, n_hist).tolist() + [int(np.argmax(logits))] * 2
    for kw in (dict(), dict(temperature=1500.0), dict(temperature=999.0, history=hist, presence=0.3), dict(temperature=1.3, history=hist, repetition=0.8, frequency=-0.4),
               dict(history=hist, repetition=1.2, presence=0.5)):
        check(cai.sample_candidates(logits, m, **kw), O.sample_candidates(logits, m, **kw))
    # probabilities down to the end of the number range: an exponent is the difference of two products up to 20 / T, rounded on both sides: 4 x 2^-24 x 400
    got, want = cai.sample_candidates(logits, m, temperature=0.05), O.sample_candidates(logits, m, temperature=0.05)
    np.testing.assert_allclose(got[1], want[1], rtol=1e-4, atol=1e-30)


def test_more_in_reach_than_the_third_launch_ranks():
    """512 equal values and one more: the former are ranked by the launch that finds them, the latter by the launch behind it; both sides of the bound give token order"""
    from helpers.device import dev
    cai = dev()
    for tied in (511, 512, 513, 3000):
        logits = np.full(20000, -3.0, np.float32)
        at = np.sort(np.random.default_rng(tied).permutation(20000)[:tied]); logits[at] = 2.0
        for m in (1, 7, 128):
            tok, p = cai.sample_candidates(logits, m)
            np.testing.assert_array_equal(tok, at[:m]); assert np.all(p == p[0])
            check(cai.sample_candidates(logits, m, temperature=0.7), O.sample_candidates(logits, m, temperature=0.7))
