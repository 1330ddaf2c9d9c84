"""The rule by which a value is in reach of the m most probable tokens, host side: how far below the first the m-th may lie before the whole row is taken, and that nothing that is
among the m falls below the bound."""
import ctypes as C

import numpy as np
import pytest

from helpers.device import cai

F = np.float32


def floor_of(value, tot, pm, t, n, divided):
    """the bound where the m-th largest of the maxima is `value`"""
    f = cai.load().cai_candidates_floor
    f.argtypes = [C.c_int, C.c_float, C.c_float, C.c_float, C.c_int, C.c_int]
    return f(int(F(value).view(np.uint32)) >> 20, tot, pm, t, n, divided)


# (nats between the first and the m-th: a quotient by the row's sum above 1e-36 was the bound of five launches, 82.9 T behind a first value that takes most of the sum)
@pytest.mark.parametrize("t,nats", [(0.02, 1.6), (0.05, 4.1), (0.1, 6.8), (0.1, 7.5), (0.1, 8.2), (0.3, 24.0), (0.7, 55.0), (0.99, 67.0), (1.3, 67.0), (100.0, 67.0), (999.0, 67.0), (1.0, 82.0), (1.0, 87.0)])
@pytest.mark.parametrize("pm,tot", [(0.9, 0.0), (0.2, 0.0), (0.2, 0.7), (0.2, 40.0)])
def test_how_far_down_the_bound_reaches(t, nats, pm, tot):
    value = pm * np.exp(-nats) * (tot or 1.0)
    if value / (tot or 1.0) > (1.4e-30 if t != 1.0 else 1.4e-38):
        got = floor_of(value, tot, pm, t, 152064, int(tot > 0))
        assert 0 < got <= int(F(value).view(np.uint32))


@pytest.mark.parametrize("t,value,tot,pm,divided", [(0.1, 0.2 * np.exp(-9.6), 0.0, 0.2, 0),                      # quotients that lose bits
                                                    (0.7, 1e-30, 0.0, 0.2, 0), (1.3, 1e-31, 0.0, 0.2, 0),            # the logarithm's floor
                                                    (1000.0, 1e-3, 0.0, 0.2, 0), (0.7, 1e-3, np.inf, 0.2, 1), (0.7, 1e-3, np.nan, 0.2, 1), (np.nan, 1e-3, 0.0, 0.2, 0),
                                                    (1.0, 1e-38, 1.0, 0.2, 1), (1.0, 1e-3, np.inf, 0.2, 1)])
def test_rows_whose_values_are_all_in_reach(t, value, tot, pm, divided):
    assert floor_of(value, tot, pm, t, 152064, divided) == 0


@pytest.mark.parametrize("t", [0.003, 0.02, 0.1, 0.5, 0.999, 1.0, 1.001, 2.5, 30.0, 999.0])
@pytest.mark.parametrize("tot", [0.0, 0.31, 1.0, 900.0])
def test_nothing_of_the_m_most_probable_lies_below_the_bound(t, tot):
    """rows with many values around the edges of the m-th one's bin and of the one below, a rounding apart, and down to the end of the number range, worked out in 32 bits as the launches do"""
    rng = np.random.default_rng(int(1000 * t) + int(tot * 10))
    n, clear = 4000, 0
    for trial in range(60):
        spread = rng.uniform(0, 12 * min(t, 5.0)) if trial % 2 else rng.uniform(0, 100 * min(t, 0.9))
        p = np.exp(-rng.uniform(0, 1, n) * spread)
        edge = F(np.exp(-rng.uniform(0, 1) * spread)).view(np.uint32) >> 20 << 20
        near = rng.permutation(n)[:1200]
        steps = rng.integers(-6, 7, 1200) + rng.choice([0, -(1 << 20), -(1 << 19), 1 << 20], 1200)
        v = p.astype(F); v[near] = np.maximum(int(edge) + steps, 1).astype(np.uint32).view(F)
        v /= v.sum(dtype=np.float64)
        v = v.astype(F)
        s = F(v.sum(dtype=F)) if tot else F(0)
        if tot:
            v = (v * F(tot)).astype(F); s = F(v.sum(dtype=F))
        with np.errstate(all="ignore"):
            q = (v / s).astype(F) if tot else v
            pm = F(q.max())
            if t != 1.0:
                inv_t = F(1) / F(t); lm = np.log(pm)
                last = np.exp((np.log(np.maximum(q, F(1e-30))) * inv_t - lm * inv_t).astype(F)).astype(F)
                q = (last * (F(1) / F(last.sum(dtype=F)))).astype(F)
        order = np.lexsort((np.arange(n), -q.astype(np.float64)))
        for m in (1, 40, 700):
            bound = floor_of(np.sort(v)[::-1][m - 1], float(s), float(pm), t, n, int(tot > 0))
            clear += bound > 0
            assert (v[order[:m]].view(np.uint32).astype(np.int64) >= bound).all(), (trial, m)
    assert clear > 20
