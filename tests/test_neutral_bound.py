"""The rule by which the radius loop passes over a radius at which no cell can
be ionized, restated in float64: whenever it says so, the excursion-set rule
ionizes no cell, whatever the field, barrier and efficiency."""
import numpy as np
from hypothesis import given, settings, strategies as st
from scipy.special import erfc, erfcinv


def stays_neutral(delta, bound, deltac, denom, zeta, fc_mean, linear):
    b = bound * (1 + 1e-4)
    if linear:
        y = 1.0 / zeta
        if not 1e-30 < y < 1.999:
            return False
        ds = deltac - denom * erfcinv(y)
        return b < ds - 1e-4 * (1 + abs(deltac) + denom + abs(ds))
    return b <= deltac and zeta * fc_mean * erfc((deltac - b) / denom) < (1 - 1e-3) * erfc((deltac - delta.mean()) / denom)


@settings(max_examples=400, deadline=None)
@given(st.integers(0, 10 ** 6), st.floats(0.01, 30.0), st.floats(0.1, 20.0), st.floats(0.05, 10.0), st.floats(0.6, 200.0),
       st.floats(1e-6, 1.9), st.booleans(), st.floats(0.0, 3.0), st.floats(-2.0, 2.0))
def test_no_cell_is_ionized_where_the_rule_skips(seed, sigma, deltac, denom, zeta, fc_mean, linear, skew, shift):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((8, 8, 8))
    d = sigma * (np.expm1(skew * x) if skew > 0.1 else x) / max(skew, 1.0) + shift * sigma
    # the bound of the rows pass: moduli of each line's modes
    X = np.abs(np.fft.rfft(d, axis=2)) / 8
    bound = (X[..., 0] + 2 * X[..., 1:].sum(-1)).max()
    assert bound >= np.abs(d).max() * (1 - 1e-12)
    if not stays_neutral(d, bound, deltac, denom, zeta, fc_mean, linear):
        return
    f = erfc((deltac - d) / denom)
    if not linear:
        f = f * (fc_mean / f.mean())
    assert not (zeta * f >= 1.0).any()
