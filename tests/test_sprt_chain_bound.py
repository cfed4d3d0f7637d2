"""The SPRT walk's decision rule (csrc/sprt_rules.hpp, chain_band and
chain_no_return) against the reference's running product, on the host.

The device compares a log f_in + b log f_out with log A instead of forming the
product f_in^a f_out^b one factor at a time, and takes the decision only
outside a margin of 1e-14 (16 + n) + 1e-13 n max(|log f_in|, |log f_out|), one
for a walk over n positions.  The product of k <= n rounded factors is off by at
most k 2^-53 (1 + O(k 2^-53)), each logarithm by an ulp or two, so the margin is
at least fifty times the largest difference.  Checked over histories and
thresholds from ratios of 1e-5 to 0.95, thresholds exactly at a product, equal
and nearly equal delta and epsilon, and products that underflow: every decided
position agrees, and where the rule says that a product below e^-690 cannot come
back (the device asks once per 64 positions), the product never exceeds A again.
The walk that is built on the rule is checked in test_sprt_rules.py.
"""
import math

import numpy as np
import pytest

np.seterr(all="ignore")


def _threshold(eps, delta, m, m_s):
    c = (1 - delta) * math.log((1 - delta) / (1 - eps)) + delta * math.log(delta / eps)
    k = (1.0 / m * c) / m_s + 1
    prev = an = k
    for _ in range(10):
        an = k + math.log(prev)
        if abs(an - prev) < 1.5e-8:
            break
        prev = an
    return an


def _side(a, b, l_in, l_out, l_a, n):
    big = a * l_in + b * l_out
    margin = 1e-14 * (16 + n) + 1e-13 * n * max(abs(l_in), abs(l_out))
    side = np.where(big > l_a + margin, 1, np.where(big < l_a - margin, 0, 2))
    return np.where((side == 0) & (big < -690.0), 3, side)


@pytest.mark.parametrize("seed", range(6))
def test_decided_positions_match_the_product(seed):
    rng = np.random.default_rng(seed)
    decided = undecided = sunk = 0
    for trial in range(300):
        n = int(rng.integers(1, 4000))
        eps = float(10 ** rng.uniform(-5, -0.02))
        delta = float(rng.choice([eps, eps * (1 + 1e-12), eps / 10, 10 ** rng.uniform(-5, -0.02), (n // 2 + 1) / (n + 1)]))
        m, m_s = [(4, 1), (7, 3), (5, 10)][trial % 3]
        f_in, f_out = delta / eps, (1 - delta) / (1 - eps)
        bits = rng.random(n) < rng.choice([0.0, 0.02, delta, eps, 0.5, 1.0])
        factors = np.where(bits, f_in, f_out)
        product = np.multiply.accumulate(factors)  # one rounded factor at a time
        thr = [_threshold(eps, delta, m, m_s), float(product[rng.integers(n)])][trial % 2]
        if not thr > 0:
            continue
        a = np.cumsum(bits)
        b = np.arange(1, n + 1) - a
        side = _side(a.astype(float), b.astype(float), math.log(f_in), math.log(f_out), math.log(thr), n)
        # positions up to the reference's stop are the ones decided in a walk
        stop = int(np.argmax(product > thr)) if (product > thr).any() else n - 1
        low = np.flatnonzero(side[:stop + 1] == 3)
        if len(low):
            # the device leaves this rule at the first such position
            first = int(low[0])
            up = max(math.log(f_in), math.log(f_out), 0.0)
            if (n - (first & ~63)) * up * (1.0 + 1e-9) < 680.0 + math.log(thr):
                assert not (product[first:] > thr).any()
                sunk += 1
            stop = first - 1
        got, want = side[:stop + 1], (product > thr)[:stop + 1]
        assert np.array_equal(got[got != 2], want[got != 2].astype(int))
        decided += int((got != 2).sum())
        undecided += int((got == 2).sum())
    assert decided > 10000
    assert undecided > 0 and sunk > 0  # the margin and the underflow rule are met by these cases
