"""How far EM frequencies and log10 likelihoods summed in read order lie from correctly rounded sums, against
the exact scorer's guards, (2 + passes / 8) (n + 64) 2^-53 of a frequency and (n + 64) 2^-53 (n + |log10 likelihood|): within a quarter and a
tenth of them, over fits of a few passes and of dozens.  At 200,000 reads of one quality the differences
pass the guards' least values (2e-12 and 1e-8), which alone would not do there."""
import math

import numpy as np
import pytest

U = 2.0 ** -53


def em(r, exact, tol=1e-6):
    """fit_allele_frequencies over the likelihood ratios r[reads, 5]; sums in read order, or correctly rounded."""
    total = (lambda x: math.fsum(x)) if exact else (lambda x: float(np.cumsum(x)[-1]))
    f = np.array([0.5 + (r.argmax(1) == b).sum() for b in range(5)])
    f /= f.sum()
    for passes in range(1, 51):
        s = (((f[0] * r[:, 0] + f[1] * r[:, 1]) + f[2] * r[:, 2]) + f[3] * r[:, 3]) + f[4] * r[:, 4]
        w = f * r / s[:, None]
        ll = total(np.log10(s))
        last, f = f, np.array([total(w[:, b]) for b in range(5)]) / len(r)
        if np.abs(f - last).max() < tol:
            break
    return f, ll, passes


@pytest.mark.parametrize("n", [30, 300, 3000, 20000, 200000])
def test_sums_in_read_order(n):
    rng = np.random.default_rng(1)
    most_f = most_ll = 0.0
    passes_seen = set()
    mixes = ([15], [40]) if n == 200000 else ([40], [3], [2, 40]) if n == 20000 else (
        [15], [15, 16, 17], range(15, 40), [3], [4], [2, 3, 5], [10, 12], [2, 40], [40])
    for quals in mixes:
        for share in (0.02, 0.4):
            e = np.minimum(10.0 ** (-rng.choice(list(quals), n) / 10.0), 0.74)
            r = np.tile((e / 4.0 / (1.0 - e))[:, None], (1, 5))
            obs = np.where(rng.random(n) < 0.7 * e, rng.integers(0, 4, n), rng.random(n) < share)
            r[np.arange(n), obs.astype(int)] = 1.0
            f, ll, passes = em(r, False)
            f0, ll0, passes0 = em(r, True)
            assert passes == passes0
            passes_seen.add(passes)
            counts = f0 > 0.5 / n   # the frequencies that are printed
            rel = float((np.abs(f - f0) / f0)[counts].max())
            assert rel <= 0.25 * (2.0 + passes / 8.0) * (n + 64) * U
            assert abs(ll - ll0) <= 0.1 * (n + 64) * U * (n + abs(ll0))
            most_f, most_ll = max(most_f, rel), max(most_ll, abs(ll - ll0))
    if n == 200000:
        assert most_f > 2e-12 and most_ll > 1e-8
    else:
        assert min(passes_seen) <= 6 and max(passes_seen) >= 30   # easy fits and slow ones
    if n <= 3000:
        assert most_f < 2e-12 and most_ll < 1e-8
