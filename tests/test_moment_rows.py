'''Moment rows of the product table (csrc/gen_rys_table.py): the Taylor series
of the highest Boys moment and of exp(-x) and the downward recursion, in the
kernels' order, against mpmath's incomplete gamma function.  Twelve Horner
steps and up to five recursion steps of positive terms: at most 15 roundings of
2.2e-16.'''
import os

import mpmath as mp
import numpy as np
import pytest

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                     'gpu4pyscf_amd', 'csrc', 'rys_table.npz')


def _boys(m, x):
    a = m + mp.mpf(1) / 2
    return mp.gammainc(a, 0, x) / (2 * mp.mpf(x)**a) if x else mp.mpf(1) / (2 * m + 1)


@pytest.mark.parametrize('n', [1, 2, 3])
def test_moments_from_rows(n):
    mp.mp.dps = 40
    t = np.load(TABLE)
    rows, step, xmax = t[f'moments{n}'], float(t['moment_step']), float(t['xmax'][n - 1])
    assert rows.shape[1] == 14 and (len(rows) - .5) * step >= xmax
    top = 2 * n - 1
    rng = np.random.default_rng(n)
    edges = [(g + .5) * step for g in (0, 1, 40)]
    xs = [0., 1e-9, .25, xmax - 1e-9] + edges + [e - 1e-12 for e in edges] + \
        list(rng.uniform(0, xmax, 40))
    for x in xs:
        g = min(int(x / step + .5), len(rows) - 1)
        d = g * step - x
        s = rows[g, 11]
        for k in range(10, -1, -1):
            s = s * d + rows[g, k]
        e = 1. / 479001600
        for k in range(11, -1, -1):
            e = e * d + 1. / float(mp.factorial(k))
        e *= rows[g, 12]
        f = s
        for m in range(top, -1, -1):
            ref = float(_boys(m, x))
            assert abs(f - ref) <= 15 * 2.2e-16 * ref, (x, m)
            if m:
                f = (2 * x * f + e) * (1. / (2 * m - 1))
