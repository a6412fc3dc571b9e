'''The one- to three-root Rys rules as the kernels form them (boys_moments and
rys_roots<N> of csrc/jk_class_kernels.h): moments from the rows of the product
table, reciprocals by a 23-bit estimate and two Newton steps, the start of the
three-root cubic in float and Newton quotients by the estimate alone, against
Gauss rules in 50 digits from mpmath's incomplete gamma function.

The bound of each node and weight is first order in the roundings: every
operation may be off by 2 x 2.2e-16 of its result, every moment by 15 x 2.2e-16
(tests/test_moment_rows.py); what each of them changes is measured by repeating
the rule in 50 digits with that one result off by 1e-20.'''
import math
import os
import re

import mpmath as mp
import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, 'gpu4pyscf_amd', 'csrc')
U = 2.2e-16
EPS = mp.mpf('1e-20')
BITS = 23               # of the hardware's reciprocal and root estimates


def _estimate(x):
    m, e = math.frexp(x)
    return math.ldexp(math.floor(m * 2**BITS) / 2**BITS, e)


class Double:
    '''The kernel's operations in FP64, without fused ones.'''
    num = float

    def op(self, x):
        return x

    def rcp(self, x):
        r = _estimate(1. / x)
        r = (1. - x * r) * r + r
        return (1. - x * r) * r + r

    def div(self, a, b):
        r = _estimate(1. / b)
        r = (1. - b * r) * r + r
        q = a * r
        return (a - b * q) * r + q

    def sqrt(self, x):
        y = _estimate(1. / math.sqrt(x))
        y = y * (.5 - x * y * (.5 * y)) + y
        y = y * (.5 - x * y * (.5 * y)) + y
        s = x * y
        return (x - s * s) * (.5 * y) + s

    def quotient(self, a, b):
        return a * _estimate(1. / b)


class Perturbed:
    '''The same in 50 digits, operation `at` off by EPS.'''
    num = mp.mpf

    def __init__(self, at=-1):
        self.at, self.n = at, 0

    def op(self, x):
        self.n += 1
        return x * (1 + EPS) if self.n - 1 == self.at else x

    def rcp(self, x):
        return self.op(1 / x)

    def div(self, a, b):
        return self.op(a / b)

    def sqrt(self, x):
        return self.op(mp.sqrt(x))

    def quotient(self, a, b):
        return self.op(a / b * (1 - mp.mpf(2)**-BITS))


def _rule(n, f, c):
    '''(nodes, weights) of the moments f with the operations c.'''
    o = c.op
    if n == 1:
        return [c.div(f[1], f[0])], [f[0]]
    if n == 2:
        idet = c.rcp(o(o(f[1] * f[1]) - o(f[0] * f[2])))
        c1 = o(o(o(f[0] * f[3]) - o(f[1] * f[2])) * idet)
        c0 = o(o(o(f[2] * f[2]) - o(f[1] * f[3])) * idet)
        disc = c.sqrt(o(o(c1 * c1) - 4 * c0))
        u2 = o((disc - c1) / 2)
        u1 = c.div(c0, u2)
        w1 = c.div(o(o(u2 * f[0]) - f[1]), o(u2 - u1))
        return [u1, u2], [w1, o(f[0] - w1)]
    third = c.num(1) / 3
    r0 = c.rcp(f[0])
    a0 = o(f[1] * r0)
    n1, n2, n3, n4 = (o(f[k + 1] - o(a0 * f[k])) for k in (1, 2, 3, 4))
    rn1 = c.rcp(n1)
    q1 = o(n2 * rn1)
    a1, b1 = o(q1 - a0), o(n1 * r0)
    m2 = o(o(n3 - o(a1 * n2)) - o(b1 * f[2]))
    m3 = o(o(n4 - o(a1 * n3)) - o(b1 * f[3]))
    rm2 = c.rcp(m2)
    a2, b2 = o(o(m3 * rm2) - q1), o(m2 * rn1)
    c2 = -o(o(a0 + a1) + a2)
    c1 = o(o(o(o(o(a0 * a1) + o(a0 * a2)) + o(a1 * a2)) - b1) - b2)
    c0 = o(o(o(b2 * a0) + o(b1 * a2)) - o(o(a0 * a1) * a2))
    p = o(c1 - o(o(c2 * c2) * third))
    q = o(o(o(o(o(c2 * c2) * c2) * (c.num(2) / 27)) - o(o(c2 * c1) * third)) + c0)
    f32 = np.float32
    rr = np.sqrt(f32(float(-p)) * f32(1 / 3))
    phi = np.arccos(np.clip(-f32(float(q)) / (f32(2) * rr * rr * rr), f32(-1), f32(1)))
    nodes, weights = [], []
    for shift in (2 * math.pi, -2 * math.pi, 0.):
        start = f32(2) * rr * np.cos((phi + f32(shift)) * f32(1 / 3))
        v = o(c.num(float(start)) - o(c2 * third))
        for _ in range(2):
            p1 = o(v - a0)
            p2 = o(o(o(v - a1) * p1) - b1)
            d2 = o(p1 + o(v - a1))
            p3 = o(o(o(v - a2) * p2) - o(b2 * p1))
            d3 = o(o(p2 + o(o(v - a2) * d2)) - b2)
            v = o(v - c.quotient(p3, d3))
        p1 = o(v - a0)
        p2 = o(o(o(v - a1) * p1) - b1)
        nodes.append(v)
        weights.append(c.rcp(o(o(r0 + o(o(p1 * p1) * rn1)) + o(o(p2 * p2) * rm2))))
    return nodes, weights


def _exact_moments(n, x):
    out = []
    for m in range(2 * n):
        a = m + mp.mpf(1) / 2
        out.append(mp.gammainc(a, 0, x) / (2 * mp.mpf(x)**a) if x else mp.mpf(1) / (2 * m + 1))
    return out


def _gauss(n, mu):
    '''Gauss rule of the moments: the orthogonal polynomial's coefficients, its
    roots, the weights from the moments.'''
    c = mp.lu_solve(mp.matrix([[mu[i + j] for j in range(n)] for i in range(n)]),
                    mp.matrix([-mu[n + i] for i in range(n)]))
    u = sorted(mp.re(r) for r in mp.polyroots([1] + [c[n - 1 - k] for k in range(n)],
                                              maxsteps=200, extraprec=200))
    w = mp.lu_solve(mp.matrix([[r**k for r in u] for k in range(n)]),
                    mp.matrix([mu[k] for k in range(n)]))
    return u, list(w)


def _table_moments(rows, step, n, x):
    g = min(int(x / step + .5), len(rows) - 1)
    d = g * step - x
    s, e = rows[g, 11], 1. / 479001600
    for k in range(10, -1, -1):
        s = s * d + rows[g, k]
    for k in range(11, -1, -1):
        e = e * d + 1. / math.factorial(k)
    e *= rows[g, 12]
    f = [0.] * (2 * n)
    f[2 * n - 1] = s
    for m in range(2 * n - 1, 0, -1):
        f[m - 1] = (2 * x * f[m] + e) * (1. / (2 * m - 1))
    return [float(v) for v in f]


@pytest.mark.parametrize('n', [1, 2, 3])
def test_rules_of_the_moment_rows(n):
    mp.mp.dps = 50
    t = np.load(os.path.join(CSRC, 'rys_table.npz'))
    rows, step, xmax = t[f'moments{n}'], float(t['moment_step']), float(t['xmax'][n - 1])
    rng = np.random.default_rng(40 + n)
    xs = [0., 1e-9, .148, .25, .25 - 1e-13, 1., xmax - 1e-9, 20.25] + list(rng.uniform(0, 3, 15)) + \
        list(rng.uniform(0, xmax, 25))
    worst = 0.
    for x in xs:
        mu = _exact_moments(n, x)
        ref = sum(_gauss(n, mu), [])
        got = sum(_rule(n, _table_moments(rows, step, n, x), Double()), [])
        c = Perturbed()
        base = sum(_rule(n, mu, c), [])
        bound = [mp.mpf(0)] * (2 * n)
        for k in range(c.n):
            for i, v in enumerate(sum(_rule(n, mu, Perturbed(k)), [])):
                bound[i] += 2 * U * abs(v - base[i]) / EPS
        for k in range(2 * n):
            off = [m * (1 + EPS) if j == k else m for j, m in enumerate(mu)]
            for i, v in enumerate(sum(_rule(n, off, Perturbed()), [])):
                bound[i] += 15 * U * abs(v - base[i]) / EPS
        for i in range(2 * n):
            assert abs(got[i] - ref[i]) <= bound[i], (x, i, float(abs(got[i] / ref[i] - 1)))
            worst = max(worst, float(abs(got[i] / ref[i] - 1)))
    print(f'[{n} roots] largest relative error of a node or weight {worst:.2e}')


def test_large_x_constants_of_the_kernel():
    '''Half of the 2n-point Gauss-Hermite rule: squared nodes and weights.'''
    text = open(os.path.join(CSRC, 'jk_class_kernels.h')).read()
    lr, lw = ([float(v) for v in re.findall(r'[\d.]+', re.search(
        r'double %s\[6\] = \{([^}]*)\}' % name, text).group(1))] for name in ('LR', 'LW'))
    for n in (1, 2, 3):
        h, w = np.polynomial.hermite.hermgauss(2 * n)
        sl = slice(n * (n - 1) // 2, n * (n + 1) // 2)
        assert abs(np.array(lr[sl]) / h[n:]**2 - 1).max() < 1e-14
        assert abs(np.array(lw[sl]) / w[n:] - 1).max() < 1e-14
