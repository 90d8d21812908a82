"""The work model's operation counts of the library's clipping pass, counted by
running a restatement of the pass (cgspline_amd/csrc/cgs_clip_wave.hpp and the
helpers of cgs_device.hpp that it calls) on numbers that count what is done to
them."""
from __future__ import annotations

import math

import pytest

from cgspline_amd import workmodel


class Num:
    """A number that counts additions, subtractions, products, quotients, roots,
    minima, maxima and compares; signs and absolute values are free."""
    ops = 0

    def __init__(self, v):
        self.v = float(v)

    def _op(self, o, f):
        Num.ops += 1
        return Num(f(self.v, o.v if isinstance(o, Num) else o))

    def __add__(self, o): return self._op(o, lambda a, b: a + b)
    def __sub__(self, o): return self._op(o, lambda a, b: a - b)
    def __rsub__(self, o): return Num(o)._op(self, lambda a, b: a - b)
    def __mul__(self, o): return self._op(o, lambda a, b: a * b)
    __rmul__ = __mul__
    def __truediv__(self, o): return self._op(o, lambda a, b: a / b if b else math.inf)
    def __rtruediv__(self, o): return Num(o) / self
    def __neg__(self): return Num(-self.v)
    def __abs__(self): return Num(abs(self.v))
    def __lt__(self, o): return bool(self._op(o, lambda a, b: a < b).v)
    def __gt__(self, o): return bool(self._op(o, lambda a, b: a > b).v)
    def __le__(self, o): return bool(self._op(o, lambda a, b: a <= b).v)
    def __ge__(self, o): return bool(self._op(o, lambda a, b: a >= b).v)


def fmin(a, b): return a._op(b, min)
def fmax(a, b): return a._op(b, max)


def root(a):
    Num.ops += 1
    return Num(math.sqrt(a.v))


def both(*conditions):
    """All of the conditions, each evaluated (straight-line code)."""
    return all(list(conditions))


def tolerance(p):
    t0, t1 = [p[3][k] - p[12][k] for k in (0, 1)], [p[15][k] - p[0][k] for k in (0, 1)]
    return both(t0[0] * t0[0] + t0[1] * t0[1] < 2.0 ** -24, t1[0] * t1[0] + t1[1] * t1[1] < 2.0 ** -24)


def hull_edge(lower, upper, A, B):
    q = A[1] - B[1]
    steep = abs(q) > 1e-7
    t = A[1] / q
    s = (1.0 - t) * A[0] + t * B[0]
    both(steep, 0.0 <= t, t <= 1.0)
    return fmin(lower, s), fmax(upper, s)


def to_hull(p):
    """A pass up to the interval it keeps."""
    tolerance(p)
    L = [(p[15][k] - p[0][k]) + (p[12][k] - p[3][k]) for k in (0, 1)]
    length = root(L[0] * L[0] + L[1] * L[1])
    if not abs(length) <= 1e-7:
        inv = 1.0 / length
        L = [L[0] * inv, L[1] * inv]
    N = [-L[1], L[0]]
    top, bot = [], []
    for i in range(4):
        d = [N[0] * p[4 * k + i][0] + N[1] * p[4 * k + i][1] for k in range(4)]
        hi = lo = d[0]
        for x in d[1:]:
            hi, lo = fmax(hi, x), fmin(lo, x)
        top.append(hi)
        bot.append(lo)
    lower, upper = Num(1.0), Num(0.0)
    x = [Num(0.0), Num(1 / 3), Num(2 / 3), Num(1.0)]
    P1, P2 = (x[0], bot[0]), (x[1], bot[1])
    for P3 in [(x[2], bot[2]), (x[3], bot[3]), (x[3], top[3]), (x[2], top[2]), (x[1], top[1]), (x[0], top[0]),
               (x[0], bot[0])]:
        P, Q = (P2[0] - P1[0], P2[1] - P1[1]), (P3[0] - P1[0], P3[1] - P1[1])
        ccw = P[0] * Q[1] - P[1] * Q[0] >= 0.0
        lower, upper = hull_edge(lower, upper, P1, P2)
        P1, P2 = (P2 if ccw else P1), P3
    lower, upper = hull_edge(lower, upper, P1, P2)
    lower = lower * (255 / 256)
    upper = upper + (1.0 - upper) * (1 / 256)
    delta = upper - lower
    both(delta > 0.8, delta < 0.0)
    return lower, upper


def slice1(c, u, iu, vv, ivv):
    c0, c1, c2, c3 = c
    p6, p5, c2 = u * c1 + iu * c0, u * c2 + iu * c1, u * c3 + iu * c2
    p8, c1 = u * p5 + iu * p6, u * c2 + iu * p5
    c0 = u * c1 + iu * p8
    p6, p5, c1 = ivv * c2 + vv * c3, ivv * c1 + vv * c2, ivv * c0 + vv * c1
    p8, c2 = ivv * p5 + vv * p6, ivv * c1 + vv * p5
    return c0, c1, c2, ivv * c2 + vv * p8


def clip(p):
    lower, upper = to_hull(p)
    mn, mx, size = Num(0.0), Num(1.0), Num(1.0)
    a, b = mn + size * lower, mx - size * (1.0 - upper)
    b - a
    iu = 1.0 - lower
    vv = (upper - lower) / iu
    ivv = 1.0 - vv
    for r in range(4):
        for k in (0, 1):
            slice1([p[4 * r + i][k] for i in range(4)], lower, iu, vv, ivv)


def split(p):
    to_hull(p)
    size = 0.5 * Num(1.0)
    Num(0.0) + size
    half = lambda x, y: 0.5 * x + 0.5 * y   # noqa: E731
    for r in range(4):
        for k in (0, 1):
            c = [p[4 * r + i][k] for i in range(4)]
            a, b, e = half(c[0], c[1]), half(c[1], c[2]), half(c[2], c[3])
            d, f = half(a, b), half(b, e)
            half(d, f)


def triangle(P, A, B):
    p, q = (A[0] - P[0], A[1] - P[1]), (B[0] - P[0], B[1] - P[1])
    det = p[0] * q[1] - q[0] * p[1]
    abs(det) < 2.0 ** -80
    det = 1.0 / det
    u = det * (q[1] * -P[0] + -q[0] * -P[1])
    both(u < 0.0, u > 1.0)
    v = det * (-p[1] * -P[0] + p[0] * -P[1])
    both(v < 0.0, u + v > 1.0)
    return u, v


def converged(p):
    tolerance(p)
    size = mn = mx = (Num(0.5), Num(0.5))
    c = triangle(p[0], p[3], p[12])
    [mn[k] + c[k] * size[k] for k in (0, 1)]
    c = triangle(p[15], p[12], p[3])
    [mx[k] - c[k] * size[k] for k in (0, 1)]


def finite_test(p):
    fin = Num(0.0)
    for q in p:
        fin = fin + (0.0 * q[0] + 0.0 * q[1])
    fin <= 0.0


@pytest.mark.parametrize("event, body", [("clips", clip), ("splits", split), ("prunes", to_hull),
                                         ("converged", converged)])
def test_operations_of_a_pass(event, body):
    net = [(Num(0.1 + i % 4 + 0.13 * i), Num(0.37 * (i // 4) - 0.4 + 0.05 * i)) for i in range(16)]
    Num.ops = 0
    body(net)
    zero = dict.fromkeys(workmodel.GPU_EVENTS, 0)
    assert workmodel.flops_of_counts({**zero, event: 1}) == Num.ops


def test_projection_tests_its_points():
    Num.ops = 0
    finite_test([(Num(1.0), Num(2.0))] * 16)
    assert workmodel.L_PROJ == workmodel.F_PROJ + Num.ops
