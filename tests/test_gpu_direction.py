"""The preconditioned search direction at the edges of its kernel's forms.

One chain's direction is kept in registers up to 8 and 16 coordinates per thread of a
1024-thread workgroup (n * ndof = 8192 and 16384) and streamed above; the column solve gives
each lane ceil(n / 64) consecutive beads.  A search capped at k iterations returns iterate
x_k, so the correction pairs are known exactly (the gradients come from the same kernel): the
step x_{k+1} - x_k has to be parallel to the two-loop recursion's direction on those pairs
(Nocedal & Wright, Alg. 7.4) with scipy's banded solves as P^-1.  The bar on the directions'
sine, 1e-8: P's condition number, 4 (m / betan^2) / sigma <= 1e5 here, times the rounding
2^-53 and the pairs' m^2 = 64 products is 7e-10, and the difference of two iterates adds
2^-53 |x| / |step| <= 1e-10.
"""
import numpy as np
import pytest
import scipy.linalg as sl

from rptunnel import Pes, Ring, specs

pytestmark = pytest.mark.gpu

SIGMA, M = 0.05, 3


def _line(sp, n):
    k = np.arange(1, n + 1)
    return (np.outer(sp.well1, n - k) + np.outer(sp.well2, k - 1)) / (n - 1)


def _solve(sp, n, betan, v):
    out = np.empty_like(v)
    for d in range(sp.ndof):
        k = sp.mass[d // sp.ndim] / betan ** 2
        ab = np.zeros((2, n))
        ab[0] = 2.0 * k + SIGMA
        ab[1, :-1] = -k
        out[d] = sl.solveh_banded(ab, v[d], lower=True)
    return out


def _direction(sp, n, betan, g, S, Y):
    q, al = g.copy(), []
    for s, y in zip(S[::-1], Y[::-1]):
        al.append(np.vdot(s, q) / np.vdot(s, y))
        q -= al[-1] * y
    r = _solve(sp, n, betan, q)
    if S:
        r *= np.vdot(S[-1], Y[-1]) / np.vdot(Y[-1], _solve(sp, n, betan, Y[-1]))
    for s, y, a in zip(S, Y, al[::-1]):
        r += s * (a - np.vdot(y, r) / np.vdot(s, y))
    return -r


@pytest.mark.parametrize("ndof,ns", [(27, [2, 3, 63, 64, 65, 128, 303]), (27, [304, 449, 512, 606]),
                                     (27, [607, 1024]), (15, [2, 1023, 1024]), (30, [273, 274, 546, 547])])
def test_preconditioned_direction(ndof, ns):
    sp = specs.evb(natom=ndof // 3)
    pes = Pes(sp)
    betan = [8.0 + 0.5 * (c % 3) for c in range(len(ns))]
    ring = Ring(pes, sp.mass, ns, betan, sp.well1, sp.well2)
    ring.set_preconditioner(SIGMA)
    x0 = [_line(sp, n) for n in ns]
    xs, gs, its = [x0], [ring.UMforceenergy(x0)[0]], []
    for k in range(1, 6):
        x, _, it, _ = ring.instanton(x0, pgtol=1e-14, factr=0.0, m=M, maxiter=k)
        xs.append(x)
        gs.append(ring.UMforceenergy(x)[0])
        its.append(it)
    checked = 0
    for c, n in enumerate(ns):
        S, Y = [], []
        for k in range(5):
            if its[k][c] < k + 1:
                break
            step, y = xs[k + 1][c] - xs[k][c], gs[k + 1][c] - gs[k][c]
            d = _direction(sp, n, betan[c], gs[k][c], S, Y)
            scale = np.abs(xs[k][c]).max() / np.abs(step).max()
            if scale > 1e5:  # a step too small to tell its direction from two iterates
                break
            d, u = d / np.linalg.norm(d), step / np.linalg.norm(step)
            assert np.linalg.norm(d - u) <= 1e-8, (n, k, np.linalg.norm(d - u))
            checked += 1
            assert np.vdot(step, y) > 2.2e-16 * np.vdot(y, y)
            S, Y = (S + [step])[-M:], (Y + [y])[-M:]
    assert checked >= 3 * len(ns)
