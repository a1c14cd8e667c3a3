"""Plans and workspaces kept between calls: a chain's fused propagation after any change of what
its plan was made from, and a ring's search after one of another size, equal those of fresh
objects bit for bit (the same kernels on the same numbers, sums in a fixed order)."""
import numpy as np
import pytest

from rptunnel import Chain, Pes, Ring, specs
from rptunnel._lib import RpError

pytestmark = pytest.mark.gpu

N, STEPS = 33, 6


def _line(sp, n):
    k = np.arange(1, n + 1)
    return (np.outer(sp.well1, n - k) + np.outer(sp.well2, k - 1)) / (n - 1)


def _chain(sp, pes, b, cursor):
    ch = Chain(pes, N, sp.mass, 2000.0 / (N + 1), 20.0, 1.0, 1e-3, sp.well1, b)
    ch.set_rng(7, 3, cursor)
    return ch


@pytest.mark.parametrize("thermostat", ["pile", "nm"])
def test_chain_calls_match_fresh_chains(thermostat):
    sp = specs.evb()
    pes = Pes(sp)
    lampath, path = specs.linear_path(sp.well1, sp.well2, npath=3)
    d1, d2 = sp.well2 - sp.well1, 0.5 * (sp.well2 - sp.well1)
    b1, b2 = sp.well2.copy(), sp.well1 + 0.6 * (sp.well2 - sp.well1)
    rng = np.random.default_rng(1)
    x, p = _line(sp, N), rng.standard_normal((sp.ndof, N))
    need = N * sp.ndof
    noise = rng.standard_normal(STEPS * need)

    def run(ch, dbdl, kw):
        if thermostat == "pile":
            return ch.propagate_pimd_pile(STEPS, dbdl, imin=1, **kw)[0]
        kw = {k: v for k, v in kw.items() if k == "noise"}
        return ch.propagate_pimd_nm(STEPS, dbdl, noutput=2, imin=1, **kw)

    kept = _chain(sp, pes, b1, 0)
    calls = [(d1, b1, {}), (d1, b1, {}), (d2, b1, {}), (d2, b1, {}), (d2, b2, {}), (d2, b2, dict(noise=noise)),
             (d2, b2, {}), (d2, b2, dict(dhdrlimit=1e9, xi=0.4)), (d2, b2, dict(dhdrlimit=1e9, xi=0.4)),
             (d2, b2, dict(noise=noise[:need // 2])), (d2, b2, {})]
    ends = b1
    kept.set_path(lampath, path)
    kept.set_state(x, p)
    cursor = 0
    for i, (dbdl, b, kw) in enumerate(calls):
        if b is not ends:
            kept.init_nm(sp.well1, b)
            ends = b
        kept.set_rng(7, 3, cursor) if i == 7 else None
        before, fresh = kept.get_state(), _chain(sp, pes, b, cursor)
        fresh.set_path(lampath, path)
        fresh.set_state(*before)
        if thermostat == "nm":  # the Poisson positions advance with the calls
            kept.set_rng(7, 3, cursor)
        if "noise" in kw and kw["noise"].size < need and thermostat == "pile":
            for ch in (kept, fresh):  # exhausted: refused, and the state stays
                with pytest.raises(RpError):
                    run(ch, dbdl, kw)
            assert all(np.array_equal(u, v) for u, v in zip(kept.get_state(), before))
            continue
        if "noise" in kw and kw["noise"].size < need:
            continue
        got, want = run(kept, dbdl, kw), run(fresh, dbdl, kw)
        assert got == want, i
        assert kept.cursor == fresh.cursor
        assert all(np.array_equal(u, v) for u, v in zip(kept.get_state(), fresh.get_state())), i
        cursor = kept.cursor


def test_search_after_a_larger_and_a_smaller_history():
    sp = specs.evb()
    pes = Pes(sp)
    ns = [17, 64, 65]
    x0 = [_line(sp, n) for n in ns]

    def ring():
        r = Ring(pes, sp.mass, ns, [8.0] * 3, sp.well1, sp.well2)
        r.set_preconditioner(0.05)
        return r

    kept = ring()
    for m, maxiter in ((3, 5), (8, 12), (2, 4), (8, 12)):
        got = kept.instanton(x0, m=m, maxiter=maxiter)
        want = ring().instanton(x0, m=m, maxiter=maxiter)
        for u, v in zip(got[0], want[0]):
            assert np.array_equal(u, v), m
        for u, v in zip(got[1:], want[1:]):
            assert np.array_equal(u, v), m


def test_state_halves():
    """x alone, p alone and both come back from the same polymer."""
    import ctypes as C

    from rptunnel import Batch
    from rptunnel import _lib as L
    sp = specs.quartic()
    pes = Pes(sp)
    a = np.array([sp.well1[0]])
    pols = [dict(n=n, betan=100.0 / (n + 1), xi=0.5, a=a, b=-a, dbdl=-2 * a, stream=i)
            for i, n in enumerate([2, 31, 256])]
    b = Batch(pes, sp.mass, pols, 20.0, 1.0, 1e-3, seed=1)
    for k, n in enumerate([2, 31, 256]):
        x, p = np.arange(1.0, n + 1)[None], -np.arange(1.0, n + 1)[None] - 0.5
        b.set_state(k, x, p)
        xg, pg = b.get_state(k)
        assert np.array_equal(xg, x) and np.array_equal(pg, p)
        for which, ref in ((0, x), (1, p)):
            out = np.zeros_like(ref)
            ptrs = [None, None]
            ptrs[which] = L.ptr(out)
            L.check(L.lib().rp_batch_get_state(b.h, C.c_int(k), ptrs[0], ptrs[1]))
            assert np.array_equal(out, ref)
