"""The EVB Hessian blocks on the matrix cores at the edges of their tiles.

Bead counts on both sides of multiples of 16; 6 to 30 dofs (one and two dof tiles, last K-chunk
full and not); wells related by no exchange, a pair in the first, the last or both dof tiles, and
a cycle.  Reference: the oracle's Vdoubleprime inside its UMhessian band (instantonmod.f90:155-217),
normwise 1e-11 as the other band tests: sums of 2 M products, 2^-53 each, with M <= 30.
"""
from dataclasses import replace

import numpy as np
import pytest

import oracle as O
from helpers import oracle_pes, rel
from rptunnel import Pes, Ring, specs

pytestmark = pytest.mark.gpu


def _evb(natom, perm=None):
    sp = specs.evb(natom=natom)
    if perm is None:
        return sp
    perm = np.array(perm, dtype=np.int32)
    return replace(sp, ip=perm, well2=sp.well1.reshape(-1, 3)[np.argsort(perm)].reshape(-1))


CASES = {
    "evb": lambda: _evb(9),
    "evb6": lambda: _evb(2),
    "evb15": lambda: _evb(5),
    "evb18": lambda: _evb(6),
    "evb30": lambda: _evb(10),
    "same": lambda: _evb(9, range(9)),
    "last": lambda: _evb(9, [0, 1, 2, 3, 4, 5, 6, 8, 7]),
    "cycle": lambda: _evb(9, [4, 1, 2, 3, 8, 5, 6, 7, 0]),
}


@pytest.mark.parametrize("name", CASES)
def test_blocks(name):
    sp = CASES[name]()
    ns = [2, 15, 16, 17, 33, 64]
    rng = np.random.default_rng(5)
    end = sp.well1 + 0.4 if np.array_equal(sp.well1, sp.well2) else sp.well2
    chains = []
    for n in ns:
        t = np.linspace(0.0, 1.0, n)
        chains.append(np.outer(sp.well1, 1.0 - t) + np.outer(end, t)
                      + 0.05 * rng.standard_normal((sp.ndof, n)))
    betan = [20.0 + k for k in range(len(ns))]
    ring = Ring(Pes(sp), sp.mass, ns, betan, sp.well1, sp.well2)
    ring.set_x(chains)
    op = oracle_pes(sp)
    for c, n in enumerate(ns):
        oc = O.Chain(n, sp.ndim, sp.natom, sp.mass, betan[c], True)
        for single in (False, True):
            assert rel(ring.UMhessian(c, single), oc.UMhessian(op, chains[c], single)) <= 1e-11, (n, single)
            # the potential's part alone, without the springs on the diagonal
            got, want = ring.UMhessian(c, single)[1:-1], oc.UMhessian(op, chains[c], single)[1:-1]
            assert rel(got, want) <= 1e-11, (n, single)
