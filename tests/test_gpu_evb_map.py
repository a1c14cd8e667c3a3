"""EVB maps between the wells that are accepted without being permutations: two atoms sent to
one, another to none.  The matrix-core kernels (ring action, Hessian blocks, batched step), which
hold the second well as a difference from the first, against the per-bead kernels, which read both
in full.  Bars as in the neighbouring tests: U_M and its gradient 1e-12, the band 1e-11, states
after 8 steps 1e-10, normwise relative."""
from dataclasses import replace

import numpy as np
import pytest

from helpers import rel
from rptunnel import Batch, Chain, Pes, Ring, specs

pytestmark = pytest.mark.gpu

# (atoms, map): none sent to the first, to the last, to one of the second dof tile, to several,
# a permutation
MAPS = [(9, [0, 1, 2, 3, 4, 5, 6, 7, 0]), (9, [8, 1, 2, 3, 4, 5, 6, 7, 8]), (9, [0, 1, 2, 3, 4, 5, 6, 4, 8]),
        (9, [3, 3, 3, 3, 3, 3, 3, 3, 3]), (5, [0, 1, 2, 3, 1]), (10, [9, 1, 2, 3, 4, 5, 6, 7, 8, 9]),
        (9, [1, 0, 2, 3, 4, 5, 6, 7, 8])]


@pytest.mark.parametrize("natom,ip", MAPS)
def test_maps_between_the_wells(natom, ip):
    sp = replace(specs.evb(natom=natom), ip=np.array(ip, dtype=np.int32))
    pes, n, betan = Pes(sp), 33, 60.0
    rng = np.random.default_rng(natom)
    t = (np.arange(n) + 1.0) / (n + 1.0)
    x = np.outer(sp.well1, 1 - t) + np.outer(sp.well2, t) + 0.05 * rng.standard_normal((sp.ndof, n))
    m = np.repeat(sp.mass, sp.ndim)
    k = m[:, None] / betan ** 2

    ring = Ring(pes, sp.mass, [n], [betan], sp.well1, sp.well2, fixedends=False)
    g, e = ring.UMforceenergy([x])
    gp, ep = pes.potforce_beads(x)
    dx = np.diff(x, axis=1)
    assert abs(e[0] - (np.sum(ep) + 0.5 * np.sum(k * dx ** 2))) <= 1e-12 * abs(e[0])
    gp[:, 1:] += k * dx
    gp[:, :-1] -= k * dx
    assert rel(g[0], gp) <= 1e-12
    band = ring.UMhessian(0)
    got, want = [], []
    for i in (0, 7, 16, n - 1):
        h = pes.Vdoubleprime(x[:, i]) / np.sqrt(np.outer(m, m))
        for r in range(1, sp.ndof):  # the bead's own part of the band, below the diagonal
            got.append(band[r, i * sp.ndof:(i + 1) * sp.ndof - r])
            want.append(np.diagonal(h, -r))
    assert rel(np.concatenate(got), np.concatenate(want)) <= 1e-11
    ring.close()

    noise = rng.standard_normal(8 * n * sp.ndof)
    p = 0.5 * rng.standard_normal(x.shape)
    ch = Chain(pes, n, sp.mass, betan, 20.0, 1.0, 1e-3, sp.well1, sp.well2)
    ch.set_state(x, p)
    for s in range(8):  # the per-bead kick
        ch.time_step_pile(noise[s * x.size:(s + 1) * x.size])
    b = Batch(pes, sp.mass, [dict(n=n, betan=betan, a=sp.well1, b=sp.well2, dbdl=sp.well2 - sp.well1)],
              20.0, 1.0, 1e-3)
    b.set_state(0, x, p)
    b.run(8, noise=noise[None])
    for got, want in zip(b.get_state(0), ch.get_state()):
        assert rel(got, want) <= 1e-10
    b.close()
