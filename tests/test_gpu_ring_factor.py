"""The block factorisation of the ring Hessian for ndof <= 32 (matrix cores, from both ends of
a chain to its middle) at the edges of its tiles: ndof on both sides of 16 and of multiples of
4, chains down to 2 beads, positive definite and indefinite, against eigvalsh of the library's
own band (the blocks the factorisation reads).  Bars as in test_gpu_ring.py: log-determinants
1e-9 relative, the lowest eigenvalue 1e-8 relative, the negative count exact."""
import numpy as np
import pytest

import oracle as O
from rptunnel import Pes, Ring, specs

pytestmark = pytest.mark.gpu


def _dense(D, ndim, seed, shift):
    """V = d.K d/2 + 0.1 sum d^4 about x0, K dense with eigenvalues from 0.01 up, less shift."""
    rng = np.random.default_rng(seed)
    Q = rng.standard_normal((D, D))
    K = 0.05 * (Q @ Q.T) / D + (0.01 - shift) * np.eye(D)
    x0 = rng.standard_normal(D)

    def potforce(x):
        d = x - x0[:, None]
        return K @ d + 0.4 * d ** 3, 0.5 * np.sum(d * (K @ d), axis=0) + 0.1 * np.sum(d ** 4, axis=0)

    def hessian(x):
        d = x - x0[:, None]
        h = np.repeat(K[None], x.shape[1], axis=0)
        h[:, np.arange(D), np.arange(D)] += 1.2 * d.T ** 2
        return h

    mass = rng.uniform(600.0, 2500.0, D // ndim)
    return Pes.host(ndim, D // ndim, potforce, hessian), x0, mass


@pytest.mark.parametrize("shift", [0.0, 0.03])
@pytest.mark.parametrize("D,ndim", [(1, 1), (2, 2), (3, 1), (4, 1), (5, 1), (8, 2), (13, 1), (15, 3), (16, 1),
                                    (17, 1), (18, 3), (20, 2), (27, 3), (28, 1), (29, 1), (31, 1), (32, 2)])
def test_factorisation_against_eigvalsh(D, ndim, shift):
    pes, x0, mass = _dense(D, ndim, D, shift)
    ns = [2, 3, 4, 5, 6, 17]
    betan = [25.0, 40.0, 18.0, 30.0, 22.0, 35.0]
    rng = np.random.default_rng(D + 100)
    xs = [x0[:, None] + 0.1 * rng.standard_normal((D, n)) for n in ns]
    ring = Ring(pes, mass, ns, betan, x0, x0)
    ring.set_x(xs)
    ld, nn, eta = ring.logdet(singlewell=False, skip_lowest=False, want_eta=True)
    for k, n in enumerate(ns):
        ev = O.detj_eigs(ring.UMhessian(k, singlewell=False))
        assert nn[k] == np.sum(ev < 0), (n, nn[k], ev[:4])
        # an absolute floor: a sum of logarithms may pass near zero
        assert abs(ld[k] - O.lndetj0(ev)) <= 1e-9 * max(abs(O.lndetj0(ev)), 1.0), (n, ld[k])
        assert abs(eta[k] - ev[0]) <= 1e-8 * abs(ev[0]), (n, eta[k], ev[:3])
    ring.close()


def test_more_chains_than_run_at_once():
    """Every chain of a batch much larger than the device holds, against the same chains alone."""
    sp = specs.evb()
    pes = Pes(sp)
    rng = np.random.default_rng(3)
    ns = [int(v) for v in rng.integers(2, 40, 3000)]
    betan = [2000.0 / n for n in ns]
    xs = [sp.well1[:, None] + 0.01 * rng.standard_normal((27, n)) for n in ns]
    ring = Ring(pes, sp.mass, ns, betan, sp.well1, sp.well1)
    ring.set_x(xs)
    ld, nn, _ = ring.logdet(singlewell=False, skip_lowest=False)
    for k in (0, 1, 777, 1500, 2998, 2999):
        one = Ring(pes, sp.mass, [ns[k]], [betan[k]], sp.well1, sp.well1)
        one.set_x([xs[k]])
        l1, n1, _ = one.logdet(singlewell=False, skip_lowest=False)
        assert n1[0] == nn[k] and l1[0] == ld[k]
        one.close()
    ring.close()
