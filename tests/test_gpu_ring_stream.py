"""The EVB action kernel at the edges of its 16-bead tiles, and the stream-ordered entry points
under torch.autograd: any stream, in order with the synchronous calls on the same ring."""
from dataclasses import replace

import numpy as np
import pytest
import torch

import oracle as O
from helpers import oracle_pes, rand_chain, rel
from rptunnel import Pes, Ring, RpError, specs
from rptunnel.autograd import ring_action

pytestmark = pytest.mark.gpu


def _evb(perm=None, natom=9):
    sp = specs.evb(natom=natom)
    return sp if perm is None else replace(sp, ip=np.array(perm, dtype=np.int32))


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("natom,perm", [(9, None), (5, None), (10, None), (9, [0, 1, 2, 3, 4, 5, 6, 8, 7]),
                                        (9, [4, 1, 2, 3, 8, 5, 6, 7, 0]), (9, list(range(9)))])
def test_evb_action_at_tile_edges(natom, perm, fixed):
    """U_M and its gradient, 1e-12 normwise relative (the bar of test_gpu_ring.py)."""
    sp = _evb(perm, natom)
    op = oracle_pes(sp)
    ns = [2, 3, 15, 16, 17, 18, 31, 32, 33, 64, 129]
    betan = [3.0 + k for k in range(len(ns))]
    xs = [rand_chain(sp, n, 7 + n, 0.05) for n in ns]
    ring = Ring(Pes(sp), sp.mass, ns, betan, sp.well1, sp.well2, fixedends=fixed)
    g, e = ring.UMforceenergy(xs)
    for k, n in enumerate(ns):
        oc = O.Chain(n, sp.ndim, sp.natom, sp.mass, betan[k], fixed)
        ge, ee = oc.UMforceenergy(op, xs[k], sp.well1, sp.well2)
        assert rel(g[k], ge) <= 1e-12 and abs(e[k] - ee) <= 1e-12 * abs(ee), (n, rel(g[k], ge))
    assert np.allclose(ring.UM(), e, rtol=1e-14)
    ring.close()


def test_streams_and_synchronous_calls_in_order():
    """ring_action on two streams and the ring's synchronous calls in between, no waits: each
    result is the one its own coordinates give."""
    sp = specs.evb()
    ns, betan = [40, 300, 17], [20.0, 9.0, 30.0]
    ring = Ring(Pes(sp), sp.mass, ns, betan, sp.well1, sp.well2)
    sets = [[rand_chain(sp, n, 50 * k + n, 0.05) for n in ns] for k in range(4)]
    want = [ring.UMforceenergy(c) for c in sets]
    flat = [torch.from_numpy(ring.pack(c)).cuda() for c in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = []
    for k in range(4):
        with torch.cuda.stream(streams[k % 2]):
            x = flat[k].clone().requires_grad_(True)
            u = ring_action(x, ring)
            (g,) = torch.autograd.grad(u.sum(), x)
            got.append((u, g))
        if k == 1:  # a synchronous call right behind the queued work: it sees that work's x
            assert np.allclose(ring.UM(), want[k][1], rtol=1e-13)
            assert np.array_equal(np.concatenate([c.reshape(-1) for c in ring.get_x()]), ring.pack(sets[k]))
    torch.cuda.synchronize()
    for (u, g), (gw, ew) in zip(got, want):
        assert rel(u.detach().cpu().numpy(), ew) <= 1e-13
        assert rel(g.cpu().numpy(), np.concatenate([c.reshape(-1) for c in gw])) <= 1e-13
    ring.close()


def test_types_sizes_and_host_potentials():
    sp = specs.coupled2d()
    ring = Ring(Pes(sp), sp.mass, [5, 3], [9.0, 7.0], sp.well1, sp.well2)
    xs = [rand_chain(sp, n, n, 0.05) for n in (5, 3)]
    g, e = ring.UMforceenergy(xs)
    flat = torch.from_numpy(ring.pack(xs))
    # float32 and a strided view are converted, as for host tensors
    for x in (flat.cuda().float(), torch.stack([flat, flat], dim=1).cuda()[:, 0]):
        x.requires_grad_(True)
        u = ring_action(x, ring)
        (gx,) = torch.autograd.grad(u.sum(), x)
        tol = 1e-5 if x.dtype == torch.float32 else 1e-13
        assert u.dtype == gx.dtype == x.dtype
        assert rel(u.detach().cpu().numpy(), e) <= tol
        assert rel(gx.cpu().numpy(), np.concatenate([c.reshape(-1) for c in g])) <= tol
    with pytest.raises(ValueError):
        ring_action(flat.cuda()[:-1], ring)
    # a potential on the host: the same values for a GPU tensor, through the host entry points
    pes = Pes.host(1, 2, lambda x: (x.copy(), 0.5 * np.sum(x * x, axis=0)))
    hring = Ring(pes, np.array([1.0, 2.0]), [4], [3.0], np.zeros(2), np.ones(2))
    x = torch.linspace(0.0, 1.0, 8, dtype=torch.float64)
    out = []
    for xx in (x.clone(), x.cuda()):
        xx.requires_grad_(True)
        u = ring_action(xx, hring)
        (gx,) = torch.autograd.grad(u.sum(), xx)
        out.append((u.detach().cpu(), gx.cpu()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    from rptunnel import _lib as L
    with pytest.raises(RpError):
        L.check(L.lib().rp_ring_action_stream(hring.h, x.cuda().data_ptr(), x.cuda().data_ptr(), None, None))
