"""Ring entry points at the edges of their input: what is not finite, chains whose blocks take
more bytes than 32 bits count, tensors that are not on the ring's GPU, streams under capture."""
import numpy as np
import pytest
import torch

from rptunnel import Pes, Ring, RpError, autograd, specs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom,value", [(9, np.nan), (9, np.copysign(np.nan, -1.0)), (9, np.inf), (9, -np.inf),
                                         (5, np.copysign(np.nan, -1.0))])
@pytest.mark.parametrize("bead", [0, 16, 32])
def test_inertia_of_a_chain_that_is_not_finite(natom, value, bead):
    """A chain with a NaN or an infinity: its determinant is NaN with no eigenvalue counted
    negative, the other chains keep theirs bit for bit, and a search for its lowest eigenvalue
    is refused."""
    sp = specs.evb(natom=natom)
    ns = [40, 33, 64, 2]
    rng = np.random.default_rng(0)
    xs = [sp.well1[:, None] + 0.01 * rng.standard_normal((sp.ndof, n)) for n in ns]
    ring = Ring(Pes(sp), sp.mass, ns, [2000.0 / n for n in ns], sp.well1, sp.well1)
    ring.set_x(xs)
    want, nn, _ = ring.logdet(skip_lowest=False)
    assert np.all(np.isfinite(want)) and np.all(nn == 0)
    xs[1][sp.ndof // 2, bead] = value
    ring.set_x(xs)
    got, nn, _ = ring.logdet(skip_lowest=False)
    assert np.isnan(got[1]) and np.all(nn == 0), nn
    assert np.array_equal(got[[0, 2, 3]], want[[0, 2, 3]])
    with pytest.raises(RpError):
        ring.logdet(skip_lowest=True)
    ring.close()


def test_determinant_of_a_chain_beyond_4_gib_of_blocks():
    """530,000 beads of 32 dofs are 4.3 GB of blocks; the beads past the 4 GiB mark sit elsewhere
    in the potential than all others.  The quartic's dofs are separable and alike here, so the
    determinant is a scalar recurrence over the beads to the 32nd power: with the reference's
    coupling S_0 = a_0, S_1 = a_1, S_i = a_i - 1 / (betan^4 S_{i-1}).  Bar, relative to a
    logarithm of 1.5e8: a few roundings of 1.1e-16 in each of 1.7e7 pivots, all alike and so
    adding up, are 1e-8, the logarithm's own rounding is as much; 2e-15 is 3e-7.  One wrong
    block of the 5,712 in question is 7."""
    D, n, mark, betan = 32, 530_000, 2 ** 32 // (32 * 32 * 8), 100.0
    sp = specs.quartic(natom=D)
    h, x0, m = sp.dp[0], sp.dp[1], sp.mass[0]
    x = np.full((D, n), x0)
    x[:, mark:] = 0.8 * x0
    ring = Ring(Pes(sp), sp.mass, [n], [betan], sp.well1, sp.well2)
    ring.set_x([x])
    ld, nn, _ = ring.logdet(skip_lowest=False)
    with pytest.raises(RpError):  # the block solve's offsets stay within 31 bits
        ring.logdet(skip_lowest=True)
    ring.close()
    a = (4.0 * h / x0 ** 2 * (3.0 * x[0] ** 2 / x0 ** 2 - 1.0) / m + 2.0 / betan ** 2).tolist()
    want, s = np.log(a[0]), a[1]
    piv = [s]
    for v in a[2:]:
        s = v - 1.0 / (betan ** 4 * s)
        piv.append(s)
    want = D * (want + np.sum(np.log(piv)))
    assert nn[0] == 0 and abs(want) > 1e8
    assert abs(ld[0] - want) <= 2e-15 * abs(want), (ld[0], want)


def test_tensors_on_another_gpu_keep_off_the_ring_streams(monkeypatch):
    """A tensor whose GPU is not the ring's goes through the host entry points, first and second
    derivatives too, and comes back to its own GPU; none of the stream-ordered calls sees it.
    With one GPU at hand the ring is made to name another one."""
    sp = specs.coupled2d()
    ns = [5, 33]
    ring = Ring(Pes(sp), sp.mass, ns, [9.0, 7.0], sp.well1, sp.well2)
    x0 = torch.from_numpy(np.random.default_rng(2).standard_normal(2 * sum(ns)))
    v = torch.linspace(-1.0, 1.0, x0.numel(), dtype=torch.float64)

    def derivatives():
        x = x0.cuda().requires_grad_(True)
        u = autograd.ring_action(x, ring)
        (g,) = torch.autograd.grad((u * u).sum(), x, create_graph=True)
        (h,) = torch.autograd.grad(g @ v.cuda(), x)
        assert u.device == g.device == h.device == x.device
        return [t.detach().cpu() for t in (u, g, h)]

    assert ring.device == torch.cuda.current_device()
    want = derivatives()
    ring.device += 1
    monkeypatch.setattr(autograd, "_call", lambda *a: pytest.fail("a stream-ordered call"))
    for got, ref in zip(derivatives(), want):
        assert torch.allclose(got, ref, rtol=1e-12, atol=0.0)
    ring.close()


@pytest.mark.parametrize("used_before", [False, True])
def test_evaluations_are_refused_under_capture(used_before):
    """A ring's evaluation under capture is an error that leaves the capture, the graph and the
    ring as they were: the graph replays what else it holds, the ring's later calls are right."""
    sp = specs.coupled2d()
    ns = [5, 33]
    ring = Ring(Pes(sp), sp.mass, ns, [9.0, 7.0], sp.well1, sp.well2)
    rng = np.random.default_rng(2)
    chains = [0.3 * rng.standard_normal((2, n)) for n in ns]
    flat = torch.from_numpy(ring.pack(chains)).cuda()
    if used_before:
        autograd.ring_action(flat + 1.0, ring)
    a = torch.arange(4.0, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        b = a + 1.0
        with pytest.raises(RpError, match="captured"):
            autograd.ring_action(flat, ring)
        c = b * 2.0
    for k in range(3):
        a.fill_(float(k))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.all(c == 2.0 * (k + 1))
        x = (flat * (1.0 + k)).requires_grad_(True)
        u = autograd.ring_action(x, ring)
        (g,) = torch.autograd.grad(u.sum(), x)
        gw, ew = ring.UMforceenergy([(1.0 + k) * v for v in chains])
        assert np.allclose(u.detach().cpu().numpy(), ew, rtol=1e-13, atol=0.0)
        assert np.allclose(g.cpu().numpy(), ring.pack(gw), rtol=1e-12, atol=1e-15)
    ring.close()
