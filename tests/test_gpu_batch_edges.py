"""The batched step kernel at the edges of its tiles and dispatch, against the oracle.

A wave holds 16 beads of one half of a chain, so the bead counts here sit on both sides of
multiples of 16 per half, odd and even, down to 2.  Potentials cover every dof tiling, the EVB
permutations the kick's difference matrix depends on (none, one pair in the first or the
last dofs, a cycle over three atoms), many polymers per workgroup and, for few dofs, per MFMA
tile.  Bars as in test_gpu_batch.py: init_path 1e-12, states after 8 steps and TI sums 1e-10
normwise relative, stream cursors exact.
"""
from dataclasses import replace

import numpy as np
import pytest

import oracle as O
from helpers import oracle_pes, rel
from rptunnel import Batch, Pes, specs
from rptunnel.batch import ANDERSEN, LANGEVIN

pytestmark = pytest.mark.gpu

TAU, DT, GAMMA, BETA, SEED = 20.0, 1.0, 1e-3, 2000.0, 19


def _evb(perm, natom=9):
    sp = specs.evb(natom=natom)
    perm = np.array(perm, dtype=np.int32)
    return replace(sp, ip=perm, well2=sp.well1.reshape(-1, 3)[np.argsort(perm)].reshape(-1))


SPECS = {
    "quartic": specs.quartic,
    "quartic30": lambda: specs.quartic(ndim=3, natom=10),
    "coupled2d": specs.coupled2d,
    "harmonic3": lambda: specs.harmonic([0.02, 0.05, 0.01], [0.1, -0.2, 0.3], [1836.0] * 3),
    "evb": specs.evb,
    "evb15": lambda: specs.evb(natom=5),
    "evb_same": lambda: _evb(range(9)),
    "evb_last": lambda: _evb([0, 1, 2, 3, 4, 5, 6, 8, 7]),
    "evb_cycle": lambda: _evb([4, 1, 2, 3, 8, 5, 6, 7, 0]),
    "evb30": lambda: specs.evb(natom=10),
    "water1": lambda: specs.water_cluster(nmol=1),
    "water2": lambda: specs.water_cluster(nmol=2),
    "water6": lambda: specs.water_cluster(nmol=6),
}
EDGES = [2, 3, 4, 15, 16, 17, 31, 32, 33, 34, 47, 63, 64, 65, 66, 95, 97, 128, 129, 191, 224, 255, 256]
CASES = [("evb", EDGES), ("quartic", EDGES), ("water1", [2, 3, 33, 64, 255]),
         ("quartic30", [5, 32, 97, 256]), ("coupled2d", [3, 32, 97, 255]),
         ("harmonic3", [2, 33, 256]), ("evb15", [31, 64, 255]), ("evb_same", [33, 64]),
         ("evb_last", [33, 64]), ("evb_cycle", [17, 128]), ("evb30", [47, 192]),
         ("water2", [2, 17, 65, 200, 256]), ("water6", [3, 32, 33, 97, 128])]


def _path(sp):
    if sp.name == "water" and sp.natom > 3:
        return specs.arc_lampath(sp.extra["path"].T), np.ascontiguousarray(sp.extra["path"].T)
    # a straight line has to lead somewhere: away from the one well of some, and not through two
    # atoms of the water monomer
    one_well = sp.name == "water" or np.array_equal(sp.well1, sp.well2)
    return specs.linear_path(sp.well1, sp.well1 + 0.05 if one_well else sp.well2, npath=2)


def _polymers(sp, path, ns, count=1):
    a, b = path[:, 0], path[:, -1]
    return [dict(n=n, betan=BETA / (n + 1), xi=0.2 + 0.6 * (k % 7) / 7, a=a,
                 b=a + (0.2 + 0.6 * (k % 7) / 7) * (b - a), dbdl=b - a, stream=5 + 3 * k + 100 * i)
            for i, n in enumerate(ns) for k in range(count)]


def _check(sp, b, pols, which, steps, thermostat, noutput, lampath, path):
    op, opath = oracle_pes(sp), O.Path(lampath, path)
    start = {k: b.get_state(k) for k in which}
    b.run(steps, imin=1)
    sums, cnt, _ = b.ti_readout()
    cur, kcur = b.cursors(), b.kick_cursors()
    for k in which:
        pol = pols[k]
        nm = O.NM(pol["n"], sp.ndim, sp.natom, sp.mass, pol["betan"], TAU, DT, GAMMA, False, pol["a"], pol["b"])
        r = O.Rng(seed=SEED, stream=pol["stream"])
        xo, po = O.init_path(nm, opath, r, pol["xi"])
        assert rel(start[k][0], xo) <= 1e-12 and rel(start[k][1], po) <= 1e-12, (pol["n"], "init")
        if thermostat == LANGEVIN:
            xo, po, dho, _ = O.propagate_pile(nm, op, r, *start[k], steps, pol["dbdl"], imin=1)
        else:
            xo, po, dho = O.propagate_andersen(nm, op, r, *start[k], steps, pol["dbdl"], noutput, imin=1)
            assert kcur[k] == r.s.kcursor
        xg, pg = b.get_state(k)
        assert cur[k] == r.cursor and cnt[k] == steps - 1
        assert rel(xg, xo) <= 1e-10 and rel(pg, po) <= 1e-10, (pol["n"], rel(xg, xo), rel(pg, po))
        assert abs(sums[k] / (steps - 1) - dho) <= 1e-10 * abs(dho)


@pytest.mark.parametrize("thermostat", [LANGEVIN, ANDERSEN])
@pytest.mark.parametrize("name,ns", CASES, ids=[c[0] for c in CASES])
def test_tile_edges(name, ns, thermostat):
    sp = SPECS[name]()
    lampath, path = _path(sp)
    pols = _polymers(sp, path, ns)
    b = Batch(Pes(sp), sp.mass, pols, TAU, DT, GAMMA, thermostat=thermostat, noutput=3, seed=SEED)
    b.set_path(lampath, path)
    b.init_path()
    _check(sp, b, pols, range(len(pols)), 8, thermostat, 3, lampath, path)


@pytest.mark.parametrize("name,n,count", [("quartic", 5, 1500), ("quartic", 64, 4097), ("coupled2d", 33, 2050),
                                          ("harmonic3", 32, 1285), ("evb", 32, 1001), ("evb15", 96, 515),
                                          ("water2", 20, 777)])
def test_polymers_sharing_a_workgroup(name, n, count):
    """More polymers than compute units: several per workgroup and, below 9 dofs, several per
    MFMA tile, with a last workgroup that is not full."""
    sp = SPECS[name]()
    lampath, path = _path(sp)
    pols = _polymers(sp, path, [n], count)
    b = Batch(Pes(sp), sp.mass, pols, TAU, DT, GAMMA, seed=SEED)
    b.set_path(lampath, path)
    b.init_path()
    _check(sp, b, pols, [0, 1, 15, 16, 17, count // 2, count - 2, count - 1], 8, LANGEVIN, 1, lampath, path)


@pytest.mark.parametrize("name,ns", [("evb", [2, 33, 159, 160, 161, 192, 193]), ("quartic", [223, 224, 225]),
                                     ("water6", [64, 65])])
@pytest.mark.parametrize("waves", [0, 8])
def test_helper_waves(name, ns, waves):
    """Few polymers take helper waves up to a bead count, unless a wave budget is set; several
    launches of a few steps each hand the stream position over between them."""
    sp = SPECS[name]()
    lampath, path = _path(sp)
    pols = _polymers(sp, path, ns, 2)
    b = Batch(Pes(sp), sp.mass, pols, TAU, DT, GAMMA, seed=SEED)
    b.set_path(lampath, path)
    b.set_launch(3, waves)
    b.init_path()
    _check(sp, b, pols, range(len(pols)), 8, LANGEVIN, 1, lampath, path)
