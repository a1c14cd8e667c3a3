"""Ring entry points at the edges of their input: what is not finite."""
import numpy as np
import pytest

from rptunnel import Pes, Ring, RpError, specs

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
