"""Member counts on a particle set that has no cells or units yet (needs an
MI355X): the gradient's are refused, as the units of the set before hold other
particles; the density's find no neighbours in cells that hold none."""
import numpy as np
import pytest

from vps import Projection, VpsError, _abi, scenes

pytestmark = pytest.mark.gpu


def test_counts_before_and_between_sets():
    sc = scenes.small_3d(12, 8, 6)
    g = Projection(sc)
    assert np.all(g.member_counts(0) == 0)
    with pytest.raises(VpsError) as e:
        g.member_counts(2)
    assert e.value.code == _abi.VPS_ERR_STATE
    g.initialize()
    assert np.all(g.member_counts(2) > 0)
    g.set_particles(sc["x"][:10], sc["v"][:10])   # 10 of 576: the counts' array holds 10
    with pytest.raises(VpsError) as e:
        g.member_counts(2)
    assert e.value.code == _abi.VPS_ERR_STATE
    g.initialize()
    assert np.all(g.member_counts(2) > 0)
    g.close()
