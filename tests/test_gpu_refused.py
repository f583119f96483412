"""Calls that are refused leave the context as it was."""
import numpy as np
import pytest

from tests.helpers import crandn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{"f_range": 9}, {"f_range": -1}, {"ngrain": 65}, {"ngrain": 0}])
def test_refused_sde_keeps_sigma(kw):
    """A later device iteration works with the Sigma, mu and Ngrain of set_sigma."""
    from tups_amd import TupsContext, TupsError

    rng = np.random.default_rng(51)
    with TupsContext(nx=4, nf=8, nl=1, beta=2.0) as c:
        sigma, other = (crandn(rng, (16 * 8,), 0.2).ravel() for _ in range(2))
        c.set_sigma(sigma, 0.25)
        with pytest.raises(TupsError):
            c.sde(other, 0.5, 2.0, **kw)
        assert np.array_equal(c.get_sigma(), sigma)
        assert c.get_mu()[0] == 0.25
