"""The crossing follows an M that tups_copy has replaced (arrays of one size only: at Nl = 5,
NR = 2, Nf = 10 the bubbles have as many elements as M)."""
import numpy as np
import pytest

from tests.helpers import crandn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_copied_m(graph):
    """Against a context whose M was uploaded: the same values, the same kernels."""
    from tups_amd import CHI, F, GAMMA, LAMBDA, M, TupsContext

    rng = np.random.default_rng(61)
    kw = dict(nx=4, nf=10, nl=5, nr=2, beta=2.0, f_damping=0.5)
    with TupsContext(**kw) as a, TupsContext(**kw) as b:
        assert np.prod(a.shape(M)) == np.prod(a.shape(CHI))
        gam = [crandn(rng, a.shape(GAMMA), 0.1) for _ in range(4)]
        lam = [crandn(rng, a.shape(LAMBDA)) for _ in range(4)]
        new = [crandn(rng, a.shape(M), 0.05) for _ in range(2)]
        for c in (a, b):
            for r in range(4):
                c.upload(GAMMA, r, gam[r])
                c.upload(F, r, gam[r])
                c.upload(LAMBDA, r, lam[r])
            c.calc_M()
            c.iteration(graph=graph)  # with the library's own M
            for p in range(2):
                c.upload(CHI, p, new[p].reshape(c.shape(CHI), order="F"))
        for k in range(2):
            a.copy(M, CHI, k)
            b.upload(M, k, new[k])
        for c in (a, b):
            c.iteration(graph=graph)
        for r in range(4):
            assert np.array_equal(a.download(M, r), b.download(M, r))
            assert np.array_equal(a.download(F, r), b.download(F, r)), r
