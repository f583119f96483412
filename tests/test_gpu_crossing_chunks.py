"""The crossing's plan kernel with four staging chunks and more: M from the host that is a tenth
or a seventh full, the densest that the plan takes (a third runs the dense form), against the
oracle at 1e-12 relative Frobenius error."""
import sys

import numpy as np
import pytest

from oracle.lattice import Lattice
from tests.helpers import crandn
from tests.test_gpu_crossing_plan import _check, _inputs, _load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nf,nl", [(4, 6, 9), (6, 10, 5)])
@pytest.mark.parametrize("fill", [0.1, 0.15])
def test_many_chunks(nx, nf, nl, fill):
    from tups_amd import M, TupsContext
    from tups_amd.runtime import M_NAMES

    print(f"crossing plan, M filled to {fill}, nx={nx} nf={nf} nl={nl}", flush=True, file=sys.stderr)
    lat = Lattice(nx, nf, nl)
    phi, phir, lam = _inputs(lat, 9)
    rng = np.random.default_rng(7)
    mt = {}
    for name in M_NAMES:
        m = crandn(rng, (nl, nl, nl, nl, lat.nibz, lat.nr), 0.1)
        mt[name] = m * (rng.random(m.shape[:4] + (1, lat.nr)) < fill)
    with TupsContext(nx=nx, nf=nf, nl=nl) as c:
        _load(c, phi, phir, lam)
        for k, name in enumerate(M_NAMES):
            c.upload(M, k, mt[name])
        _check(c, lat, phi, phir, lam, mt, [0, lat.nq - 1])
