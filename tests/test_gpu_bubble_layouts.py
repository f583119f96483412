"""calc_chi in every layout of the weights and of the lanes that its launch chooses among: narrow
and wide groups, 64 and 16 lanes a workgroup; against numpy at 1e-12."""
import sys

import numpy as np
import pytest

from oracle.lattice import Lattice
from tests.helpers import crandn, rel_fro
from tests.test_gpu_bubble import BETA, TOL, _chi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nf,nl,ngrain", [(4, 10, 9, 3),   # narrow groups, 16 lanes
                                             (4, 10, 5, 2), (4, 2, 5, 4),
                                             (4, 6, 9, 16),   # wide groups, 16 lanes
                                             (6, 14, 9, 6), (8, 24, 9, 8), (8, 18, 1, 5),
                                             (8, 34, 9, 1),   # narrow groups, 64 lanes
                                             (8, 34, 9, 2)])  # wide groups, 64 lanes
def test_chi_layouts(nx, nf, nl, ngrain):
    from tups_amd import CHI, TupsContext

    print(f"chi nx={nx} nf={nf} nl={nl} ngrain={ngrain}", flush=True, file=sys.stderr)
    lat = Lattice(nx, nf, nl)
    rng = np.random.default_rng(81)
    sigma = crandn(rng, (lat.nc * nf,), 0.2).ravel()
    sh = crandn(rng, (nx, nx), 0.1)
    with TupsContext(nx=nx, nf=nf, nl=nl, beta=BETA) as c:
        qx, qy, qw = c.q_map()
        c.calc_chi(sigma, 0.15, ngrain, sh)
        got = [c.download(CHI, p) for p in range(2)]
    for q in sorted({0, len(qx) // 2, len(qx) - 1}):
        exp = _chi(lat, sigma, sh, 0.15, ngrain, (int(qx[q]), int(qy[q]), int(qw[q])))
        for p in range(2):
            assert rel_fro(got[p][:, :, :, q], exp[p]) < TOL, (q, p)
