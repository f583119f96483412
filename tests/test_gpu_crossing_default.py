"""The crossing at Nl = 1 in the form that is chosen without autotuning, at the boxes where the
choice changes and where tiles and groups of momenta have remainders (1 to 45 IBZ momenta),
against the oracle at 1e-12 relative Frobenius error."""
import sys

import numpy as np
import pytest

from oracle import parquet as P
from oracle.lattice import Lattice
from tests.helpers import crandn, rel_fro

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("nx,nf", [(2, 2), (2, 16), (4, 6), (6, 16), (8, 14), (16, 16), (4, 18), (6, 34), (4, 56),
                                   (4, 58), (6, 64), (4, 66)])
def test_default_form(nx, nf):
    from tups_amd import F, GAMMA, LAMBDA, PHIR, TupsContext

    print(f"crossing default nx={nx} nf={nf}", flush=True, file=sys.stderr)
    lat = Lattice(nx, nf, 1)
    rng = np.random.default_rng(71)
    phi = [crandn(rng, (nf, nf, lat.nq)) for _ in range(4)]
    phir = [crandn(rng, (nf * nf, lat.nw, lat.nr)) for _ in range(4)]
    lam = [crandn(rng, (nf, nf, lat.nw)) for _ in range(4)]
    qs = sorted({0, lat.nw - 1, lat.nq // 2, lat.nq - 1})
    with TupsContext(nx=nx, nf=nf, nl=1) as c:
        for r in range(4):
            c.upload(GAMMA, r, phi[r])
            c.upload(PHIR, r, phir[r])
            c.upload(LAMBDA, r, lam[r])
        c.calc_M()
        c.calculate_PAE()
        got = [c.download(F, r)[:, :, qs] for r in range(4)]
    exp = P.calculate_pae(lat, phi, lam, phir, P.calc_m_tensors(lat), qs=qs)
    for r in range(4):
        assert rel_fro(got[r], exp[r][:, :, qs]) < TOL, r
