"""The default ladder tile at its edges: tiles cut to one block, two and three blocks of rows
and columns, frequency boxes that are no multiple of a chunk, uniform and uneven, against the
oracle.  Bar: the FP64 path's relative Frobenius error 1e-12 per matrix.
"""
import sys

import numpy as np
import pytest

from oracle import bse as B
from oracle.lattice import Lattice
from tests.helpers import random_chi_compact, random_vertices, rel_fro

pytestmark = pytest.mark.gpu
TOL = 1e-12

# D = 2, 18, 34, 66, 98, 114, 210 / 10, 30, 70, 90, 110, 130 / 18, 54, 90, 126, 198
BOXES = [(1, n) for n in (2, 18, 34, 66, 98, 114, 210)] + [(5, n) for n in (2, 6, 14, 18, 22, 26)] + \
        [(9, n) for n in (2, 6, 10, 14, 22)]


def _case(nl, nf, nq):
    rng = np.random.default_rng(1000 * nl + nf)
    d = nl * nf
    return (random_vertices(rng, d, nq), random_vertices(rng, d, nq),
            [random_chi_compact(rng, nl, nf, nq, 3.0) for _ in range(2)])


def _expect(nx, nl, nf, gam, fv, chi, f):
    lat = Lattice(nx, nf, nl)
    return B.bse_ladder(lat, gam, fv, [B.chi_compact_to_dense(lat, x) for x in chi], 2.0, f)


@pytest.mark.parametrize("nl,nf", BOXES)
def test_cut_tiles(nl, nf):
    from tups_amd import CHI, F, GAMMA, TupsContext

    print(f"ladder tile nl={nl} nf={nf}", flush=True, file=sys.stderr)
    nq = 3
    gam, fv, chi = _case(nl, nf, nq)
    exp = _expect(4, nl, nf, gam, fv, chi, 0.7)
    with TupsContext(nx=4, nf=nf, nl=nl, nq=nq, beta=2.0, f_damping=0.7) as c:
        for r in range(4):
            c.upload(GAMMA, r, gam[r])
            c.upload(F, r, fv[r])
        for p in range(2):
            c.upload(CHI, p, chi[p])
        c.BSE(0)
        for r in range(4):
            got = c.download(GAMMA, r)
            for q in range(nq):
                assert rel_fro(got[..., q], exp[r][..., q]) < TOL, (r, q)


def test_cut_tiles_in_one_uneven_batch():
    from tups_amd import CHI, F, GAMMA, TupsBatch

    cases = [_case(nl, nf, 1) for nl, nf in BOXES]
    exp = [_expect(4, nl, nf, *case, 0.7) for (nl, nf), case in zip(BOXES, cases)]
    with TupsBatch(4, [nf for _, nf in BOXES], [nl for nl, _ in BOXES], beta=2.0, f_damping=0.7) as b:
        for r in range(4):
            b.upload(GAMMA, r, [c[0][r][..., 0] for c in cases])
            b.upload(F, r, [c[1][r][..., 0] for c in cases])
        for p in range(2):
            b.upload(CHI, p, [c[2][p][..., 0] for c in cases])
        b.BSE()
        b.sync()
        for r in range(4):
            got = b.download(GAMMA, r)
            for i, e in enumerate(exp):
                assert rel_fro(got[i], e[r][..., 0]) < TOL, (r, BOXES[i])
