"""The split ladder's preparation of B at the edges of its lane assignment: half a wave per
matrix up to 32 frequencies, the whole wave along them above, more than one pass above 64;
columns beyond D left out of whole and partial workgroups.  Against the oracle, at the split
path's own bound (12 moduli).
"""
import sys

import numpy as np
import pytest

from oracle import bse as B
from oracle.lattice import Lattice
from tests.helpers import random_chi_compact, random_vertices, rel_fro

pytestmark = pytest.mark.gpu
SPLIT_TOL = 1e-10


@pytest.mark.parametrize("nl,nf", [(1, 2), (1, 30), (1, 32), (1, 34), (1, 66), (1, 130),
                                   (5, 2), (5, 26), (5, 32), (5, 34), (5, 66),
                                   (9, 2), (9, 22), (9, 32), (9, 34)])
def test_preparation_edges(nl, nf):
    from tups_amd import BSE_LADDER_SPLIT, CHI, F, GAMMA, TupsContext

    print(f"split preparation nl={nl} nf={nf}", flush=True, file=sys.stderr)
    rng = np.random.default_rng(100 * nl + nf)
    nq = 3
    lat = Lattice(4, nf, nl)
    gam, fv = random_vertices(rng, nl * nf, nq), random_vertices(rng, nl * nf, nq)
    chic = [random_chi_compact(rng, nl, nf, nq, 3.0) for _ in range(2)]
    exp = B.bse_ladder(lat, gam, fv, [B.chi_compact_to_dense(lat, x) for x in chic], 2.0, 0.5)
    with TupsContext(nx=4, nf=nf, nl=nl, nq=nq, beta=2.0, f_damping=0.5) as c:
        c.set_split(12, 2)  # a ragged last pass over a workspace with earlier residues in it
        for p in range(2):
            c.upload(CHI, p, chic[p])
        for _ in range(2):
            for r in range(4):
                c.upload(GAMMA, r, gam[r])
                c.upload(F, r, fv[r])
            c.BSE(0, mode=BSE_LADDER_SPLIT)
            for r in range(4):
                assert rel_fro(c.download(GAMMA, r), exp[r]) < SPLIT_TOL, r
