"""The closed form's LU blocks at their edges, with rows swapped at most columns: orders just
above a multiple of 64, with a last block of 2 to 62 columns, one block only, and register
sub-panels of one and two rows a thread beside the form in memory.

Bar per matrix, relative to X = Gamma + Phi: the backward-stable solve's 8 D eps cond(A) for the
direct mode; for the refined one the residual tolerance 1e-12 times cond(A).
"""
import sys

import numpy as np
import pytest

from oracle import bse as B
from oracle.lattice import Lattice
from tests.helpers import random_chi_compact, random_vertices

pytestmark = pytest.mark.gpu
BETA, NX = 2.0, 4


@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("nl,nf", [(1, 2), (1, 62), (1, 66), (5, 26), (5, 30), (9, 14), (9, 22), (9, 30)])
def test_block_edges(nl, nf, variant):
    from tups_amd import BSE_CLOSED_IR, BSE_CLOSED_LU, CHI, F, GAMMA, TupsContext
    from tups_amd.runtime import K_BSE_CLOSED, K_BSE_IR

    print(f"closed LU nl={nl} nf={nf} variant={variant}", flush=True, file=sys.stderr)
    rng = np.random.default_rng(17 * nl + nf)
    lat = Lattice(NX, nf, nl)
    d, nq = nl * nf, 2
    gam = random_vertices(rng, d, nq, diag=0.0, scale=3.0)
    chic = [random_chi_compact(rng, nl, nf, nq, 3.0) for _ in range(2)]
    dense = [B.chi_compact_to_dense(lat, x) for x in chic]
    exp = B.bse_closed(lat, gam, dense, BETA)
    kappa = [c * 2.0 / (BETA * NX * NX) for c in (0.5, 0.5, -0.25, 0.25)]
    for mode, kernel in ((BSE_CLOSED_LU, K_BSE_CLOSED), (BSE_CLOSED_IR, K_BSE_IR)):
        with TupsContext(nx=NX, nf=nf, nl=nl, nq=nq, beta=BETA, f_damping=0.5) as c:
            c.set_variant(variant, kernel)
            for r in range(4):
                c.upload(GAMMA, r, gam[r])
                c.upload(F, r, gam[r])
            for p in range(2):
                c.upload(CHI, p, chic[p])
            c.BSE(0, mode=mode)
            got = [c.download(GAMMA, r) for r in range(4)]
        for r in range(4):
            for q in range(nq):
                a = np.eye(d) - kappa[r] * gam[r][..., q] @ dense[r // 2][..., q]
                x = gam[r][..., q] + exp[r][..., q]
                bar = np.linalg.cond(a) * (8 * d * 2.0 ** -53 if mode == BSE_CLOSED_LU else 1e-12)
                err = np.linalg.norm(got[r][..., q] - exp[r][..., q]) / np.linalg.norm(x)
                assert err < max(bar, 1e-14), (mode, r, q, err, bar)
