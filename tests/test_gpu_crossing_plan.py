"""The crossing over the nonzero elements of M (Nl > 1): row packing, staging chunks and
column tiles at the sizes where they have remainders, and M arrays of other patterns than
the library's own (uploaded ones), against the oracle at 1e-12 relative Frobenius error."""
import sys

import numpy as np
import pytest

from oracle import parquet as P
from oracle.lattice import Lattice
from tests.helpers import crandn, rel_fro

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _say(*a):
    print(*a, flush=True, file=sys.stderr)


def _inputs(lat, seed):
    rng = np.random.default_rng(seed)
    phi = [crandn(rng, (lat.nz, lat.nz, lat.nq)) for _ in range(4)]
    phir = [crandn(rng, (lat.nz ** 2, lat.nw, lat.nr)) for _ in range(4)]
    lam = [crandn(rng, (lat.nf, lat.nf, lat.nw)) for _ in range(4)]
    return phi, phir, lam


def _load(c, phi, phir, lam):
    from tups_amd import GAMMA, LAMBDA, PHIR

    for r in range(4):
        c.upload(GAMMA, r, phi[r])
        c.upload(PHIR, r, phir[r])
        c.upload(LAMBDA, r, lam[r])


def _check(c, lat, phi, phir, lam, mt, qs):
    from tups_amd import F

    exp = P.calculate_pae(lat, phi, lam, phir, mt, qs=qs)
    c.calculate_PAE()
    for r in range(4):
        got = c.download(F, r)[:, :, qs]
        err = rel_fro(got, exp[r][:, :, qs])
        _say(f"  channel {r}: {err:.2e}")
        assert err < TOL


# NIBZ = 3, 6, 10, 15, 21: rows of a class below, at and beyond one block of 16;
# Nf^2 = 4 .. 484: less than a column tile, whole tiles, remainders of 4
@pytest.mark.parametrize("nx,nf,nl", [(4, 2, 5), (4, 10, 9), (6, 6, 5), (6, 10, 9), (8, 4, 9), (10, 6, 5), (6, 22, 5)])
def test_plan_parity(nx, nf, nl):
    from tups_amd import TupsContext

    lat = Lattice(nx, nf, nl)
    _say(f"crossing plan nx={nx} nf={nf} nl={nl} nibz={lat.nibz}")
    phi, phir, lam = _inputs(lat, 5)
    qs = sorted({0, lat.nq - 1, lat.nq // 2, lat.nw - 1})
    with TupsContext(nx=nx, nf=nf, nl=nl) as c:
        _load(c, phi, phir, lam)
        c.calc_M()
        _check(c, lat, phi, phir, lam, P.calc_m_tensors(lat), qs)


def test_zero_elements_are_exact_and_the_others_kept():
    """calc_M writes exact zeros where the oracle has rounding noise, and only there."""
    from tups_amd import M, TupsContext
    from tups_amd.runtime import M_NAMES

    lat = Lattice(6, 4, 9)
    mt = P.calc_m_tensors(lat)
    with TupsContext(nx=6, nf=4, nl=9) as c:
        c.calc_M()
        for k, name in enumerate(M_NAMES):
            got, exp = c.download(M, k), mt[name]
            assert np.abs(exp[got == 0]).max() < 1e-13  # rounding of sums of 36 terms of order one
            assert np.abs(exp[got != 0]).min() > 1e-4
            assert np.abs(got - exp).max() < 1e-12


@pytest.mark.parametrize("fill", [0.0, 0.04, 0.3, 1.0])
def test_uploaded_m_of_any_pattern(fill):
    """M from the host: empty, sparse without structure, half full (more inner indices per
    group than one staging chunk holds), dense (the dense form); then the library's own again."""
    from tups_amd import M, TupsContext
    from tups_amd.runtime import M_NAMES

    nx, nf, nl = 4, 6, 9
    lat = Lattice(nx, nf, nl)
    _say(f"crossing with uploaded M, fill {fill}")
    phi, phir, lam = _inputs(lat, 6)
    rng = np.random.default_rng(7)
    mt = {}
    for name in M_NAMES:
        m = crandn(rng, (nl, nl, nl, nl, lat.nibz, lat.nr), 0.1)
        mt[name] = m * (rng.random(m.shape[:4] + (1, lat.nr)) < fill)
    qs = [0, lat.nq - 1]
    with TupsContext(nx=nx, nf=nf, nl=nl) as c:
        _load(c, phi, phir, lam)
        c.calc_M()
        c.calculate_PAE()
        for k, name in enumerate(M_NAMES):
            c.upload(M, k, mt[name])
        _check(c, lat, phi, phir, lam, mt, qs)
        c.calc_M()
        _check(c, lat, phi, phir, lam, P.calc_m_tensors(lat), qs)


def test_graph_follows_a_new_m():
    """A captured iteration runs with the M uploaded after its capture."""
    from tups_amd import CHI, F, GAMMA, LAMBDA, M, TupsContext

    nx, nf, nl = 4, 6, 5
    lat = Lattice(nx, nf, nl)
    rng = np.random.default_rng(8)
    g, f = ([crandn(rng, (lat.nz, lat.nz, lat.nq), 0.1) for _ in range(4)] for _ in range(2))
    chi = [crandn(rng, (nl, nl, nf, lat.nq)) for _ in range(2)]
    lam = [crandn(rng, (nf, nf, lat.nw)) for _ in range(4)]
    new = [crandn(rng, (nl, nl, nl, nl, lat.nibz, lat.nr), 0.05) for _ in range(4)]
    with TupsContext(nx=nx, nf=nf, nl=nl) as a, TupsContext(nx=nx, nf=nf, nl=nl) as b:
        for c in (a, b):
            for r in range(4):
                c.upload(GAMMA, r, g[r])
                c.upload(F, r, f[r])
                c.upload(LAMBDA, r, lam[r])
            for p in range(2):
                c.upload(CHI, p, chi[p])
            c.calc_M()
        for it in range(6):
            if it == 3:
                for c in (a, b):
                    for k in range(4):
                        c.upload(M, k, new[k])
            a.iteration(graph=True)
            b.iteration(graph=False)
            for r in range(4):
                assert np.array_equal(a.download(F, r), b.download(F, r)), (it, r)
                assert np.array_equal(a.download(GAMMA, r), b.download(GAMMA, r)), (it, r)
