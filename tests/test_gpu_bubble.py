"""The bubbles from the table of Green's functions where their launch changes: weight groups
(Nl = 9), slots that are not the wedge in order, a coarse graining whose table takes several
passes, and the self-energy in chunks of q slots; against numpy or the oracle at 1e-12."""
import sys

import numpy as np
import pytest

from oracle import sde as S
from oracle.lattice import Lattice
from tests.helpers import crandn, rel_fro

pytestmark = pytest.mark.gpu
TOL = 1e-12
BETA = 2.0


def _say(*a):
    print(*a, flush=True, file=sys.stderr)


def _green(lat, sigma, sigma_h, mu, ng, lo, n):
    """G(kx, ky, gx, gy, nu) for nu = lo .. lo + n - 1 (get_green_coarse on whole arrays)."""
    nx, nf = lat.nx, lat.nf
    half = (ng + 1) // 2
    p = 2 * np.pi / nx * (np.arange(nx)[:, None] + (np.arange(1, ng + 1) - half)[None, :] / ng)
    e = -2 * np.cos(p)[:, None, :, None] - 2 * np.cos(p)[None, :, None, :]
    nu = np.arange(lo, lo + n)
    s = np.empty((nx, nx, n), complex)
    inside = (nu >= 1) & (nu <= nf)
    s[:, :, inside] = sigma.reshape(nx, nx, nf)[:, :, nu[inside] - 1]
    s[:, :, ~inside] = sigma_h[:, :, None]
    z = 1j * np.pi / BETA * (2.0 * (nu - nf // 2 - 1) + 1.0)
    return 1.0 / (z - e[..., None] + mu - s[:, :, None, None, :])


def _chi(lat, sigma, sigma_h, mu, ng, q):
    """calc_chi of one 1-based (qx, qy, w): (Nl, Nl, Nf) ph and pp."""
    nf = lat.nf
    qx, qy, w = q
    i = np.arange(lat.nx)
    gk = _green(lat, sigma, sigma_h, mu, ng, 1, nf)
    gp = _green(lat, sigma, sigma_h, mu, ng, w, nf)
    kq = np.ix_((i + qx - 1) % lat.nx, (i + qy - 1) % lat.nx)
    qk = np.ix_((qx - 1 - i) % lat.nx, (qy - 1 - i) % lat.nx)
    ph = (gk * gp[kq]).mean(axis=(2, 3))
    pp = (gk * gp[qk][:, :, ::-1, ::-1, ::-1]).mean(axis=(2, 3))
    return [np.einsum("xyn,xya,xyb->abn", x, lat.ff, lat.ff) for x in (ph, pp)]


# Ngrain = 64 at Nx = 8: 4096 grains of 66 KB, beyond the 256 MiB that one pass holds
@pytest.mark.parametrize("nx,nf,nl,ngrain,nq", [(4, 10, 9, 2, 0), (6, 6, 5, 1, 7), (4, 34, 1, 3, 500), (8, 34, 1, 64, 0)])
def test_chi_table(nx, nf, nl, ngrain, nq):
    from tups_amd import CHI, TupsContext

    _say(f"chi from the table nx={nx} nf={nf} nl={nl} ngrain={ngrain} nq={nq}")
    lat = Lattice(nx, nf, nl)
    rng = np.random.default_rng(3)
    sigma = crandn(rng, (lat.nc * nf,), 0.2).ravel()
    sh = crandn(rng, (nx, nx), 0.1)
    with TupsContext(nx=nx, nf=nf, nl=nl, nq=nq, beta=BETA) as c:
        if nq:  # slots in no order, some of them twice
            p = [(x, y) for x in range(1, nx // 2 + 2) for y in range(1, x + 1)]
            pick = rng.integers(0, len(p), nq)
            c.set_q_map([p[i][0] for i in pick], [p[i][1] for i in pick], rng.integers(1, nf // 2 + 1, nq))
        qx, qy, qw = c.q_map()
        c.calc_chi(sigma, 0.15, ngrain, sh)
        got = [c.download(CHI, p) for p in range(2)]
    n = len(qx)
    for q in sorted({0, 1, n // 2, n - 1}) if ngrain < 64 else [0, n - 1]:
        exp = _chi(lat, sigma, sh, 0.15, ngrain, (int(qx[q]), int(qy[q]), int(qw[q])))
        for p in range(2):
            err = rel_fro(got[p][:, :, :, q], exp[p])
            assert err < TOL, (q, p, err)


# 135 q slots: two chunks; f_range 2: the folded edges; Nz = 18, 40: 32 and 64 lanes of L3
@pytest.mark.parametrize("nx,nf,nl,f_range,use_u2", [(8, 18, 1, 0, False), (4, 8, 5, 2, False), (4, 18, 1, 1, True)])
def test_sde_launches(nx, nf, nl, f_range, use_u2):
    from oracle import gtau as T
    from tups_amd import GAMMA, LAMBDA, TupsContext

    _say(f"sde nx={nx} nf={nf} nl={nl} f_range={f_range} use_u2={use_u2}")
    rng = np.random.default_rng(4)
    lat = Lattice(nx, nf, nl)
    u, mu = 2.0, 0.15
    gv = [crandn(rng, (lat.nz, lat.nz, lat.nq), 0.3) for _ in range(4)]
    lam = [crandn(rng, (nf, nf, lat.nw), 1.0) for _ in range(4)]
    sigma = crandn(rng, (lat.nc * nf,), 0.2).ravel()
    sh = sigma.reshape(nx, nx, nf)[:, :, nf - 1].copy()
    with TupsContext(nx=nx, nf=nf, nl=nl, beta=BETA) as c:
        for r in range(4):
            c.upload(GAMMA, r, gv[r])
            c.upload(LAMBDA, r, lam[r])
        second = 0.0
        if use_u2:
            c.set_sigma(sigma, mu)
            m, _, _ = c.gkw_grt(u, 1.0, mu, cal_chi=True)
            second = T.order_2nd(lat, T.grt(lat, sigma, m, BETA, 1), u, BETA, 1)
        got = c.sde(sigma, mu, u, f_range=f_range, use_u2=use_u2)
    exp = S.calc_sde(lat, gv, (lam[0], lam[1]), sigma, sh, mu, BETA, u, f_range=f_range, use_u2=use_u2) + second
    assert rel_fro(got, exp) < TOL
