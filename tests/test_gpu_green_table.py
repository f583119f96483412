"""The table of Green's functions in several passes (more than 256 MiB): the full iteration,
whose calc_chi and self-energy then build it in shapes of their own, against the separate
calls, and the self-energy against the oracle."""
import sys

import numpy as np
import pytest

from oracle import sde as S
from oracle.lattice import Lattice
from tests.helpers import crandn, random_vertices, rel_fro

pytestmark = pytest.mark.gpu
TOL = 1e-12
BETA = 2.0


def _say(*a):
    print(*a, flush=True, file=sys.stderr)


# (4, 16), f_range 8: several passes over the enlarged box, one over the box itself;
# (6, 58), f_range 1: the table over the box itself is the larger one
@pytest.mark.parametrize("nx,nf,f_range", [(4, 16, 8), (6, 58, 1)])
def test_iteration_with_several_passes(nx, nf, f_range):
    from tups_amd import CHI, F, GAMMA, LAMBDA, TupsContext

    _say(f"iteration nx={nx} nf={nf} f_range={f_range} ngrain=64")
    u, mu = 2.0, 0.15
    rng = np.random.default_rng(31)
    lat = Lattice(nx, nf, 1)
    sigma = crandn(rng, (lat.nc * nf,), 0.2).ravel()
    gam = random_vertices(rng, lat.nz, lat.nq, diag=0.5, scale=0.05)
    fv = random_vertices(rng, lat.nz, lat.nq, diag=0.5, scale=0.05)
    lam = [crandn(rng, (nf, nf, lat.nw), 0.1) for _ in range(4)]

    def load(c):
        for r in range(4):
            c.upload(GAMMA, r, gam[r])
            c.upload(F, r, fv[r])
            c.upload(LAMBDA, r, lam[r])
        c.calc_M()

    with TupsContext(nx=nx, nf=nf, nl=1, beta=BETA, f_damping=0.5) as c:
        load(c)
        c.calc_chi(sigma, mu, 64)
        c.BSE(0)
        c.calc_PhiR(0)
        c.calculate_PAE()
        exp_sigma = c.sde(sigma, mu, u, ngrain=64, f_range=f_range)
        c.gamma_update()
        exp = [c.download(w, r) for w in (GAMMA, F) for r in range(4)] + [c.download(CHI, p) for p in range(2)]
    for graph in (False, True):
        with TupsContext(nx=nx, nf=nf, nl=1, beta=BETA, f_damping=0.5) as c:
            load(c)
            c.set_sigma(sigma, mu, 64)
            c.iteration_full(u, graph=graph, f_range=f_range)
            got = [c.download(w, r) for w in (GAMMA, F) for r in range(4)] + [c.download(CHI, p) for p in range(2)]
            assert rel_fro(c.get_sigma(), exp_sigma) < TOL
        for i, (a, b) in enumerate(zip(got, exp)):
            assert rel_fro(a, b) < TOL, (graph, i)


def test_self_energy_with_several_passes(monkeypatch):
    """Nx = 4, Nf = 16, Ngrain = 64, f_range = 8, against the oracle with its auxiliary bubbles
    formed by matrix products."""
    from tups_amd import GAMMA, LAMBDA, TupsContext

    nx, nf, ng, fr, u, mu = 4, 16, 64, 8, 2.0, 0.15
    lat = Lattice(nx, nf, 1)
    rng = np.random.default_rng(32)
    gv = [crandn(rng, (lat.nz, lat.nz, lat.nq), 0.3) for _ in range(4)]
    lam = [crandn(rng, (nf, nf, lat.nw), 1.0) for _ in range(4)]
    sigma = crandn(rng, (lat.nc * nf,), 0.2).ravel()
    sh = sigma.reshape(nx, nx, nf)[:, :, nf - 1].copy()

    def chi_aux(lat, sigma, sigma_h, mu, beta, ngrain=1, f_range=0):
        ext, lo = (2 * f_range + 1) * nf, 1 - f_range * nf
        nu = np.arange(lo, (f_range + 1) * nf + lat.nw)  # nu + w - 1 and Nf - nu + w included
        half = (ng + 1) // 2
        p = 2 * np.pi / nx * (np.arange(nx)[:, None] + (np.arange(1, ng + 1) - half)[None, :] / ng)
        e = -2 * np.cos(p)[:, None, :, None] - 2 * np.cos(p)[None, :, None, :]  # (kx, ky, gx, gy)
        z = 1j * np.pi / beta * (2.0 * (nu - nf // 2 - 1) + 1.0)
        s = np.where(((nu >= 1) & (nu <= nf))[:, None, None],
                     sigma.reshape(nx, nx, nf)[:, :, np.clip(nu, 1, nf) - 1].transpose(2, 0, 1), sigma_h[None])
        g = 1.0 / (z[:, None, None, None, None] - e[None] + mu - s[:, :, :, None, None])
        a = g[:ext].reshape(ext, -1)
        out = np.zeros((2, ext, lat.nq), complex)
        i, o = np.arange(nx), np.arange(ext)
        for q0 in range(0, lat.nq, lat.nw):
            qx, qy = int(lat.qx[q0]) - 1, int(lat.qy[q0]) - 1
            kq = g[:, (i + qx) % nx][:, :, (i + qy) % nx].reshape(len(nu), -1)
            qk = g[:, (qx - i) % nx][:, :, (qy - i) % nx][:, :, :, ::-1, ::-1].reshape(len(nu), -1)
            mph, mpp = a @ kq.T, a @ qk.T
            for q in range(q0, q0 + lat.nw):
                w = int(lat.qw[q])
                out[0, :, q] = mph[o, o + w - 1]
                out[1, :, q] = mpp[o, (nf - (o + lo) + w) - lo]
        return out * lat.ff[0, 0, 0] / ng ** 2

    monkeypatch.setattr(S, "chi_aux", chi_aux)
    exp = S.calc_sde(lat, gv, (lam[0], lam[1]), sigma, sh, mu, BETA, u, ngrain=ng, f_range=fr)
    _say("self-energy nx=4 nf=16 f_range=8 ngrain=64")
    with TupsContext(nx=nx, nf=nf, nl=1, beta=BETA) as c:
        for r in range(4):
            c.upload(GAMMA, r, gv[r])
            c.upload(LAMBDA, r, lam[r])
        got = c.sde(sigma, mu, u, ngrain=ng, f_range=fr)
    assert rel_fro(got, exp) < TOL
