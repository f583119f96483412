"""What the refined closed form returns has been checked: the X that it returns meets the
tolerance, the residual that it reports is that X's, and a loose tolerance is met by the first X
that does.  Below D = 128 with the inverse, above it with LU factors.

The residual |Gamma - A X|_F / |Gamma|_F is formed again from the returned Phi in extended
precision.  It differs from the library's own by the rounding of Phi = X - Gamma and of the
library's FP64 sums: 8 eps (1 + |A|_2) |X|_F / |Gamma|_F.
"""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NX, BETA = 4, 2.0
ALPHA = 1.0 / (BETA * NX * NX)  # 1 / 32
KAPPA = [2 * c * ALPHA for c in (0.5, 0.5, -0.25, 0.25)]
EPS = 2.0 ** -52


def _say(*a):
    print(*a, flush=True, file=sys.stderr)


def _solve(a, t, tol):
    """Gamma with I - kappa_r Gamma chi = a for every channel, chi = 1 / (|kappa| t): solved; per
    channel the residual of what is returned and the bar on its rounding; (steps, residual)."""
    from tups_amd import BSE_CLOSED_IR, CHI, F, GAMMA, TupsContext

    d = a.shape[0]
    gam = [np.sign(k) * (np.eye(d) - a) * t[None, :] for k in KAPPA]
    with TupsContext(nx=NX, nf=d, nl=1, nq=1, beta=BETA, f_damping=0.5) as c:
        for r in range(4):
            c.upload(GAMMA, r, gam[r][:, :, None])
            c.upload(F, r, gam[r][:, :, None])
        for p in range(2):
            c.upload(CHI, p, (1.0 / (abs(KAPPA[2 * p]) * t)).astype(complex).reshape(1, 1, d, 1))
        c.set_refinement(tol, 10)
        c.BSE(0, mode=BSE_CLOSED_IR)
        info = c.solve_info()
        phi = [c.download(GAMMA, r)[:, :, 0] for r in range(4)]
    own, bar = [], []
    for r in range(4):
        g, x = gam[r].astype(np.clongdouble), gam[r].astype(np.clongdouble) + phi[r]
        chi = 1.0 / (abs(KAPPA[r]) * t)
        res = g - x + np.longdouble(KAPPA[r]) * ((g * chi[None, :]) @ x)
        n = float(np.linalg.norm(gam[r]))
        own.append(float(np.sqrt((np.abs(res) ** 2).sum())) / n)
        bar.append(8 * EPS * (1 + np.linalg.norm(a, 2)) * float(np.sqrt((np.abs(x) ** 2).sum())) / n)
    return max(own), max(bar), info


def _well_conditioned(d, seed):
    rng = np.random.default_rng(seed)
    return np.eye(d) + 0.2 / np.sqrt(d) * (rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))


@pytest.mark.parametrize("d", [2, 72, 130])
def test_reported_residual_is_that_of_the_result(d):
    _say(f"refined closed form, reported residual, D={d}")
    own, bar, (steps, res) = _solve(_well_conditioned(d, 41), np.full(d, 0.5), 1e-12)
    _say(f"  steps {steps} residual {res:.2e} own {own:.2e} bar {bar:.2e}")
    assert own <= 1e-12
    assert abs(own - res) <= bar


@pytest.mark.parametrize("d", [72, 130])
def test_loose_tolerance_is_met_without_further_steps(d):
    """One FP32 solve leaves about 1e-7."""
    _say(f"refined closed form, loose tolerance, D={d}")
    own, bar, (steps, res) = _solve(_well_conditioned(d, 42), np.full(d, 0.5), 1e-4)
    assert steps == 0 and abs(own - res) <= bar + 1e-3 * res and own <= 1e-4


@pytest.mark.parametrize("d", [72, 130])
def test_step_that_loses_the_tolerance_is_taken_back(d):
    """A of two blocks.  The 2 x 2 block [[1 + e, 1 - e/2], [1 - e/2, 1 + 2^-23 + e]], e just
    below 2^-24, rounds to [[1, 1], [1, 1 + 2^-23]] in FP32, whose determinant is 2.5 times
    smaller: every refinement step makes its residual 1.4 to 1.6 times larger (2.3 s after one
    step and 3.6 s after two; FP32 arithmetic of the block in numpy, in either order of its
    sums).  It enters with the weight s that puts 2.3 s at 0.8e-12 |Gamma|_F: X meets 1e-12
    after one step, when the other block is at a few 1e-13, and would miss it after two."""
    _say(f"refined closed form, step taken back, D={d}")
    e = 0.999 * 2.0 ** -24
    a = np.zeros((d, d), complex)
    a[:2, :2] = [[1 + e, 1 - e / 2], [1 - e / 2, 1 + 2.0 ** -23 + e]]
    a[2:, 2:] = _well_conditioned(d - 2, 43)
    s = 2.0 ** -40
    t = np.full(d, 2.3 * s / (0.8e-12 * np.linalg.norm(np.eye(d - 2) - a[2:, 2:])))
    t[:2] = s
    own, _, (steps, res) = _solve(a, t, 1e-12)
    _say(f"  steps {steps} residual {res:.3e} own {own:.3e}")
    assert own <= 1e-12
    assert steps == 1 and abs(own - res) <= 0.01 * res
