"""The work that users of this framework have it do, as cases that a timing program can run.

A case names one of the public paths and its sizes:

  iteration  the loop body of a run (tups_run): the whole iteration on the device as a
             replayed graph, then mu and the convergence check read back
  steps      the crossing step by step, as a driver that owns the loop calls it: calc_PhiR,
             calculate_PAE
  ladder     BSE(ite) in one of its forms over a batch of transfer points: the FP64 ladder,
             the split ladder, the closed form, the refined closed form
  batch      the batching form: every transfer point with its own box, one launch
  finish     what follows the last iteration: calc_Gkw_Grt with cal_chi, the bare
             bubbles, the susceptibilities

Inputs are made from the seed alone.  The vertices stay on the device; what run() returns
of them is the resident arrays themselves, which are read when somebody looks at them.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from tups_amd import (BSE_CLOSED_IR, BSE_CLOSED_LU, BSE_LADDER_FP64, BSE_LADDER_SPLIT, CHI, F, GAMMA, LAMBDA,
                      TupsBatch, TupsContext)

MODES = {"fp64": BSE_LADDER_FP64, "split": BSE_LADDER_SPLIT, "closed": BSE_CLOSED_LU, "refined": BSE_CLOSED_IR}
# c_r of the four channels d, m, s, t, and the bubble (0: ph, 1: pp) that each takes
C_CHANNEL = (0.5, 0.5, -0.25, 0.25)
BUBBLE = (0, 0, 1, 1)
U0 = 2.0
DAMPING = 0.5


def listed():
    return [
        # The reference's own CPU case (4 x 4, 16 frequencies): a few launches of little work,
        # latency counts.
        {"name": "iteration-nx4-nf16-nl1", "kind": "iteration", "nx": 4, "nf": 16, "nl": 1, "beta": 2.0, "filling": 1.0,
         "f_range": 0, "ngrain": 1, "use_u2": True, "mode": "fp64"},
        # The parameter file that the reference ships (16 x 16, 64 frequencies, one form factor).
        {"name": "iteration-nx16-nf64-nl1", "kind": "iteration", "nx": 16, "nf": 64, "nl": 1, "beta": 5.0,
         "filling": 1.0, "f_range": 0, "ngrain": 1, "use_u2": True, "mode": "fp64"},
        # Five form factors on 8 x 8, away from half filling: the production size of the vertex path.
        {"name": "iteration-nx8-nf64-nl5", "kind": "iteration", "nx": 8, "nf": 64, "nl": 5, "beta": 2.0,
         "filling": 0.9, "f_range": 0, "ngrain": 2, "use_u2": True, "mode": "fp64"},
        # Nine form factors on a small box whose orders are multiples of no tile, an enlarged
        # frequency box and the split ladder.
        {"name": "iteration-nx6-nf22-nl9", "kind": "iteration", "nx": 6, "nf": 22, "nl": 9, "beta": 2.0,
         "filling": 0.95, "f_range": 1, "ngrain": 1, "use_u2": False, "mode": "split"},
        # The crossing with nine form factors, where it is the larger half of an iteration.
        {"name": "steps-nx8-nf32-nl9", "kind": "steps", "nx": 8, "nf": 32, "nl": 9, "beta": 2.0},
        # The crossing with one form factor on the shipped box: streams of the vertices.
        {"name": "steps-nx16-nf64-nl1", "kind": "steps", "nx": 16, "nf": 64, "nl": 1, "beta": 2.0},
        # The batched-BSE workload in FP64 and in the split form: 1024 transfer points of order 320.
        {"name": "ladder-fp64-d320", "kind": "ladder", "nx": 8, "nf": 64, "nl": 5, "nq": 1024, "beta": 2.0,
         "mode": "fp64"},
        {"name": "ladder-split-d320", "kind": "ladder", "nx": 8, "nf": 64, "nl": 5, "nq": 1024, "beta": 2.0,
         "mode": "split"},
        # The closed form over the transfer points of the whole 8 x 8 wedge, direct and refined.
        {"name": "ladder-closed-d320", "kind": "ladder", "nx": 8, "nf": 64, "nl": 5, "nq": 480, "beta": 2.0,
         "mode": "closed"},
        {"name": "ladder-refined-d320", "kind": "ladder", "nx": 8, "nf": 64, "nl": 5, "nq": 480, "beta": 2.0,
         "mode": "refined"},
        # Boxes that shrink with the bosonic frequency and 1, 5 or 9 form factors by momentum.
        {"name": "batch-uneven-nx8", "kind": "batch", "nx": 8, "momenta": 32, "nw": 16, "nf": 64, "nf_min": 16,
         "nls": "159", "beta": 2.0},
        # The end of a run on 8 x 8 with five form factors.
        {"name": "finish-nx8-nf64-nl5", "kind": "finish", "nx": 8, "nf": 64, "nl": 5, "beta": 2.0, "ngrain": 4,
         "f_range": 0},
    ]


def _even(rng, lo, hi):
    """An even size, spread evenly over its logarithm."""
    return max(lo, 2 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2))


def draw(rng: random.Random):
    kind = rng.choice(["iteration", "iteration", "steps", "ladder", "ladder", "ladder", "batch", "finish"])
    nl = rng.choice([1, 5, 9])
    beta = round(rng.uniform(1.0, 3.0), 3)
    if kind == "batch":
        hi = _even(rng, 12, 64)
        return {"kind": "batch", "nx": 8, "momenta": rng.randint(3, 24), "nw": rng.randint(3, 16), "nf": hi,
                "nf_min": _even(rng, 4, hi), "nls": rng.choice(["159", "15", "59", "1", "5", "9"]), "beta": beta}
    if kind == "ladder":
        mode = rng.choice(["fp64", "fp64", "split", "closed", "refined"])
        nf = _even(rng, 8, {1: 128, 5: 80, 9: 64}[nl])
        d = nf * nl
        most = (6e10 if mode in ("closed", "refined") else 1.3e11) / (4.0 * d ** 3)
        nq = int(math.exp(rng.uniform(math.log(8), math.log(max(16, min(4096, most, 6e7 / d ** 2))))))
        return {"kind": "ladder", "nx": 8, "nf": nf, "nl": nl, "nq": nq, "beta": beta, "mode": mode}
    nx = 2 * rng.randint(2, {1: 10, 5: 5, 9: 4}[nl])
    wedge = (nx // 2 + 1) * (nx // 2 + 2) // 2
    top = {1: 96, 5: 56, 9: 40}[nl]
    while top > 8 and wedge * top / 2 * (nl * top) ** 2 > 4.5e7:
        top -= 2
    nf = _even(rng, 8, top)
    case = {"kind": kind, "nx": nx, "nf": nf, "nl": nl, "beta": beta}
    if kind == "finish":
        case |= {"nx": min(nx, 16), "ngrain": rng.randint(1, 5), "f_range": rng.choice([0, 0, 1])}
    if kind == "iteration":
        case |= {"filling": round(rng.uniform(0.85, 1.0), 3), "f_range": rng.choice([0, 0, 1]),
                 "ngrain": rng.randint(1, 3), "use_u2": rng.random() < 0.7, "mode": rng.choice(["fp64", "fp64", "split"])}
    return case


# --- inputs ---------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _generator(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(seed)
    return g


def _form_factors(nx, nl):
    """(nl, nx * nx): the site, the four nearest and the four diagonal bonds, of unit mean square."""
    k = 2.0 * math.pi / nx * torch.arange(nx, dtype=torch.float64, device=_device())
    x, y = k[:, None].expand(nx, nx), k[None, :].expand(nx, nx)
    cx, cy, sx, sy = x.cos(), y.cos(), x.sin(), y.sin()
    r2 = math.sqrt(2.0)
    f = [torch.ones_like(cx), cx + cy, cx - cy, r2 * sx, r2 * sy, 2 * cx * cy, -2 * sx * sy,
         r2 * (sx * cy + cx * sy), r2 * (cx * sy - sx * cy)]
    return torch.stack(f[:nl]).reshape(nl, nx * nx)


def _bubbles(nx, nf, nl, beta, momenta, omegas):
    """The bare tight-binding bubbles at half filling, ph and pp: (q, nf, nl, nl) blocks in the
    form factors, scaled per q as in the batched workload so that the ladder contracts."""
    dev = _device()
    k = 2.0 * math.pi / nx * torch.arange(nx, dtype=torch.float64, device=dev)
    eps = -2.0 * (k.cos()[:, None] + k.cos()[None, :])
    f = _form_factors(nx, nl)
    n = torch.arange(1, nf + 1, dtype=torch.float64, device=dev)
    out = torch.empty((2, len(momenta), nf, nl, nl), dtype=torch.complex128, device=dev)

    def g0(e, nu):  # (k, frequencies)
        z = (2.0 * (nu - nf // 2 - 1) + 1.0) * math.pi / beta
        return 1.0 / torch.complex(-e.reshape(-1, 1).expand(-1, nf), z[None, :].expand(e.numel(), -1))

    gk = g0(eps, n)
    i = torch.arange(nx, device=dev)
    for q, ((qx, qy), w) in enumerate(zip(momenta, omegas)):
        kq = eps[(i + qx) % nx][:, (i + qy) % nx]
        qk = eps[(qx - i) % nx][:, (qy - i) % nx]
        for p, b in enumerate((gk * g0(kq, n + w), gk * g0(qk, nf + 1 + w - n))):
            out[p, q] = torch.einsum("kn,ak,bk->nab", b, f.to(b.dtype), f.to(b.dtype))
    alpha = 1.0 / (beta * nx * nx)
    size = out.abs().sum(-1).amax(dim=(2, 3), keepdim=True)[..., None]  # the row sums bound the blocks
    kappa = torch.tensor([alpha, alpha / 2], dtype=torch.float64, device=dev).reshape(2, 1, 1, 1, 1)
    return out * (0.85 / (kappa * 1.6 * U0 * size))


def _vertex(gen, nq, d):
    """U on the diagonal and complex Gaussian noise of variance (0.3 U)^2 / D: (q, column, row)."""
    v = torch.randn((nq, d, d), dtype=torch.complex128, device=_device(), generator=gen) * (0.3 * U0 / math.sqrt(d))
    v.diagonal(dim1=1, dim2=2).add_(U0)
    return v


def _ladder_inputs(case, seed):
    nx, nf, nl, nq = case["nx"], case["nf"], case["nl"], case["nq"]
    gen = _generator(seed)
    r = random.Random(seed)
    momenta = [(r.randrange(nx), r.randrange(nx)) for _ in range(nq)]
    omegas = [q % max(1, nf // 2) for q in range(nq)]
    chi = _bubbles(nx, nf, nl, case["beta"], momenta, omegas)
    # at the first iteration F equals G; the closed forms do not read F
    both = case["mode"] in ("fp64", "split")

    def vertices():
        for _ in range(4):
            g = _vertex(gen, nq, nl * nf)
            yield g, _vertex(gen, nq, nl * nf) if both else g

    return chi, vertices()


def _batch_boxes(case):
    nf, nl = [], []
    for m in range(case["momenta"]):
        for w in range(case["nw"]):
            f = case["nf"] - (case["nf"] - case["nf_min"]) * w / max(1, case["nw"] - 1)
            nf.append(max(2, 2 * round(f / 2)))
            nl.append(int(case["nls"][m % len(case["nls"])]))
    return nf, nl


def _batch_inputs(case, seed):
    """Per q: the four G, the four F as (column, row), and the two bubbles as (nf, nl, nl)."""
    nf, nl = _batch_boxes(case)
    gen = _generator(seed)
    r = random.Random(seed)
    nx = case["nx"]
    chi = []
    for q, (f, l) in enumerate(zip(nf, nl)):
        c = _bubbles(nx, f, l, case["beta"], [(r.randrange(nx), r.randrange(nx))], [q % case["nw"]])
        chi.append(c[:, 0])
    vertex = [[_vertex(gen, 1, f * l)[0] for f, l in zip(nf, nl)] for _ in range(8)]
    return nf, nl, vertex[:4], vertex[4:], chi


def _sigma(case, seed):
    """A self-energy of the shape that the iterations meet: second order in U, local up to a
    few per cent, Sigma(-nu) = conj Sigma(nu)."""
    nx, nf, beta = case["nx"], case["nf"], case["beta"]
    r = random.Random(seed)
    a, b, c = (r.uniform(0.5, 1.0) for _ in range(3))
    k = 2.0 * np.pi / nx * np.arange(nx)
    eps = -2.0 * (np.cos(k)[:, None] + np.cos(k)[None, :])
    nu = (2 * (np.arange(nf) - nf // 2) + 1) * np.pi / beta
    s = U0 ** 2 / 4 * (a + 0.05 * b * eps[:, :, None]) / (1j * nu + 1j * np.sign(nu)) + 0.02 * c * eps[:, :, None]
    return s.reshape(-1)


def _lambda(c):
    for r, v in enumerate((U0, -U0, 2.0 * U0, 0.0)):
        c.upload(LAMBDA, r, np.full((c.nf, c.nf, c.nw), v, dtype=np.complex128, order="F"))


class Resident(list):
    """Arrays that stay on the device, read when they are looked at.  complex128, the
    transfer point first, then column and row."""

    def __init__(self, read):
        super().__init__([read])

    def __iter__(self):
        return list.__getitem__(self, 0)()


def _host(t):
    return t.cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        nf, nl, g, f, chi = _batch_inputs(case, seed)
        b = TupsBatch(case["nx"], nf, nl, beta=case["beta"], f_damping=DAMPING)
        for r in range(4):
            b.upload_packed(GAMMA, r, _host(torch.cat([v.reshape(-1) for v in g[r]])))
            b.upload_packed(F, r, _host(torch.cat([v.reshape(-1) for v in f[r]])))
        for p in range(2):
            b.upload_packed(CHI, p, _host(torch.cat([x[p].reshape(-1) for x in chi])))

        def packed():
            for r in range(4):
                yield np.concatenate([v.ravel(order="F") for v in b.download(GAMMA, r)])

        return {"kind": kind, "b": b, "out": Resident(packed)}
    if kind == "ladder":
        c = TupsContext(nx=case["nx"], nf=case["nf"], nl=case["nl"], nq=case["nq"], beta=case["beta"],
                        f_damping=DAMPING)
        chi, vertices = _ladder_inputs(case, seed)
        for p in range(2):
            c.upload(CHI, p, _host(chi[p]).transpose(3, 2, 1, 0))
        for r, (g, f) in enumerate(vertices):
            c.upload(GAMMA, r, _host(g).T)
            c.upload(F, r, _host(f).T)
        return {"kind": kind, "c": c, "mode": MODES[case["mode"]],
                "out": Resident(lambda: (c.download(GAMMA, r).T for r in range(4)))}
    c = TupsContext(nx=case["nx"], nf=case["nf"], nl=case["nl"], beta=case["beta"], f_damping=DAMPING)
    _lambda(c)
    if kind == "steps":
        for r in range(4):
            c.synth_vertex(GAMMA, r, seed, 0.0, 1.0)
        c.calc_M()
        c.calc_PhiR()
        c.sync()
        return {"kind": kind, "c": c, "out": Resident(lambda: (c.download(F, r).T for r in range(4)))}
    if kind == "finish":
        sigma, vertices = _finish_inputs(case, seed)
        c.set_sigma(sigma, 0.1, ngrain=case["ngrain"])
        for r, (f, phi) in enumerate(vertices):
            c.upload(F, r, _host(f).T)
            c.upload(GAMMA, r, _host(phi).T)
        return {"kind": kind, "c": c, "f_range": case["f_range"]}
    scale = 0.1 / math.sqrt(c.nz)
    for r in range(4):
        c.synth_vertex(GAMMA, r, seed, 0.25, scale)
        c.synth_vertex(F, r, seed, 0.25, scale)
    c.calc_M()
    c.set_sigma(_sigma(case, seed), 0.0, ngrain=case["ngrain"])

    def resident():
        for w in (F, GAMMA):
            for r in range(4):
                yield c.download(w, r).T
        yield c.get_sigma()

    return {"kind": kind, "c": c, "args": {"mode": MODES[case["mode"]], "graph": True, "f_range": case["f_range"],
                                           "use_u2": case["use_u2"], "n_particle": case["filling"]},
            "out": Resident(resident)}


def _finish_inputs(case, seed):
    nq = (case["nx"] // 2 + 1) * (case["nx"] // 2 + 2) // 2 * (case["nf"] // 2)
    gen = _generator(seed)
    d = case["nl"] * case["nf"]

    def vertices():
        for _ in range(4):
            f = _vertex(gen, nq, d)
            yield f, 0.1 * _vertex(gen, nq, d)

    return _sigma(case, seed), vertices()


# --- one pass -------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "batch":
        state["b"].BSE()
        return state["out"]
    c = state["c"]
    if kind == "ladder":
        if state["mode"] in (BSE_CLOSED_LU, BSE_CLOSED_IR):
            for r in range(4):
                c.copy(GAMMA, F, r)  # the solve replaces G by Phi; F keeps this iteration's G
        c.BSE(0, mode=state["mode"])
        return state["out"]
    if kind == "steps":
        c.calc_PhiR()
        c.calculate_PAE()
        return state["out"]
    if kind == "finish":
        mu, _, grt = c.gkw_grt(U0, 1.0, 0.1, cal_chi=True)
        ph, pp, ph_ff, pp_ff = c.chi0()
        return {"mu": mu, "grt": grt, "chi0": [ph, pp, ph_ff, pp_ff], "sus": c.calc_sus(U0, f_range=state["f_range"])}
    c.iteration_full(U0, **state["args"])
    mu, _ = c.get_mu()
    change = c.conv()
    return {"mu": mu, "sigma_avg": change["sigma_avg"], "f_max": change["f_max"], "resident": state["out"]}


# --- what a pass cannot do without ------------------------------------------------------

def _nq(case):
    return (case["nx"] // 2 + 1) * (case["nx"] // 2 + 2) // 2 * (case["nf"] // 2)


def _crossing_macs(case):
    """Complex products of calculate_PAE: for every target entry in a routine's frequency box a
    sum over the two inner form factors and the shells."""
    nf, nl = case["nf"], case["nl"]
    nw, nr = nf // 2, {1: 1, 5: 4, 9: 6}[nl]
    a, b = np.meshgrid(np.arange(1, nf + 1), np.arange(1, nf + 1), indexing="ij")
    hits = 0
    for w in range(1, nw + 1):
        d = b - a
        band = ((d >= 0) & (d + 1 <= nw)) | ((d < 0) & (1 - d <= nw))
        s, t = a + b + w - nf - 1, nf + 3 - w - a - b
        pp = ((s >= 1) & (s <= nw)) | ((t >= 2) & (t <= nw))
        s, t = w - a - b + nf + 1, a + b - w - nf + 1
        ph = ((s >= 1) & (s <= nw)) | ((t >= 2) & (t <= nw))
        hits += int(2 * band.sum() + pp.sum() + ph.sum())
    return 2.0 * hits * _nq(case) / nw * nl ** 4 * nr


def work(case):
    kind = case["kind"]
    if kind == "batch":
        d = [f * l for f, l in zip(*_batch_boxes(case))]
        return {"bytes": 16.0 * 4 * 3 * sum(x * x for x in d), "flops": 16.0 * 4 * sum(float(x) ** 3 for x in d)}
    d = case["nf"] * case["nl"]
    if kind == "ladder":
        # two complex products of the order per matrix; the closed forms: a factorisation and D solves
        per = 16.0 if case["mode"] in ("fp64", "split") else 8.0 / 3.0 + 8.0
        arrays = 3 if case["mode"] in ("fp64", "split") else 2
        return {"bytes": 16.0 * 4 * arrays * d * d * case["nq"], "flops": per * 4 * float(d) ** 3 * case["nq"]}
    vertex = 16.0 * d * d * _nq(case)
    if kind == "finish":
        ext = (2 * case["f_range"] + 1) ** 2
        fine = (case["nx"] * case["ngrain"]) ** 2
        return {"bytes": 4 * vertex * (1 if ext == 1 else 2),
                "flops": 4.0 * 4 * 8 * d * d * ext * _nq(case) + 8.0 * fine * case["nf"] ** 2}
    nr = {1: 1, 5: 4, 9: 6}[case["nl"]]
    phir = 16.0 * d * d * (case["nf"] // 2) * nr
    crossing = 8.0 * _crossing_macs(case)
    if kind == "steps":
        # Phi in, F out, four channels, and the shells
        return {"bytes": 4 * (2 * vertex + phir), "flops": crossing}
    # G and F in, F and G out, the shells between
    return {"bytes": 4 * (4 * vertex + phir), "flops": 16.0 * 4 * float(d) ** 3 * _nq(case) + crossing}


# --- the same in 64 bits, without the framework ------------------------------------------

def _mix(chi, v):
    """chi (nf, nl, nl) blocks times v, for stacks: v as (q, column, row) -> the rows mixed."""
    q, nf, nl, _ = chi.shape
    x = v.reshape(q, v.shape[1], nl, nf)
    return torch.einsum("qnab,qcbn->qcan", chi, x).reshape(v.shape)


def _exact_ladder(g, f, chi, c, alpha):
    """Matrices as (q, column, row), so a product A B is bmm(B, A) here."""
    t = torch.bmm(_mix(chi, f), g) + torch.bmm(_mix(chi, g), f)
    return c * DAMPING * alpha * t + (1.0 - DAMPING) * (f - g)


def _exact_closed(g, chi, kappa):
    """(I - kappa G chi)^-1 G - G by the doubling of the geometric series, which contracts here."""
    nl, nf = chi.shape[2], chi.shape[1]
    eye = torch.eye(nl * nf, dtype=g.dtype, device=g.device).expand_as(g)
    a = kappa * torch.bmm(_mix(chi, eye.contiguous()), g)
    x, p = g.clone(), a
    for _ in range(9):
        x = x + torch.bmm(x, p)
        p = torch.bmm(p, p)
    return x - g


def _exact_finish(case, seed):
    """Grt and the susceptibilities; the bare bubbles' spline quadrature has no 64-bit value of its own."""
    dev = _device()
    nx, nf, nl, beta, ng = case["nx"], case["nf"], case["nl"], case["beta"], case["ngrain"]
    fr, mu = case["f_range"], 0.1
    sigma, vertices = _finish_inputs(case, seed)
    s = torch.from_numpy(sigma).to(dev).reshape(nx, nx, nf)
    half = (ng + 1) // 2
    g = torch.arange(1, ng + 1, dtype=torch.float64, device=dev)
    p = 2 * math.pi / nx * (torch.arange(nx, dtype=torch.float64, device=dev)[:, None] + (g[None, :] - half) / ng)
    eps = -2.0 * (p.cos()[:, None, :, None] + p.cos()[None, :, None, :])  # (kx, ky, gx, gy)

    def green(lo, hi):  # (kx, ky, gx, gy, frequency lo .. hi - 1 of a box that starts at 1)
        n = torch.arange(lo, hi, device=dev)
        z = 1j * math.pi / beta * (2.0 * (n.double() - nf // 2 - 1) + 1.0)
        inside = (n >= 1) & (n <= nf)
        se = torch.where(inside, s[:, :, (n - 1).clamp(0, nf - 1)], s[:, :, nf - 1:nf])
        return 1.0 / (z - eps[..., None] + mu - se[:, :, None, None, :])

    # G(k, tau) on the fine grid and its transform
    n = torch.arange(1, nf + 1, device=dev)
    z = 1j * math.pi / beta * (2.0 * (n.double() - nf // 2 - 1) + 1.0)
    tau = beta / (nf - 1) * torch.arange(nf, dtype=torch.float64, device=dev)
    phase = torch.exp(-z[:, None] * tau[None, :])
    gt = ((green(1, nf + 1) - 1.0 / (z - eps[..., None] + mu)) @ phase).real / beta
    x = (eps - mu)[..., None]
    gt = gt - torch.exp(-tau * x - torch.nn.functional.softplus(-beta * x))
    m = ((torch.arange(nx, device=dev)[:, None] * ng + torch.arange(1, ng + 1, device=dev)[None, :] - half) % (nx * ng))
    fine = torch.empty((nx * ng, nx * ng, nf), dtype=torch.complex128, device=dev)
    fine[m.reshape(-1)[:, None], m.reshape(-1)[None, :]] = gt.permute(0, 2, 1, 3, 4).reshape(nx * ng, nx * ng, nf).to(fine.dtype)
    grt = torch.fft.fft2(fine, dim=(0, 1)) / (nx * ng) ** 2

    k = 2.0 * math.pi / nx * torch.arange(nx, dtype=torch.float64, device=dev)
    px, py = k[:, None].expand(nx, nx), k[None, :].expand(nx, nx)
    ext4 = torch.stack([torch.ones_like(px), px.cos() - py.cos(), px.sin(), px.sin() * py.sin()]).reshape(4, -1)
    ff = _form_factors(nx, nl) / nx
    weight = torch.einsum("fk,lk->flk", ext4, ff).to(torch.complex128)
    ext = (2 * fr + 1) * nf
    lo = -fr * nf + 1
    nw = nf // 2
    gk = green(lo, lo + ext)
    wide = green(lo, lo + ext + nw)
    i = torch.arange(nx, device=dev)
    wedge = [(a, b) for a in range(nx // 2 + 1) for b in range(a + 1)]
    norm = 1.0 / (nx ** 4 * beta ** 2)
    pairs = torch.empty((2, len(wedge) * nw, 4, nl, ext), dtype=torch.complex128, device=dev)
    for mm, (a, b) in enumerate(wedge):
        kq = wide[(i + a) % nx][:, (i + b) % nx]
        qk = wide[(a - i) % nx][:, (b - i) % nx].flip(2, 3)
        for w in range(nw):
            for t, o in enumerate((gk * kq[..., w:w + ext], gk * qk[..., w:w + ext].flip(-1))):
                pairs[t, mm * nw + w] = torch.einsum("flk,kn->fln", weight, o.mean(dim=(2, 3)).reshape(nx * nx, ext))
    q = len(wedge) * nw
    sus = torch.empty((4, 4, q), dtype=torch.complex128, device=dev)
    bare = (U0, -U0, 2 * U0, 0.0)
    pick = (torch.arange(lo, lo + ext, device=dev) - 1).clamp(0, nf - 1)
    box = slice(fr * nf, (fr + 1) * nf)
    for r, (f, phi) in enumerate(vertices):
        o = pairs[BUBBLE[r]]
        f, phi = f.reshape(q, nl, nf, nl, nf), phi.reshape(q, nl, nf, nl, nf)  # (column l, nu, row l, nu)
        inner = torch.einsum("qfan,qanbm,qfbm->fq", o[..., box], f, o[..., box])
        if fr:
            wide_phi = phi[:, :, pick][:, :, :, :, pick].clone()
            wide_phi[:, 0, :, 0, :] += bare[r] * nx * nx
            wide_phi[:, :, box, :, box] = 0.0
            inner = inner + torch.einsum("qfan,qanbm,qfbm->fq", o, wide_phi, o)
        sus[r] = inner * norm
    return {"mu": mu, "grt": grt, "chi0": [None] * 4, "sus": sus}


def exact(case, seed):
    kind = case["kind"]
    alpha = 1.0 / (case["beta"] * case["nx"] ** 2)
    if kind == "ladder":
        chi, vertices = _ladder_inputs(case, seed)
        # chi is kept as (nu, column, row)
        chi = chi.transpose(-1, -2)
        if case["mode"] in ("fp64", "split"):
            return [_exact_ladder(g, f, chi[BUBBLE[r]], C_CHANNEL[r], alpha).cpu()
                    for r, (g, f) in enumerate(vertices)]
        return [_exact_closed(g, chi[BUBBLE[r]], 2 * C_CHANNEL[r] * alpha).cpu() for r, (g, _) in enumerate(vertices)]
    if kind == "batch":
        nf, nl, g, f, chi = _batch_inputs(case, seed)
        out = []
        for r in range(4):
            out.append(torch.cat([_exact_ladder(a[None], b[None], x[BUBBLE[r]][None].transpose(-1, -2), C_CHANNEL[r],
                                                alpha).reshape(-1) for a, b, x in zip(g[r], f[r], chi)]).cpu())
        return out
    if kind == "finish":
        return _exact_finish(case, seed)
    return None  # chains of steps, each of which has its own checks
