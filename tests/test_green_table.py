"""Shapes of the table of Green's functions (csrc/green_shape.h, compiled for the host): what is
reserved holds every shape that is built in it, and its passes hold every grain once."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "tups_amd" / "csrc"
HARNESS = """
#include "green_shape.h"
using namespace tups;
extern "C" void shape(int nc, int nf, int nw, int ng, int fr, long long budget, long long* o) {
  const GreenShape t = green_shape(nc, nf, nw, ng, fr, (size_t)budget);
  o[0] = t.lo; o[1] = t.len; o[2] = t.ng2; o[3] = t.grains; o[4] = t.split; o[5] = t.plain;
  o[6] = (long long)t.bytes(nc); o[7] = t.passes();
  o[8] = (long long)green_reserve_bytes(nc, nf, nw, ng, fr, (size_t)budget);
}
extern "C" long long default_budget() { return (long long)kGreenTabBytes; }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("green")
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", str(d / "h.cpp"), "-o",
                    str(d / "h.so")], check=True)
    so = C.CDLL(str(d / "h.so"))
    so.default_budget.restype = C.c_longlong
    return so


def _shape(lib, nx, nf, ng, fr, budget):
    o = (C.c_longlong * 9)()
    lib.shape(nx * nx, nf, nf // 2, ng, fr, C.c_longlong(budget), o)
    return dict(zip(("lo", "len", "ng2", "grains", "split", "plain", "bytes", "passes", "reserved"), o))


# the real budget over large boxes, and small ones that force small boxes to several passes
@pytest.mark.parametrize("budget,nxs,nfs", [(0, range(2, 66, 2), range(2, 130, 4)),
                                            (1 << 16, (2, 4, 6, 8), range(2, 42, 2)),
                                            (100000, (2, 4, 6, 8), range(2, 42, 2))])
def test_reserved_table_holds_every_shape(lib, budget, nxs, nfs):
    """f_range: calc_sde, calc_sus and the full iteration; 0: calc_chi within the full iteration,
    which builds its own shape when the enlarged one takes several passes."""
    budget = budget or lib.default_budget()
    bad, split = [], 0
    for nx in nxs:
        for nf in nfs:
            for ng in range(1, 65):
                s0 = _shape(lib, nx, nf, ng, 0, budget)
                for fr in (0, 1, 2, 8):
                    s = _shape(lib, nx, nf, ng, fr, budget)
                    split += s["split"]
                    if max(s["bytes"], s0["bytes"]) > s["reserved"]:
                        bad.append((nx, nf, ng, fr, s0["bytes"], s["reserved"]))
    assert split > 0
    assert not bad, (len(bad), bad[:5])


@pytest.mark.parametrize("nx,nf,ng,fr", [(2, 2, 1, 0), (4, 6, 5, 0), (4, 6, 5, 1), (4, 6, 4, 2), (6, 10, 8, 8)])
def test_passes_hold_every_grain_once(lib, nx, nf, ng, fr):
    """A pass from grain g0 on holds `grains` of them and their mirror images: the pairs (g, Ng^2
    - 1 - g) of all passes are those of one table, and the lattice point has a slot of its own."""
    per = None
    for budget in (1, 1 << 12, 1 << 14, 1 << 16, 1 << 20, 1 << 26):
        s = _shape(lib, nx, nf, ng, fr, budget)
        per = nx * nx * s["len"] * 16
        seen = []
        for p in range(s["passes"]):
            g0 = p * s["grains"]
            seen += [g0 + i for i in range(min(s["grains"], s["ng2"] - g0))]
        assert seen == list(range(s["ng2"]))
        if s["split"]:
            assert s["plain"] == 2 * s["grains"] and s["bytes"] == (2 * s["grains"] + 1) * per
            assert s["grains"] == 1 or 2 * s["grains"] * per <= budget
        else:
            assert s["passes"] == 1 and s["plain"] < s["ng2"] and s["bytes"] == s["ng2"] * per
            assert s["ng2"] == 1 or s["bytes"] <= budget
        # frequencies: the box, k + q and q - k of the enlarged box, k - q of the self-energy
        assert s["lo"] <= min(1 - fr * nf, 2 - nf // 2)
        assert s["lo"] + s["len"] - 1 >= (fr + 1) * nf + nf // 2 - 1
