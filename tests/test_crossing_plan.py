"""The plan of the crossing over the nonzero elements of M (csrc/crossing_plan.cpp, compiled for
the host): every product that M asks for is done once, from a staged row, by the row's block."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "tups_amd" / "csrc"
HARNESS = """
#include "crossing_plan.h"
#include <cstring>
using namespace tups;
static PaePlanHost p;
extern "C" void plan(const uint8_t* sup, const int* rows, int nrows, int nl, int nibz, int kk, long long* o) {
  build_pae_plan(std::vector<uint8_t>(sup, sup + 4LL * nl * nl * kk), std::vector<int>(rows, rows + nrows), nl, nibz, kk, p);
  o[0] = p.groups[0]; o[1] = p.groups[1]; o[2] = p.chunks; o[3] = p.chunk_len; o[4] = p.steps;
}
extern "C" long long get(int which, int* out) {
  const std::vector<int>* v[] = {&p.ubeg, &p.ulist, &p.seg, &p.kidx, &p.kj, &p.step_blk, &p.brow, &p.used, &p.used_by};
  if (out) std::memcpy(out, v[which]->data(), v[which]->size() * sizeof(int));
  return (long long)v[which]->size();
}
extern "C" int constant(int i) { const int c[] = {kPlanRows, kPlanSlots, kPlanBlocks, kPlanChunk}; return c[i]; }
"""
NAMES = ("ubeg", "ulist", "seg", "kidx", "kj", "step_blk", "brow", "used", "used_by")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", str(d / "h.cpp"),
                    str(CSRC / "crossing_plan.cpp"), "-o", str(d / "h.so")], check=True)
    so = C.CDLL(str(d / "h.so"))
    so.get.restype = C.c_longlong
    return so


def _plan(lib, sup, rows, nl, nibz, kk):
    sup = np.ascontiguousarray(sup, dtype=np.uint8)
    rows = np.ascontiguousarray(rows, dtype=np.int32)
    o = (C.c_longlong * 5)()
    lib.plan(sup.ctypes.data_as(C.c_void_p), rows.ctypes.data_as(C.c_void_p), len(rows), nl, nibz, kk, o)
    out = dict(zip(("g0", "g1", "chunks", "chunk_len", "steps"), o))
    for i, n in enumerate(NAMES):
        v = np.zeros(lib.get(i, None), dtype=np.int32)
        lib.get(i, v.ctypes.data_as(C.c_void_p))
        out[n] = v
    return out


# fill 0.1 at Nl = 9: several staging chunks, still less than half of the dense form's steps
@pytest.mark.parametrize("fill", [0.0, 0.04, 0.1, 0.15, 0.3, 1.0])
@pytest.mark.parametrize("nl,nibz,nr,subset", [(5, 3, 4, False), (5, 15, 4, True), (9, 6, 6, False), (9, 10, 6, True)])
def test_products_done_once(lib, nl, nibz, nr, subset, fill):
    rng = np.random.default_rng(int(100 * fill) + nl + nibz)
    rmax, slots, blocks, chunk = (lib.constant(i) for i in range(4))
    nl2, kk = nl * nl, nl * nl * nr
    sup = (rng.random((4, nl2, kk)) < fill).astype(np.uint8)
    rows = np.flatnonzero(rng.random(nl2 * nibz) < 0.4) if subset else np.zeros(0, int)
    p = _plan(lib, sup, rows, nl, nibz, kk)
    wanted = list(rows) if subset else list(range(nl2 * nibz))
    ng, nc = p["g0"] + p["g1"], p["chunks"]
    brow = p["brow"].reshape(ng, blocks, rmax)
    ubeg = p["ubeg"].reshape(ng, 2, nc + 1)
    seg = p["seg"].reshape(ng, 2, nc, blocks, 2)
    kj, step_blk = p["kj"].reshape(-1, 4), p["step_blk"]
    by = dict(zip(p["used"], p["used_by"]))
    assert p["chunk_len"] <= chunk < 256 and len(step_blk) == p["steps"] == len(p["kidx"])
    assert (seg[..., 1] - seg[..., 0]).max(initial=0) <= 64  # one lane holds a k-step's rows
    done = np.zeros(p["steps"], int)
    for pair in range(2):
        groups = range(p["g0"]) if pair == 0 else range(p["g0"], ng)
        got = sorted(r for g in groups for r in brow[g].ravel() if r >= 0)
        assert got == sorted(wanted)  # every row in one block
        for g in groups:
            for rt in range(2):
                cover = [dict() for _ in range(blocks)]
                for c in range(nc):
                    u = p["ulist"][ubeg[g, rt, c]:ubeg[g, rt, c + 1]]
                    assert len(u) <= p["chunk_len"] and len(set(u)) == len(u)
                    if c + 1 < nc and len(u) == 0:  # the kernel stops at the first empty chunk
                        assert ubeg[g, rt, nc] == ubeg[g, rt, c]
                    assert all(by[j] >> (2 * pair + rt) & 1 for j in u)
                    for b in range(blocks):
                        for s in range(*seg[g, rt, c, b]):
                            done[s] += 1
                            assert step_blk[s] == (g * blocks + b) * 2 + rt
                            for k in range(4):
                                at = p["kidx"][s] >> (8 * k) & 255
                                assert at < len(u)
                                if kj[s, k] >= 0:
                                    assert u[at] == kj[s, k]
                                    cover[b][kj[s, k]] = cover[b].get(kj[s, k], 0) + 1
                for b in range(blocks):
                    r = brow[g, b]
                    need = set()
                    for x in r[r >= 0]:
                        need |= set(np.flatnonzero(sup[2 * pair + rt, x % nl2]))
                    assert set(cover[b]) == need and all(n == 1 for n in cover[b].values())
    assert (done == 1).all()


def test_chunks_of_the_plan_form(lib):
    """Nl = 9, NIBZ = 6, NR = 6: a random M is planned up to a fill between 0.2 and 0.3 (less than
    half of the dense form's k-steps), with several staging chunks from 0.04 on."""
    nl2, kk = 81, 486
    dense = 2 * ((nl2 * 6 + 15) // 16) * 2 * ((kk + 3) // 4)
    chunks = {}
    for fill in (0.04, 0.1, 0.15, 0.3):
        sup = np.random.default_rng(7).random((4, nl2, kk)) < fill
        p = _plan(lib, sup, [], 9, 6, kk)
        chunks[fill] = p["chunks"] if 2 * p["steps"] <= dense else 0
    assert chunks[0.04] >= 2 and chunks[0.1] > chunks[0.04] and chunks[0.15] > 0 and chunks[0.3] == 0, chunks
