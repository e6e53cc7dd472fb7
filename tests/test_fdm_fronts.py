"""The host plan of the default field solve (csrc/fdm_front.cpp), executed in
numpy: dense operators per front formed from L and U as the device forms them,
the solve up and down the tree of fronts through the plan's own tables
(positions, boundaries, contribution rows, assembly lists, tasks), against
scipy's triangular solves of the same factors.

Systems: SuperLU factors of FDM plans (the pattern a blob holds), factors
whose L and U^T differ in pattern (off-diagonal pivots, so the union has to be
closed under fill), systems smaller than one leaf, a forest of disconnected
parts, a chain (no branching), a dense system wider than the widest front and
a star whose hub takes more than four contributions.
"""
from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

sp = pytest.importorskip("scipy.sparse")
import scipy.sparse.linalg as spla  # noqa: E402

CSRC = Path(__file__).resolve().parents[1] / "neurips2026_smart_building_challenge_amd" / "csrc"
DRIVER = r"""
#include "fdm_front.h"
#include <string.h>
static sbf::FrontPlan P;
extern "C" void plan(int n, const int* lp, const int* li, const int* up, const int* ui) {
    sbf::RowTerms l(n), u(n);
    for (int i = 0; i < n; i++) {
        for (int e = lp[i]; e < lp[i + 1]; e++) l[i].push_back({li[e], 1.0});
        for (int e = up[i]; e < up[i + 1]; e++) u[i].push_back({ui[e], 1.0});
    }
    sbf::plan_fronts(l, u, &P);
}
#define GET(name, v) extern "C" long name(void* out) { \
    long b = (long)((v).size() * sizeof((v)[0])); if (out) { memcpy(out, (v).data(), b); } return b; }
GET(fronts, P.fronts) GET(pos, P.pos) GET(front_of, P.front_of) GET(local_of, P.local) GET(bperm, P.bperm)
GET(brow, P.brow) GET(arow, P.arow) GET(xsrc, P.xsrc) GET(tasks, P.tasks) GET(levels, P.levels)
extern "C" void scalars(long* o) { o[0] = P.n_leaf; o[1] = P.n_c; o[2] = (long)P.ops; }
"""
FRONT = np.dtype([(k, np.int32) for k in ("off", "w", "r", "brow", "c", "arow")] + [("f", np.int64), ("k", np.int64)])
AROW = np.dtype([("s", np.int32, 4), ("xb", np.int32), ("xe", np.int32), ("pad", np.int32, 2)])
TASK = np.dtype([("front", np.int32), ("tile", np.int32)])
LEVEL = np.dtype([(k, np.int32) for k in ("f0", "nf", "k0", "nk", "wmax")])


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    d = tmp_path_factory.mktemp("fronts")
    (d / "driver.cpp").write_text(DRIVER)
    so = d / "fronts.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-I", str(CSRC),
                    str(CSRC / "fdm_front.cpp"), str(d / "driver.cpp"), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def plan_of(lib, L, U):
    ip = lambda a: np.ascontiguousarray(a, np.int32)
    lo, up = sp.tril(L, -1).tocsr(), sp.triu(U, 1).tocsr()
    lo.sort_indices()
    up.sort_indices()
    args = [ip(lo.indptr), ip(lo.indices), ip(up.indptr), ip(up.indices)]
    lib.plan(L.shape[0], *(a.ctypes.data_as(ctypes.c_void_p) for a in args))
    out = {}
    for name, dt in (("fronts", FRONT), ("pos", np.int32), ("front_of", np.int32), ("local_of", np.int32),
                     ("bperm", np.int32), ("brow", np.int32), ("arow", AROW), ("xsrc", np.int32), ("tasks", TASK),
                     ("levels", LEVEL)):
        f = getattr(lib, name)
        f.restype = ctypes.c_long
        buf = np.zeros(f(None), np.uint8)
        f(buf.ctypes.data_as(ctypes.c_void_p))
        out[name] = buf.view(dt)
    sc = (ctypes.c_long * 3)()
    lib.scalars(sc)
    out["n_leaf"], out["n_c"], out["ops"] = sc[0], sc[1], sc[2]
    return out


def execute(P, L, U, b):
    """The solve of one right-hand side through the plan's tables; rows in permuted order."""
    n = L.shape[0]
    L, U = L.tocsr(), U.tocsr()
    pos, fronts = P["pos"], P["fronts"]
    assert sorted(pos) == list(range(n))
    perm = np.argsort(pos)              # front order -> permuted row
    W, X = np.zeros(n), np.full(n, np.nan)
    W[pos] = b
    Y, C = np.full(n, np.nan), np.full(P["n_c"] + 1, np.nan)
    C[P["n_c"]] = 0.0
    blocks = []
    for f in fronts:
        c = perm[f["off"]:f["off"] + f["w"]]
        assert np.all(np.diff(c) > 0) and np.all(P["local_of"][c] == np.arange(f["w"]))
        B = P["bperm"][f["brow"]:f["brow"] + f["r"]]
        assert np.all(np.diff(B) > 0) and np.all(P["brow"][f["brow"]:f["brow"] + f["r"]] == pos[B])
        assert f["brow"] % 4 == 0
        Lc, Uc = L[c][:, c].toarray(), U[c][:, c].toarray()
        Li, Ui = np.linalg.inv(Lc), np.linalg.inv(Uc)
        K = np.hstack([Ui @ Li, -Ui @ U[c][:, B].toarray()])
        blocks.append((c, -L[B][:, c].toarray() @ Li, K, B))

    def gathered(row):
        a = P["arow"][row]
        src = list(a["s"]) + list(P["xsrc"][a["xb"]:a["xe"]])
        assert all(0 <= s <= P["n_c"] for s in src)
        v = C[src].sum()
        assert np.isfinite(v), "a contribution read before it was written"
        return v

    done = np.zeros(len(fronts), int)
    for h, lv in enumerate(P["levels"]):
        seen = {}
        for t in P["tasks"][lv["f0"]:lv["f0"] + lv["nf"]]:
            seen.setdefault(int(t["front"]), []).append(int(t["tile"]))
        for t in P["tasks"][lv["k0"]:lv["k0"] + lv["nk"]]:   # K's tasks cover every row of every front
            done[t["front"]] += min(16, fronts[t["front"]]["w"] - 16 * t["tile"])
            assert fronts[t["front"]]["w"] <= lv["wmax"]
        new = {}
        for fi, tiles in seen.items():
            f, (c, F, K, B) = fronts[fi], blocks[fi]
            assert tiles == list(range(max((int(f["r"]) + 15) // 16, 1 if h else 0)))
            v = W[f["off"]:f["off"] + f["w"]].copy()
            if h:
                v += [gathered(f["arow"] + q) for q in range(f["w"])]
                Y[f["off"]:f["off"] + f["w"]] = v
            new[fi] = F @ v + ([gathered(f["arow"] + f["w"] + q) for q in range(f["r"])] if h else 0.0)
        for fi, v in new.items():
            C[fronts[fi]["c"]:fronts[fi]["c"] + fronts[fi]["r"]] = v
    assert np.array_equal(done, fronts["w"])
    for h in range(len(P["levels"]) - 1, -1, -1):
        lv = P["levels"][h]
        for fi in sorted({int(t["front"]) for t in P["tasks"][lv["k0"]:lv["k0"] + lv["nk"]]}):
            f, (c, F, K, B) = fronts[fi], blocks[fi]
            s = slice(f["off"], f["off"] + f["w"])
            X[s] = K @ np.concatenate([(Y if h else W)[s], X[pos[B]]])
    return X[pos]


def superlu(A, **kw):
    lu = spla.splu(A.tocsc(), **kw)
    return lu.L.tocsc(), lu.U.tocsc()


def systems():
    from neurips2026_smart_building_challenge_amd.scenario import fdm as F

    rng = np.random.default_rng(5)
    for spec in (F.FdmSpec(rows=120, cols=90, rooms=7, margin=6, seed=3), F.FdmSpec(rows=61, cols=203, rooms=3, margin=5)):
        yield spec.name, superlu(F.make_plan(spec).A, permc_spec="MMD_AT_PLUS_A")
    R = sp.random(700, 700, 0.004, random_state=1) + sp.diags(rng.uniform(0.05, 0.4, 700))   # pivots off the diagonal
    yield "unsymmetric", superlu(R + sp.eye(700) * 0.01, permc_spec="COLAMD")
    for n in (1, 5, 64, 65):
        yield f"dense{n}", superlu(sp.csc_matrix(rng.normal(size=(n, n)) + 3 * n * np.eye(n)), permc_spec="NATURAL")
    yield "dense600", superlu(sp.csc_matrix(rng.normal(size=(600, 600)) + 60 * np.eye(600)), permc_spec="NATURAL")
    tri = lambda n: sp.diags([np.full(n - 1, -1.0), np.full(n, 2.5), np.full(n - 1, -1.2)], [-1, 0, 1])
    yield "chain", superlu(tri(1500), permc_spec="NATURAL")
    yield "forest", superlu(sp.block_diag([tri(300), tri(17), F.make_plan(F.FdmSpec(rows=40, cols=44, rooms=2, margin=3)).A,
                                           sp.eye(3)]), permc_spec="MMD_AT_PLUS_A")
    n, hub = 40 * 70 + 30, 30   # forty chains that all reach the same 30 columns
    S = sp.block_diag([tri(70)] * 40 + [sp.eye(hub) * 300.0]).tolil()
    for b in range(40):
        S[n - hub:, 70 * b + 69] = -0.1
        S[70 * b + 69, n - hub:] = -0.1
    yield "star", superlu(S, permc_spec="NATURAL")


def test_front_plan_solves(planner):
    rng = np.random.default_rng(9)
    names, extras, high = [], 0, 0
    for name, (L, U) in systems():
        n = L.shape[0]
        P = plan_of(planner, L, U)
        b = rng.normal(size=n)
        x = execute(P, L, U, b)
        ref = spla.spsolve_triangular(U.tocsr(), spla.spsolve_triangular(L.tocsr(), b, lower=True, unit_diagonal=True),
                                      lower=False)
        # two backward-stable solves of one system: eps times its condition (dense inverses of the
        # small blocks included), measured 1e-15..2e-12; a wrong entry or row gives errors of order 1
        assert np.max(np.abs(x - ref)) <= 1e-9 * np.max(np.abs(ref)), name
        names.append(name)
        extras += int(np.sum(P["arow"]["xe"] > P["arow"]["xb"]))
        high = max(high, len(P["levels"]))
        fr = P["fronts"]
        assert fr["w"].max() <= 256 and fr["w"].sum() == n
        assert P["ops"] == sum(64 * ((f["r"] + 15) // 16 * ((f["w"] + 3) // 4)
                                     + (f["w"] + 15) // 16 * ((f["w"] + 3) // 4 + (f["r"] + 3) // 4)) for f in fr)
    assert len(names) == 11 and extras > 0 and high >= 5
