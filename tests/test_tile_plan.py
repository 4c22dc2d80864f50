"""CPU checks of the plan of the tiled sparse factorisation (xg_tileplan.h,
the host code whose arrays the kernels of xg_tiles.hip read): positions a
bijection onto the columns' slots, every index in bounds, each level's
updates onto tiles of later levels only, and the factorisation and sweeps
run in numpy exactly as the launches run them -- level by level, from the
task lists -- solving the oracle's assembled tangents to rounding; for
layered, moved, scattered and coincident node positions, fixed DOFs inside
the model and several components."""
import os
import subprocess

import numpy as np
import pytest

from tests import _oracle
from xara_amd import meshes

HERE = os.path.dirname(os.path.abspath(__file__))
T = 64
NAMES = ("pos wid colptr row lev levptr levcol upptr uptgt upsrc srcg srca srck fwptr fwrow fwsrc fwg fwk "
         "bwptr bwcol bwsrc bwg bwr").split()


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("tileplan") / "tile_plan_driver")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "tile_plan_driver.cpp")], check=True)
    return exe


def plan(driver, tmp_path, rp, ci, eq, crd, max_tiles=1e6, max_flops=1e15):
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    with open(fin, "wb") as f:
        np.array([len(rp) - 1, len(crd), eq.shape[1], crd.shape[1], len(ci)], np.int32).tofile(f)
        for a in (rp, ci, eq):
            np.asarray(a, np.int32).tofile(f)
        np.asarray(crd, np.float64).tofile(f)
        np.array([max_tiles, max_flops]).tofile(f)
    subprocess.run([driver, fin, fout], check=True)
    o = np.fromfile(fout, np.int32)
    if not o[0]:
        return None
    P, at = dict(nt=int(o[1]), nlev=int(o[2])), 3
    for name in NAMES:
        n = o[at]
        P[name] = o[at + 1:at + 1 + n]
        at += 1 + n
    assert at == len(o)
    return P


def check_indices(P, n):
    nt, cp = P["nt"], P["colptr"]
    pos = P["pos"]
    assert len(pos) == n and len(np.unique(pos)) == n and pos.min() >= 0
    assert np.array_equal(np.bincount(pos // T, minlength=nt), P["wid"]) and np.all(pos % T < P["wid"][pos // T])
    assert P["wid"].min() >= 1 and P["wid"].max() <= T
    slots = len(P["row"]) + nt
    col_of = np.repeat(np.arange(nt), np.diff(cp) + 1)  # column of each slot
    row_of = np.concatenate([np.concatenate([[k], P["row"][cp[k]:cp[k + 1]]]) for k in range(nt)])
    assert np.all(row_of >= col_of) and row_of.max() < nt
    for k in range(nt):
        assert np.all(np.diff(P["row"][cp[k]:cp[k + 1]]) > 0)
        assert np.all(P["lev"][P["row"][cp[k]:cp[k + 1]]] > P["lev"][k])
    assert np.array_equal(np.sort(P["levcol"]), np.arange(nt)) and P["levptr"][-1] == nt
    assert P["upptr"][-1] == len(P["uptgt"]) and P["upsrc"][-1] == len(P["srcg"]) == len(P["srca"])
    assert P["fwptr"][-1] == len(P["fwrow"]) and P["fwsrc"][-1] == len(P["fwg"]) == len(P["fwk"])
    for l in range(P["nlev"]):
        t = np.arange(P["upptr"][l], P["upptr"][l + 1])
        assert len(np.unique(P["uptgt"][t])) == len(t)  # one workgroup per target
        for i in t:
            s = slice(P["upsrc"][i], P["upsrc"][i + 1])
            g, a, tgt = P["srcg"][s], P["srca"][s], P["uptgt"][i]
            assert len(g) and g.max() < slots and tgt < slots
            # from this level's columns, or earlier ones of a run that ends in it
            assert np.all(P["lev"][col_of[g]] <= l) and np.array_equal(col_of[g], col_of[a])
            assert P["lev"][col_of[tgt]] > l and np.all(np.diff(col_of[g]) > 0)
            assert np.all(row_of[g] == row_of[tgt]) and np.all(row_of[a] == col_of[tgt])
            assert np.all(g != a + 0 * g) or row_of[tgt] == col_of[tgt]
            assert np.array_equal(P["srck"][s], (P["wid"][col_of[g]] + 15) // 16 * 16)
        f = np.arange(P["fwptr"][l], P["fwptr"][l + 1])
        assert len(np.unique(P["fwrow"][f])) == len(f)
        for i in f:
            s = slice(P["fwsrc"][i], P["fwsrc"][i + 1])
            assert np.all(row_of[P["fwg"][s]] == P["fwrow"][i]) and np.array_equal(col_of[P["fwg"][s]], P["fwk"][s])
            assert np.all(P["lev"][P["fwk"][s]] == l)
        w = np.arange(P["bwptr"][l], P["bwptr"][l + 1])
        assert len(np.unique(P["bwcol"][w])) == len(w)
        for i in w:
            s = slice(P["bwsrc"][i], P["bwsrc"][i + 1])
            assert np.all(col_of[P["bwg"][s]] == P["bwcol"][i]) and np.array_equal(row_of[P["bwg"][s]], P["bwr"][s])
            assert np.all(P["lev"][P["bwr"][s]] == l)
    assert P["bwptr"][-1] == len(P["bwcol"]) and P["bwsrc"][-1] == len(P["bwg"]) == len(P["bwr"])
    return row_of, col_of


def solve(P, K, b, row_of, col_of):
    """The launches in numpy: gather, levels of panel and update, sweeps."""
    nt, cp, pos = P["nt"], P["colptr"], P["pos"]
    n, npad = len(pos), T * nt
    D = np.zeros((npad, npad))
    D[np.ix_(pos, pos)] = K
    A = np.stack([D[T * i:T * i + T, T * j:T * j + T] for i, j in zip(row_of, col_of)])
    held = np.zeros((nt, nt), bool)
    held[row_of, col_of] = True
    for i in range(nt):
        for j in range(i):
            assert held[i, j] or not D[T * i:T * i + T, T * j:T * j + T].any()
    for k in range(nt):
        for i in range(P["wid"][k], T):
            A[cp[k] + k, i, i] = 1.0
    G = np.zeros_like(A)
    for l in range(P["nlev"]):
        for k in P["levcol"][P["levptr"][l]:P["levptr"][l + 1]]:
            d = cp[k] + k
            inv = np.linalg.inv(A[d])
            w16 = (P["wid"][k] + 15) // 16 * 16
            inv[w16:], inv[:, w16:] = 0, 0
            G[d] = inv
            for s in range(d + 1, d + 1 + cp[k + 1] - cp[k]):
                G[s] = A[s] @ inv
        for t in range(P["upptr"][l], P["upptr"][l + 1]):
            for s in range(P["upsrc"][t], P["upsrc"][t + 1]):
                kc = P["srck"][s]
                A[P["uptgt"][t]] -= G[P["srcg"][s]][:, :kc] @ A[P["srca"][s]][:, :kc].T
    Y, X = np.zeros((nt, T)), np.zeros((nt, T))
    Y.reshape(-1)[pos] = b
    for l in range(P["nlev"]):
        for t in range(P["fwptr"][l], P["fwptr"][l + 1]):
            for s in range(P["fwsrc"][t], P["fwsrc"][t + 1]):
                Y[P["fwrow"][t]] -= G[P["fwg"][s]] @ Y[P["fwk"][s]]
    for k in range(nt):
        X[k] = G[cp[k] + k] @ Y[k]
    for l in range(P["nlev"] - 1, -1, -1):
        for t in range(P["bwptr"][l], P["bwptr"][l + 1]):
            for s in range(P["bwsrc"][t], P["bwsrc"][t + 1]):
                X[P["bwcol"][t]] -= G[P["bwg"][s]].T @ X[P["bwr"][s]]
    return X.reshape(-1)[pos]


def models(case):
    rng = np.random.default_rng(3)
    if case in ("quad", "quad_moved"):
        mesh = meshes.quad_strip(33, 9)
        if case == "quad_moved":
            mesh["crds"] += rng.uniform(-0.03, 0.03, mesh["crds"].shape)
        o = _oracle.oracle_model(2, 2)
        meshes.build_quad_strip(o, mesh)
        return o, mesh["crds"]
    if case == "quad_fixed":  # fixed nodes inside cut the model in parts
        mesh = meshes.quad_strip(24, 5)
        o = _oracle.oracle_model(2, 2)
        mesh["fixed_nodes"] = np.array([t for t in mesh["node_tags"] if (t - 1) % 25 in (0, 12)], np.int32)
        meshes.build_quad_strip(o, mesh)
        o.fix(30, 0, 1)
        return o, mesh["crds"]
    if case == "brick":
        mesh = meshes.brick_cube(6)
        mesh["crds"][:, 0] += 0.02 * rng.normal(size=len(mesh["crds"]))
        o = _oracle.oracle_model(3, 3)
        meshes.build_brick_cube(o, mesh)
        return o, mesh["crds"]
    fr = meshes.rc_frame_3d(3, 2, 5) if case == "frame3d" else meshes.rc_frame_2d(9, 3)
    o = _oracle.oracle_model(3, 6) if case == "frame3d" else _oracle.oracle_model(2, 3)
    (meshes.build_rc_frame_3d if case == "frame3d" else meshes.build_rc_frame_2d)(o, fr)
    return o, fr["crds"]


@pytest.mark.parametrize("where", ["own", "scattered", "one_point"])
@pytest.mark.parametrize("case", ["quad", "quad_moved", "quad_fixed", "brick", "frame3d", "frame2d"])
def test_plan_solves(driver, tmp_path, case, where):
    """The order uses the coordinates only to choose its cuts: any will do."""
    o, crd = models(case)
    o.setup()
    rp, ci = o.csr_pattern()
    K = np.zeros((o.neq, o.neq))
    K[np.repeat(np.arange(o.neq), np.diff(rp)), ci] = o.form_tangent()
    rng = np.random.default_rng(4)
    if where == "scattered":
        crd = rng.normal(size=crd.shape)
    elif where == "one_point":
        crd = np.zeros_like(crd)
    P = plan(driver, tmp_path, rp, ci, o.node_eqns(), crd)
    row_of, col_of = check_indices(P, o.neq)
    x = rng.normal(size=o.neq)
    b = K @ x
    got = solve(P, K, b, row_of, col_of)
    # backward error: a block elimination of an SPD matrix is stable to a
    # small multiple of n eps |K| |x|
    assert np.abs(K @ got - b).max() <= 1e-13 * len(b) * np.abs(K).max() * np.abs(got).max()
    o.close()


def test_limits_refuse(driver, tmp_path):
    o, crd = models("quad")
    o.setup()
    rp, ci = o.csr_pattern()
    eq = o.node_eqns()
    P = plan(driver, tmp_path, rp, ci, eq, crd)
    tiles = len(P["row"]) + P["nt"]
    assert plan(driver, tmp_path, rp, ci, eq, crd, max_tiles=tiles) is not None
    assert plan(driver, tmp_path, rp, ci, eq, crd, max_tiles=tiles - 1) is None
    assert plan(driver, tmp_path, rp, ci, eq, crd, max_flops=1e3) is None
    o.close()
