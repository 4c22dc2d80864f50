"""GPU parity of the tiled sparse factorisation (xg_tiles.hip) against the
CPU oracle's direct solve, at the edges of its sizes: the fewest equations
it takes, columns of 1 to 64 equations, one to many levels, DOFs fixed inside
the model, 1 to many sources per update; single solves, the allocation-free
solve bit for bit, and the paired solves of DisplacementControl."""
import os
import time

import numpy as np
import pytest
import torch

from tests import _oracle
from xara_amd import _lib, meshes
from xara_amd.model import Model, XaraError

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def build(case, m):
    kind, *size = case
    if kind == "quad":
        mesh = meshes.quad_strip(*size)
        mesh["crds"] = mesh["crds"] + np.random.default_rng(1).uniform(-0.02, 0.02, mesh["crds"].shape)
        meshes.build_quad_strip(m, mesh)
        m.fix(mesh["tip"] - 2, 0, 1)
        return mesh["tip"], 2, 1e-3, np.random.default_rng(2).normal(0, 1e-3, mesh["crds"].shape)
    if kind == "brick":
        mesh = meshes.brick_cube(size[0])
        meshes.build_brick_cube(m, mesh)
        return int(mesh["load_tags"][0]), 3, -1e-3, np.random.default_rng(2).normal(0, 1e-4, mesh["crds"].shape)
    fr = meshes.rc_frame_3d(*size)
    meshes.build_rc_frame_3d(m, fr)
    U = np.random.default_rng(2).normal(0, 1e-2, (len(fr["crds"]), 6))
    U[:, 3:] *= 1e-4
    return fr["roof"], 1, 2.0, U


CASES = [("quad", 14, 13), ("quad", 15, 13), ("quad", 5, 40), ("quad", 97, 1), ("quad", 61, 17), ("brick", 5),
         ("brick", 9), ("frame", 3, 2, 6), ("frame", 7, 1, 11)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "_".join(map(str, c)))
def test_tiled_solve_matches_oracle(case):
    print(f"case: tiled solve {case}", flush=True)
    ndm, ndf = {"quad": (2, 2), "brick": (3, 3), "frame": (3, 6)}[case[0]]
    g, o = Model(ndm, ndf), _oracle.oracle_model(ndm, ndf)
    for m in (g, o):
        node, dof, incr, U = build(case, m)
        if case[0] == "quad":
            m.load(node, 0.0, 1.0)
        m.system("GpuBlockPCG", 1e-13, 1000)
        m.setup()
        m.set_trial_disp(U)
        m.update()
        m.form_tangent(values=False)
    # residual: the iteration's own stop test (1e-13 |b|) and the rounding of
    # the product it is formed with, eps sum |A| |x| per row; solutions to
    # the condition number times the rounding, below the parity bar of 1e-9
    rp, ci = o.csr_pattern()
    absA = np.abs(o.form_tangent())
    row = np.repeat(np.arange(o.neq), np.diff(rp))
    for seed in range(3):
        B = np.random.default_rng(seed).normal(size=g.neq)
        c0 = g.counters()
        X = g.solve(B)
        c1 = g.counters()
        assert g.preconditioner() == "tiled" and c1["band_bw"] > 0 and c1["cg_iters"] - c0["cg_iters"] <= 2
        noise = np.bincount(row, absA * np.abs(X)[ci], o.neq)
        assert np.linalg.norm(o.spmv(X) - B) <= 1e-13 * np.linalg.norm(B) + 4 * EPS * np.linalg.norm(noise)
        assert relerr(X, o.solve(B)) <= 1e-9
        Xn = np.zeros_like(X)
        assert g._b.solve_noalloc(g._h, B.ctypes.data_as(_lib.P_D), Xn.ctypes.data_as(_lib.P_D)) == 0
        assert np.array_equal(X, Xn)
    for m in (g, o):
        m.revert_to_start()
        m.test("NormUnbalance", 1e-6 if case[0] != "frame" else 1e-3, 30)
        m.integrator("DisplacementControl", node, dof, incr)
        assert m.analyze(3) == 0
    assert relerr(g.trial_disp(), o.trial_disp()) <= 1e-9
    assert abs(g.load_factor - o.load_factor) <= 1e-9 * abs(o.load_factor)
    for m in (g, o):
        m.close()


def test_equation_limit():
    """384 equations (16 x 12 x 2) stay with the solves that take fewer, 385
    (one more DOF freed at the clamped end) are factored; the same solutions
    with and without."""
    for free in (0, 1):
        m = Model(2, 2)
        mesh = meshes.quad_strip(16, 11)
        if free:
            mesh["fixed_nodes"] = mesh["fixed_nodes"][1:]
        meshes.build_quad_strip(m, mesh)
        if free:
            m.fix(1, 1, 0)
        m.cg_config(wide=True)
        m.setup()
        assert m.neq == 384 + free
        m.form_tangent(values=False)
        assert m.preconditioner() == ("tiled" if free else "band")
        B = np.ones(m.neq)
        X = m.solve(B)
        m.cg_config(wide=False)
        assert m.preconditioner() == "band"
        assert relerr(X, m.solve(B)) <= 1e-9
        m.close()


def test_large_solid_goes_on_with_the_factor():
    """A solid whose factor costs many PCG iterations starts with block
    Jacobi; the plastic tangent that needs more is factored, and the steps
    after it, until revertToStart: the same trajectory as block Jacobi alone
    to the solver's tolerance, in fewer iterations, and the same again."""
    print("case: large solid 25^3", flush=True)
    runs = []
    for wide in (True, False):
        m = Model(3, 3)
        mesh = meshes.brick_cube(25)
        meshes.build_brick_cube(m, mesh)
        m.system("GpuBlockPCG", 1e-12, 20000)
        m.cg_config(wide=wide)
        m.test("NormUnbalance", 1e-7, 30)
        m.integrator("LoadControl", 93.0)
        m.setup()
        for again in range(2 if wide else 1):
            m.revert_to_start()
            c0 = m.counters()
            t = []
            for _ in range(3):
                assert m.analyze(1) == 0
                t.append(m.trial_disp())
                if wide and not t[1:]:
                    assert m.preconditioner() == "jacobi"  # elastic: not worth a factor
            c = m.counters()
            assert m.preconditioner() == ("tiled" if wide else "jacobi")
            runs.append((np.array(t), c["cg_iters"] - c0["cg_iters"]))
        m.close()
    (a, ia), (b, ib), (c, ic) = runs
    assert relerr(a, c) <= 1e-9 and relerr(b, c) <= 1e-9
    assert ia < 0.8 * ic and ib < 0.8 * ic


def test_failed_setup_leaves_no_thread():
    """The plan is built on a thread beside the set-up and reads the model's
    numbering and coordinates: a set-up that fails (here on an element of no
    length, while the plan of 40,000 loose nodes is being built) returns with
    that thread ended, and the corrected model is set up as a fresh one is."""
    print("case: failed set-up with 40,000 loose nodes", flush=True)
    fr = meshes.rc_frame_3d(3, 3, 6)
    fresh, m = Model(3, 6), Model(3, 6)
    for g in (fresh, m):
        meshes.build_rc_frame_3d(g, fr)
    fresh.setup()  # the runtime's own threads exist from here on
    loose = np.arange(10**6, 10**6 + 40000, dtype=np.int32)
    m.nodes(loose, np.random.default_rng(1).uniform(0, 1e4, (len(loose), 3)))
    below, top = (int(np.flatnonzero(fr["node_tags"] == t)[0]) for t in fr["columns"][-1])
    tag = fr["node_tags"][top:top + 1]
    m.nodes(tag, fr["crds"][below:below + 1])
    for _ in range(2):
        before = set(os.listdir("/proc/self/task"))
        with pytest.raises(XaraError, match="zero length"):
            m.setup()
        time.sleep(0.005)  # a joined thread's entry goes a moment later
        assert set(os.listdir("/proc/self/task")) <= before
    m.nodes(tag, fr["crds"][top:top + 1])
    m.fix_many(loose, np.ones((len(loose), 6), np.int32))
    m.setup()
    B = np.random.default_rng(0).normal(size=m.neq)
    X = []
    for g in (m, fresh):
        g.form_tangent(values=False)
        X.append(g.solve(B))
        assert g.preconditioner() == "tiled"
        g.close()
    assert np.array_equal(*X)


def frame_model(size, integrator):
    m = Model(3, 6)
    fr = meshes.rc_frame_3d(*size)
    meshes.build_rc_frame_3d(m, fr)
    m.system("GpuBlockPCG", 1e-12, 20000)
    if integrator == "Newmark":
        m.masses(fr["load_tags"], np.tile([1.0, 1.0, 1.0, 0, 0, 0], (len(fr["load_tags"]), 1)))
    m.integrator(integrator, *((0.5, 0.25) if integrator == "Newmark" else (1.0,)))
    return m


def taken(make):
    """(model set up, device bytes its set-up took)"""
    m = make()
    free = torch.cuda.mem_get_info()[0]
    m.setup()
    return m, free - torch.cuda.mem_get_info()[0]


def test_factor_memory_is_taken_when_a_solve_uses_it():
    """A model set up as a transient takes no memory for the factor (2 x 57
    MB for this 9 x 9 x 12 frame); its first static solve does, and is the one
    of a model set up for static steps.  The allocation-free solve before it
    goes without the factor."""
    print("case: factor memory, 9 x 9 x 12 frame", flush=True)
    frame_model((3, 3, 6), "LoadControl").setup()
    st, a = taken(lambda: frame_model((9, 9, 12), "LoadControl"))
    tr, b = taken(lambda: frame_model((9, 9, 12), "Newmark"))
    assert a - b > 90 << 20
    B = np.random.default_rng(0).normal(size=st.neq)
    st.form_tangent(values=False)
    X = st.solve(B)
    tr.integrator("LoadControl", 1.0)
    tr.form_tangent(values=False)
    Xn = np.zeros_like(X)
    assert tr._b.solve_noalloc(tr._h, B.ctypes.data_as(_lib.P_D), Xn.ctypes.data_as(_lib.P_D)) == 0
    assert tr.preconditioner() == "jacobi" and relerr(Xn, X) <= 1e-8
    assert np.array_equal(tr.solve(B), X)
    assert tr.preconditioner() == st.preconditioner() == "tiled"
    assert tr._b.solve_noalloc(tr._h, B.ctypes.data_as(_lib.P_D), Xn.ctypes.data_as(_lib.P_D)) == 0
    assert np.array_equal(Xn, X)
    st.close()
    tr.close()


@pytest.mark.parametrize("case", [("brick", 25), ("quad", 40, 7), ("frame", 5, 5, 8)],
                         ids=lambda c: "_".join(map(str, c)))
def test_without_memory_for_the_factor(case, monkeypatch):
    """A model whose factor finds no memory (here: more than XG_TILE_MIB
    allows) is set up and solved as without the factor: the band factor where
    the band is narrow, else block Jacobi, step for step."""
    print(f"case: no memory for the factor {case}", flush=True)
    ndm, ndf = {"quad": (2, 2), "brick": (3, 3), "frame": (3, 6)}[case[0]]
    runs = []
    for mib in (None, "1"):
        if mib:
            monkeypatch.setenv("XG_TILE_MIB", mib)
        m = Model(ndm, ndf)
        node, dof, incr, _ = build(case, m)
        m.system("GpuBlockPCG", 1e-12, 20000)
        m.cg_config(wide=mib is not None)
        if case[0] == "brick":
            m.test("NormUnbalance", 1e-7, 30)
            m.integrator("LoadControl", 93.0)
        else:
            if case[0] == "quad":
                m.load(node, 0.0, 1.0)
            m.test("NormUnbalance", 1e-6 if case[0] == "quad" else 1e-3, 30)
            m.integrator("DisplacementControl", node, dof, incr)
        m.setup()
        assert m.analyze(3) == 0
        assert m.preconditioner() == ("band" if case[0] == "quad" else "jacobi")
        runs.append((m.trial_disp(), m.counters()["cg_iters"]))
        m.close()
    assert np.array_equal(runs[0][0], runs[1][0]) and runs[0][1] == runs[1][1]


@pytest.mark.parametrize("size", [(20, 11), (20, 20), (31, 9)], ids=lambda c: "_".join(map(str, c)))
def test_factor_without_enough_supports_gives_way(size):
    """A strip with no support, or with one node held, under loads in balance:
    the last pivots are rounding, of either sign.  Where they all come out
    positive the PCG fails with the factor, which is dropped for block Jacobi
    as it is where one does not."""
    for held in ((), (1, 0), (1, 1)):
        for seed in range(4):
            print(f"case: too few supports {size} {held} {seed}", flush=True)
            mesh = meshes.quad_strip(*size)
            rng = np.random.default_rng(seed)
            m = Model(2, 2)
            m.nodes(mesh["node_tags"], mesh["crds"] + rng.uniform(-0.02, 0.02, mesh["crds"].shape))
            mat = meshes.J2_STEEL
            m.nDMaterial("J2Plasticity", 1, mat["K"], mat["G"], mat["sig0"], mat["sigInf"], mat["delta"], mat["H"])
            m.elements("quad", mesh["ele_tags"], mesh["conn"], 1.0, 1)
            if held:
                m.fix(int(mesh["node_tags"][0]), *held)
            m.system("GpuBlockPCG", 1e-10, 20000)
            m.setup()
            m.form_tangent(values=False)
            assert m.preconditioner() == "tiled"
            b = m.spmv(1e-3 * rng.normal(size=m.neq))
            assert np.linalg.norm(m.spmv(m.solve(b)) - b) <= 1.1e-10 * np.linalg.norm(b)
            m.close()


@pytest.mark.parametrize("wide", [True, False], ids=["tiled", "band"])
@pytest.mark.parametrize("control", ["load", "displacement"])
def test_dropped_factor_keeps_the_warm_start(control, wide):
    """Elastic fibers of a negative modulus: no pivot is positive, so the
    exact factor is dropped for every matrix, and block Jacobi solves the
    negative definite system.  A step's first solve (LoadControl) and the
    solves for the reference load (DisplacementControl; with the band factor
    the predictor's only) still start from the last one's solution: of 4
    solves 3 end at once, of 12 solves 7 (3)."""
    print(f"case: warm start without the factor, {control} {wide}", flush=True)
    fr = meshes.rc_frame_2d(24, 15)
    its = []
    for warm in (True, False):
        m = Model(2, 3)
        m.nodes(fr["node_tags"], fr["crds"])
        m.fix_many(fr["fixed_nodes"], np.ones((len(fr["fixed_nodes"]), 3), np.int32))
        m.uniaxialMaterial("Elastic", 1, -2e5)
        m.section("Fiber", 1, [(y, 0.0, 1e4, 1) for y in (-200.0, -100.0, 100.0, 200.0)])
        m.geomTransf("Linear", 1)
        conn = np.concatenate([fr["columns"], fr["beams"]])
        m.elements("dispBeamColumn", np.arange(1, len(conn) + 1), conn, 1, 1, 5)
        P = np.zeros((len(fr["floor_nodes"]), 3))
        P[:, 0] = 1.0
        m.loads(fr["floor_nodes"], P)
        m.system("GpuBlockPCG", 1e-8, 50000)
        m.cg_config(warm=warm, wide=wide)
        m.test("NormUnbalance", 1e-2, 20)
        if control == "load":
            m.integrator("LoadControl", 10.0)
        else:
            m.integrator("DisplacementControl", fr["roof"], 1, 5.0)
        m.setup()
        assert m.neq > 1024 and m.preconditioner() == ("tiled" if wide else "band")
        assert m.analyze(4) == 0
        c = m.counters()
        assert c["band_fallbacks"] > 0
        its.append(c["cg_iters"])
        m.close()
    assert its[0] < (0.6 if wide or control == "load" else 0.8) * its[1]


def test_large_solid_tries_block_jacobi_again(monkeypatch):
    """A solid that has gone on with the factor tries block Jacobi again after
    64 factored matrices: while the steps stay hard every solve is finished by
    the factor, elastic unloading returns to iterations at the next try."""
    print("case: large solid 25^3 unloaded", flush=True)
    monkeypatch.setenv("XG_PC_REUSE", "0")  # count a factor for every matrix
    m = Model(3, 3)
    mesh = meshes.brick_cube(25)
    meshes.build_brick_cube(m, mesh)
    m.system("GpuBlockPCG", 1e-10, 20000)
    m.test("NormUnbalance", 1e-7, 30)
    m.integrator("LoadControl", 93.0)
    m.setup()
    b = np.zeros(m.neq)
    m.set_load_factor(1.0)
    b[:] = m.form_unbalance()
    m.set_load_factor(0.0)
    assert m.analyze(3) == 0
    U = m.trial_disp()

    def solves(scale, n):
        its, on = [], []
        m.set_trial_disp(scale * U)
        m.update()
        for _ in range(n):
            m.form_tangent(values=False)
            c = m.counters()["cg_iters"]
            X = m.solve(b)
            its.append(m.counters()["cg_iters"] - c)
            on.append(m.preconditioner() == "tiled")
        return its, on, X
    its, on, X = solves(1.02, 90)  # loading on: block Jacobi alone would not do
    assert on == [True] * 90
    assert 1 <= sum(i > 30 for i in its) <= 2  # the tries
    its, on, Xe = solves(0.98, 70)
    assert max(its[:1]) <= 3 and on[0] and not on[-1]
    assert on == sorted(on, reverse=True) and 1 <= sum(on) <= 64
    assert min(its[sum(on):]) > 30
    m.close()
