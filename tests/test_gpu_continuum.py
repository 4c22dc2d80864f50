"""GPU parity of the J2 continuum path (stdBrick, FourNodeQuad) against the
CPU oracle through the C-ABI: numbering and CSR pattern bit-exact, stresses,
tangents, assembled systems and converged trajectories to 1e-9 relative."""
import numpy as np
import pytest

from tests import _oracle
from xara_amd import meshes
from xara_amd.model import Model, XaraError

pytestmark = pytest.mark.gpu

RTOL = 1e-9  # relative tolerance of the FP64 parity bar


def relerr(a, b):
    a, b = np.asarray(a), np.asarray(b)
    scale = np.max(np.abs(b))
    return 0.0 if scale == 0 else float(np.max(np.abs(a - b)) / scale)


def cube_pair(n, system="GpuPCG", pressure=1.0):
    mesh = meshes.brick_cube(n)
    models = []
    for m in (Model(3, 3), _oracle.oracle_model(3, 3)):
        meshes.build_brick_cube(m, mesh, pressure=pressure)
        m.system(system, 1e-13, 20000)
        m.setup()
        models.append(m)
    return mesh, models


def random_field(mesh, scale, seed):
    rng = np.random.default_rng(seed)
    crd = mesh["crds"]
    U = scale * (np.sin(3.1 * crd @ np.array([1.0, 0.7, 0.3]))[:, None] * rng.normal(size=(1, 3))
                 + 0.3 * rng.normal(size=crd.shape))
    U[mesh["node_tags"] <= 0] = 0
    return U


def test_numbering_and_csr_bit_exact():
    print("case: brick cube 5^3 numbering", flush=True)
    mesh, (g, o) = cube_pair(5)
    assert np.array_equal(g.node_eqns(), o.node_eqns())
    rg, cg = g.csr_pattern()
    ro, co = o.csr_pattern()
    assert np.array_equal(rg, ro) and np.array_equal(cg, co)


@pytest.mark.parametrize("n,seed", [(3, 0), (6, 1)])
def test_brick_update_stress_tangent(n, seed):
    print(f"case: brick update n={n} seed={seed}", flush=True)
    mesh, (g, o) = cube_pair(n)
    npts = 8 * n ** 3
    for step in range(3):
        U = random_field(mesh, 2e-3 * (step + 1), seed + 10 * step)
        for m in (g, o):
            m.set_trial_disp(U)
            m.update()
        for what in ("stress", "tangent", "plastic"):
            a, b = g.point_data(what, npts), o.point_data(what, npts)
            assert relerr(a, b) <= RTOL, (what, step, relerr(a, b))
        # some points must be plastic for the check to mean anything
        xi = o.point_data("plastic", npts)[:, 6]
        assert (xi > 0).any()
        for m in (g, o):
            m.commit()


def test_brick_assembly_parity():
    print("case: brick assembly n=4", flush=True)
    mesh, (g, o) = cube_pair(4)
    U = random_field(mesh, 3e-3, 7)
    for m in (g, o):
        m.set_trial_disp(U)
        m.update()
        m.set_load_factor(50.0)
    Kg, Ko = g.form_tangent(), o.form_tangent()
    assert relerr(Kg, Ko) <= RTOL
    Bg, Bo = g.form_unbalance(), o.form_unbalance()
    assert relerr(Bg, Bo) <= RTOL
    tag = int(mesh["ele_tags"][17])
    assert relerr(g.element_tangent(tag), o.element_tangent(tag)) <= RTOL
    assert relerr(g.element_resisting_force(tag), o.element_resisting_force(tag)) <= RTOL


def test_brick_tangent_into_csr_matches_element_matrices(monkeypatch):
    """formTangent of a stdBrick-only model straight into the CSR values
    (k_brick_tangent_csr: no element matrices, the J2 blocks in closed form)
    against the element-matrix path (k_brick_tangent's BaT D Bb + the gather
    assembly, XG_BRICK_TANGENT_CSR=0): the same values to rounding
    (1e-13 of the largest entry) on a plastic state of a 7^3 cube, and again
    after a commit and a further update."""
    print("case: brick tangent into CSR, 7^3", flush=True)
    n = 7
    mesh = meshes.brick_cube(n)
    U = random_field(mesh, 4e-3, 3)
    out = []
    for env in ("1", "0"):
        monkeypatch.setenv("XG_BRICK_TANGENT_CSR", env)
        m = Model(3, 3)
        meshes.build_brick_cube(m, mesh)
        m.system("GpuBlockPCG", 1e-12, 1000)
        m.setup()
        m.set_trial_disp(U)
        assert m.update() == 0
        plastic = float((m.point_data("plastic", 8 * n ** 3)[:, 6] > 0).mean())
        K1 = m.form_tangent()
        m.commit()
        m.set_trial_disp(1.5 * U)
        assert m.update() == 0
        K2 = m.form_tangent()
        out.append((K1, K2, plastic))
        m.close()
    (a1, a2, pa), (b1, b2, pb) = out
    assert pa == pb and pa > 0.2
    assert relerr(a1, b1) <= 1e-13
    assert relerr(a2, b2) <= 1e-13
    assert relerr(a1, a2) > 1e-6


@pytest.mark.parametrize("system,fmt", [("GpuPCG", "auto"), ("GpuBlockPCG", "auto"), ("GpuBlockPCG", "sym")])
def test_pcg_solve_matches_direct(system, fmt):
    print(f"case: pcg {system} {fmt}", flush=True)
    mesh, (g, o) = cube_pair(5, system=system)
    g.spmv_config(fmt)
    for m in (g, o):
        m.form_tangent(values=False)
    rng = np.random.default_rng(3)
    b = rng.normal(size=g.neq)
    xg, xo = g.solve(b), o.solve(b)
    assert relerr(xg, xo) <= 1e-9
    assert relerr(g.spmv(xg), b) <= 1e-11


@pytest.mark.parametrize("fmt", ["auto", "sym"])
def test_brick_pushover_trajectory(fmt):
    """Reduced cube under top pressure, LoadControl + Newton: converged
    displacement and plastic state after every step."""
    print(f"case: brick pushover n=4 spmv {fmt}", flush=True)
    n = 4
    mesh, (g, o) = cube_pair(n)
    g.spmv_config(fmt)
    npts = 8 * n ** 3
    for m in (g, o):
        m.test("NormUnbalance", 1e-9, 30)
        m.integrator("LoadControl", 40.0)
    for step in range(8):
        for m in (g, o):
            assert m.analyze(1) == 0
        assert relerr(g.trial_disp(), o.trial_disp()) <= RTOL, step
        assert relerr(g.point_data("stress", npts), o.point_data("stress", npts)) <= RTOL
    assert (o.point_data("plastic", npts)[:, 6] > 0).any()


def test_quad_strip_displacement_control():
    """C0 workload at reduced size: plane-strain J2 strip, DisplacementControl
    on the free-end top node, 10 steps of 0.001."""
    print("case: quad strip 16x4 displacement control", flush=True)
    mesh = meshes.quad_strip(16, 4)
    res = []
    for m in (Model(2, 2), _oracle.oracle_model(2, 2)):
        meshes.build_quad_strip(m, mesh)
        m.load(mesh["tip"], 0.0, 1.0)
        m.system("GpuPCG", 1e-13, 20000)
        m.test("NormUnbalance", 1e-8, 25)
        m.integrator("DisplacementControl", mesh["tip"], 2, 0.001)
        m.setup()
        traj = []
        for step in range(10):
            assert m.analyze(1) == 0
            traj.append((m.trial_disp().copy(), m.load_factor))
        res.append(traj)
    for (ug, lg), (uo, lo) in zip(*res):
        assert relerr(ug, uo) <= RTOL
        assert abs(lg - lo) <= RTOL * abs(lo)


def _spmv_models():
    mesh = meshes.brick_cube(4)
    m = Model(3, 3)
    meshes.build_brick_cube(m, mesh, pressure=1.0)
    yield "brick", m
    mesh = meshes.quad_strip(12, 3)
    m = Model(2, 2)
    meshes.build_quad_strip(m, mesh)
    yield "quad", m
    fr = meshes.rc_frame_3d(2, 2, 3)
    conn, _ = meshes.frame_elements(fr)
    m = Model(3, 6)
    meshes.build_rc_frame_per_element(m, fr, meshes.default_theta(len(conn)))
    yield "frame3d", m


@pytest.mark.parametrize("lanes", [0, 4, 32])
def test_node_blocked_spmv_matches_csr(lanes):
    """The node-blocked column indices address the same entries in the same
    order as the CSR column indices: y = K x is bitwise the same."""
    for name, m in _spmv_models():
        print(f"case: spmv {name} lanes {lanes}", flush=True)
        m.setup()
        rng = np.random.default_rng(7)
        m.set_trial_disp(1e-4 * rng.normal(size=(m.num_nodes, m.ndf)))
        m.update()
        m.form_tangent(values=False)
        x = rng.normal(size=m.neq)
        m.spmv_config("csr", lanes)
        y_csr = m.spmv(x)
        m.spmv_config("auto", lanes)
        y_nb = m.spmv(x)
        assert np.array_equal(y_nb, y_csr)
        K = m.form_tangent()
        rp, ci = m.csr_pattern()
        rows = np.repeat(np.arange(m.neq), np.diff(rp))
        y_ref = np.zeros(m.neq)
        np.add.at(y_ref, rows, K * x[ci])
        assert relerr(y_nb, y_ref) <= 1e-13
        m.close()


@pytest.mark.parametrize("lanes", [0, 8, 64])
def test_symmetric_spmv_matches_csr(lanes):
    """The block-symmetric copy (upper node blocks, lower ones read
    transposed) gives K x to rounding, and follows a new assembly; where it
    does not apply (6 DOFs per node) the node-blocked product is used."""
    for name, m in _spmv_models():
        print(f"case: sym spmv {name} lanes {lanes}", flush=True)
        m.setup()
        rng = np.random.default_rng(9)
        m.spmv_config("sym", lanes)
        x = rng.normal(size=m.neq)
        rp, ci = m.csr_pattern()
        rows = np.repeat(np.arange(m.neq), np.diff(rp))
        for step in range(2):
            m.set_trial_disp((step + 1) * 1e-4 * rng.normal(size=(m.num_nodes, m.ndf)))
            m.update()
            K = m.form_tangent()
            y_ref = np.zeros(m.neq)
            np.add.at(y_ref, rows, K * x[ci])
            y = m.spmv(x)
            assert relerr(y, y_ref) <= 1e-13, (name, step)
        m.close()


def test_pcg_solve_csr_layout():
    print("case: pcg csr layout", flush=True)
    mesh, (g, o) = cube_pair(5, system="GpuBlockPCG")
    g.spmv_config("csr")
    for m in (g, o):
        m.form_tangent(values=False)
    b = np.random.default_rng(4).normal(size=g.neq)
    assert relerr(g.solve(b), o.solve(b)) <= 1e-9


def test_pcg_graph_replay_matches_eager_launches():
    """PCG chunks replayed from a captured graph, and the alpha / beta
    reductions fused into the vector kernels, give the same iterates, bit
    for bit, as the separate launches issued one by one and as another chunk
    length: a frame DisplacementControl pushover (two solution vectors per
    iteration, hence two graphs, with element updates between the replays)
    interleaved with direct solves into a third buffer."""
    print("case: pcg graph replay vs eager", flush=True)
    fr = meshes.rc_frame_2d(3, 2)
    conn, _ = meshes.frame_elements(fr)
    theta = meshes.default_theta(len(conn))
    runs = []
    for chunk, graph, fuse in ((16, True, True), (16, False, False), (10, True, True), (16, False, True),
                               (16, True, False)):
        m = Model(2, 3)
        meshes.build_rc_frame_per_element(m, fr, theta)
        m.system("GpuBlockPCG", 1e-12, 100000)
        m.cg_config(chunk, graph, fuse, small=False)
        P = np.zeros((len(fr["floor_nodes"]), 3))
        P[:, 0] = 1.0
        m.loads(fr["floor_nodes"], P)
        m.test("NormUnbalance", 1e-5, 40)
        m.integrator("DisplacementControl", fr["roof"], 1, 6.0)
        m.setup()
        b = np.random.default_rng(11).normal(size=m.neq)
        t = []
        for step in range(6):
            assert m.analyze(1) == 0
            t.append(m.trial_disp().copy())
            t.append(m.solve(b))
        t.append(np.array([m.counters()["cg_iters"]], dtype=float))
        runs.append(t)
        m.close()
    for other in runs[1:]:
        for a, c in zip(runs[0], other):
            assert np.array_equal(a, c)
    with pytest.raises(XaraError):
        Model(2, 3).cg_config(7, True)


@pytest.mark.parametrize("system", ["GpuPCG", "GpuBlockPCG"])
def test_single_workgroup_pcg_matches_launch_per_step(system):
    """The whole-solve kernels of small systems (one workgroup, one launch)
    against the kernel-per-step PCG: the same converged trajectories over a
    2D frame pushover (3 DOFs per node, half bandwidth 11) and quad strips
    of half bandwidths 13, 43 and 59 (the band factor's column-frame kernel
    up to 44, its shifting-window kernel above), all
    taken by the band-Cholesky-preconditioned solve (the tiled factor off),
    which then needs at most three iterations per solve; and over a 3x3x3 3D frame (half
    bandwidth 77 > 63, taken by the (block-)Jacobi one-workgroup solve),
    whose iteration counts agree within rounding's reach."""
    fr = meshes.rc_frame_2d(3, 2)
    conn, _ = meshes.frame_elements(fr)
    theta = meshes.default_theta(len(conn))
    strips = {"quad": (meshes.quad_strip(16, 4), 13), "quad19": (meshes.quad_strip(40, 19, ly=10.0), 43),
              "quad27": (meshes.quad_strip(40, 27, ly=14.0), 59)}
    fr3 = meshes.rc_frame_3d(3, 3, 3)
    for case in ("frame", "quad", "quad19", "quad27", "frame3d"):
        print(f"case: small pcg {system} {case}", flush=True)
        res = []
        for small in (True, False):
            if case == "frame":
                m = Model(2, 3)
                meshes.build_rc_frame_per_element(m, fr, theta)
                P = np.zeros((len(fr["floor_nodes"]), 3))
                P[:, 0] = 1.0
                m.loads(fr["floor_nodes"], P)
                node, dof, du, tol = fr["roof"], 1, 6.0, 1e-5
            elif case in strips:
                mesh = strips[case][0]
                m = Model(2, 2)
                meshes.build_quad_strip(m, mesh)
                m.load(mesh["tip"], 0.0, 1.0)
                node, dof, du, tol = mesh["tip"], 2, 0.001, 1e-8
            else:
                m = Model(3, 6)
                meshes.build_rc_frame_3d(m, fr3)
                node, dof, du, tol = fr3["roof"], 1, 6.0, 1e-5
            m.system(system, 1e-12, 100000)
            m.cg_config(16, True, True, small=small, wide=False)
            m.test("NormUnbalance", tol, 40)
            m.integrator("DisplacementControl", node, dof, du)
            m.setup()
            t = []
            for step in range(6):
                assert m.analyze(1) == 0
                t.append(m.trial_disp().copy())
            c = m.counters()
            if case in strips and small:
                assert c["band_bw"] == strips[case][1], c["band_bw"]
            assert m.preconditioner() == ("band" if small and case != "frame3d" else "jacobi")
            res.append((np.array(t), c["cg_iters"], c["solves"]))
            m.close()
        (a, ia, sa), (b, ib, sb) = res
        assert relerr(a, b) <= 1e-9
        if case == "frame3d":
            # the sums' order differs, and on an ill-conditioned frame rounding
            # moves the iteration at which a solve crosses its tolerance
            assert abs(ia - ib) <= 0.1 * ib
        else:
            assert ia <= 3 * sa and ib > 3 * sb


@pytest.mark.parametrize("case", ["brick", "frame3d"])
def test_pcg_warm_start_same_trajectory_fewer_iterations(case):
    """Warm starts of the chunked PCG (XG_CG_WARM: under LoadControl a step's
    first solve from the previous step's first solution, DisplacementControl's
    reference-load solves from the previous one) against starts from zero:
    the same converged trajectory to 1e-9 on a brick LoadControl pushover
    past first yield (with far fewer PCG iterations: the elastic steps' first
    solves start from the answer) and on a 3D RC frame DisplacementControl
    pushover (where only the reference-load solves start warm, a few percent
    of the iterations, within the spread that rounding gives the rest)."""
    print(f"case: warm start {case}", flush=True)
    res = []
    for warm in (True, False):
        if case == "brick":
            mesh = meshes.brick_cube(6)
            m = Model(3, 3)
            meshes.build_brick_cube(m, mesh, pressure=1.0)
            m.system("GpuBlockPCG", 1e-12, 20000)
            m.test("NormUnbalance", 1e-8, 30)
            m.integrator("LoadControl", 20.0)
            nsteps = 8
        else:
            fr = meshes.rc_frame_3d(3, 3, 4)
            m = Model(3, 6)
            meshes.build_rc_frame_3d(m, fr)
            m.system("GpuBlockPCG", 1e-12, 100000)
            m.test("NormUnbalance", 1e-5, 40)
            m.integrator("DisplacementControl", fr["roof"], 1, 8.0)
            nsteps = 6
        m.cg_config(16, True, True, small=False, warm=warm)
        m.setup()
        traj = []
        for _ in range(nsteps):
            assert m.analyze(1) == 0
            traj.append(m.trial_disp().copy())
        res.append((np.array(traj), m.counters()["cg_iters"]))
        m.close()
    (a, ia), (b, ib) = res
    assert relerr(a, b) <= 1e-9
    if case == "brick":
        assert ia < 0.5 * ib, (ia, ib)
    else:
        # the warm reference-load solves save a few percent; the rest of the
        # count moves with rounding by as much (with the section sums in
        # 16-lane rows: 4,596 warm against 4,393 cold)
        assert ia <= 1.1 * ib, (ia, ib)


def test_morton_sweep_order_matches_equation_order(monkeypatch):
    """XG_SYM_ORDER=1: the symmetric product's block rows stored and swept in
    the Morton order of their nodes, the chunked PCG in that order (b and x
    permuted at the ends of a solve, the block inverses once per matrix).
    Against the equation order: the product through xg_spmv to 1e-13 (each
    row sums the same entries in the same order, but of a pair of blocks the
    order keeps the other one, and the assembled K_IJ and K_JI^T differ in the
    last bits), a solve to 1e-9, the allocation-free solve bit for bit with the
    ordinary one, and a warm-started LoadControl pushover to 1e-9."""
    from xara_amd import _lib
    print("case: morton sweep order cube 8^3", flush=True)
    mesh = meshes.brick_cube(8)
    models = []
    for order in ("1", "0"):
        monkeypatch.setenv("XG_SYM_ORDER", order)
        m = Model(3, 3)
        meshes.build_brick_cube(m, mesh, pressure=1.0)
        m.system("GpuBlockPCG", 1e-12, 20000)
        m.cg_config(16, True, True, small=False)
        m.setup()
        models.append(m)
    monkeypatch.delenv("XG_SYM_ORDER")
    a, b = models
    rng = np.random.default_rng(11)
    U = random_field(mesh, 1e-3, 12)
    for m in models:
        m.set_trial_disp(U)
        m.update()
        m.form_tangent(values=False)
    x = rng.normal(size=a.neq)
    for m in models:
        m.spmv_config("sym")
    ya, yb = a.spmv(x), b.spmv(x)
    assert relerr(ya, yb) <= 1e-13
    assert np.abs(ya).max() > 0
    for m in models:
        m.spmv_config("auto")
    B = rng.normal(size=a.neq)
    Xa, Xb = a.solve(B), b.solve(B)
    assert relerr(Xa, Xb) <= 1e-9
    lib = _lib.load()
    X2 = np.zeros(a.neq)
    assert lib.solve_noalloc(a._h, B.ctypes.data_as(_lib.P_D), X2.ctypes.data_as(_lib.P_D)) == 0, lib.error()
    assert np.array_equal(Xa, X2)
    traj = []
    for m in models:
        m.revert_to_start()
        m.set_load_factor(0.0)
        m.test("NormUnbalance", 1e-8, 30)
        m.integrator("LoadControl", 25.0)
        t = []
        for _ in range(5):
            assert m.analyze(1) == 0
            t.append(m.trial_disp().copy())
        traj.append(np.array(t))
    assert relerr(traj[0], traj[1]) <= 1e-9
    for m in models:
        m.close()


def test_revert_to_start_and_to_last_commit():
    """Domain::revertToStart after a plastic trial gives back the fresh model
    (its closing update at zero displacement forms the elastic tangent,
    Domain.cpp:1941-1958); Domain::revertToLastCommit updates at the
    committed displacements (Domain.cpp:1925-1939).  GPU and oracle alike."""
    print("case: brick revert to start / to last commit", flush=True)
    n = 3
    mesh, (g, o) = cube_pair(n, system="GpuBlockPCG")
    npts = 8 * n ** 3
    D0 = o.point_data("tangent", npts).copy()
    U = np.zeros((len(mesh["crds"]), 3))
    U[:, 2] = -2.2e-3 * mesh["crds"][:, 2]
    for m in (g, o):
        m.set_trial_disp(U)
        m.update()
    assert (o.point_data("plastic", npts)[:, 6] > 0).all()
    for m in (g, o):
        m.revert_to_start()
    assert np.array_equal(o.point_data("tangent", npts), D0)
    for what in ("tangent", "stress", "plastic"):
        assert relerr(g.point_data(what, npts), o.point_data(what, npts)) <= RTOL, what
    assert relerr(g.form_tangent(), o.form_tangent()) <= RTOL
    # commit a plastic state, try a larger trial, revert to the commit
    for m in (g, o):
        m.set_trial_disp(U)
        m.update()
        m.commit()
        m.set_trial_disp(2 * U)
        m.update()
        m.revert()
    for what in ("stress", "tangent", "plastic"):
        assert relerr(g.point_data(what, npts), o.point_data(what, npts)) <= RTOL, what
    assert relerr(g.form_unbalance(), o.form_unbalance()) <= RTOL


def _pcg_iterations(K, b, blocks, rtol):
    """PCG iteration count of the GPU solver's recurrence (x0 = 0, stop when
    r.r <= rtol^2 b.b) with an exact block-Jacobi preconditioner."""
    Minv = np.zeros_like(K)
    for eqs in blocks:
        Minv[np.ix_(eqs, eqs)] = np.linalg.inv(K[np.ix_(eqs, eqs)])
    x, r = np.zeros_like(b), b.copy()
    z = Minv @ r
    p, rz, bb = z.copy(), r @ z, b @ b
    for it in range(1, 10 * len(b)):
        q = K @ p
        alpha = rz / (p @ q)
        x += alpha * p
        r -= alpha * q
        z = Minv @ r
        rz_new = r @ z
        if r @ r <= rtol * rtol * bb:
            return it
        p = z + (rz_new / rz) * p
        rz = rz_new
    return -1


@pytest.mark.parametrize("system", ["GpuPCG", "GpuBlockPCG"])
def test_block_jacobi_with_partly_fixed_nodes(system):
    """Roller base (z fixed, x and y free) plus two pinned corners: nodal
    blocks of 3 and of 2 free DOFs.  The GPU PCG takes the iterations of an
    exact (block-)Jacobi PCG run in numpy on the same matrix, and both
    preconditioners give the direct solution."""
    print(f"case: partly fixed nodes {system}", flush=True)
    n = 4
    mesh = meshes.brick_cube(n)
    base = mesh["fixed_nodes"]
    flags = np.zeros((len(base), 3), np.int32)
    flags[:, 2] = 1
    flags[0, :] = 1
    flags[-1, :] = 1
    rtol = 1e-10
    g, o = Model(3, 3), _oracle.oracle_model(3, 3)
    for m in (g, o):
        meshes.build_brick_cube(m, dict(mesh, fixed_nodes=base[:0]), pressure=1.0)
        m.fix_many(base, flags)
        m.system(system, rtol, 20000)
        m.setup()
        m.form_tangent(values=False)
    K = np.zeros((g.neq, g.neq))
    rp, ci = g.csr_pattern()
    K[np.repeat(np.arange(g.neq), np.diff(rp)), ci] = g.form_tangent()
    eqs = g.node_eqns()
    if system == "GpuBlockPCG":
        blocks = [row[row >= 0] for row in eqs if (row >= 0).any()]
        assert {len(bl) for bl in blocks} == {2, 3}
    else:
        blocks = [[a] for a in range(g.neq)]
    b = np.random.default_rng(5).normal(size=g.neq)
    c0 = g.counters()["cg_iters"]
    x = g.solve(b)
    its = g.counters()["cg_iters"] - c0
    ref = _pcg_iterations(K, b, blocks, rtol)
    assert abs(its - ref) <= 2, (its, ref)
    assert relerr(x, o.solve(b)) <= 1e-9


def test_band_factor_kept_for_an_unchanged_matrix(monkeypatch):
    """The 64 x 16 FourNodeQuad strip stays elastic through a
    DisplacementControl pushover, so every tangent after the first equals
    the first bit for bit: its band factor is kept (counted in band_reuses)
    instead of formed again, and the trajectory equals, bit for bit, the one
    with every matrix factored (XG_PC_REUSE=0)."""
    print("case: band factor reuse on the elastic quad strip", flush=True)
    mesh = meshes.quad_strip(64, 16)
    runs = []
    for reuse in ("1", "0"):
        monkeypatch.setenv("XG_PC_REUSE", reuse)
        m = Model(2, 2)
        meshes.build_quad_strip(m, mesh)
        m.load(mesh["tip"], 0.0, 1.0)
        m.system("GpuBlockPCG", 1e-14, 100000)
        m.test("NormUnbalance", 1e-8, 25)
        m.integrator("DisplacementControl", mesh["tip"], 2, 0.001)
        m.setup()
        traj = []
        for k in range(8):
            assert m.analyze(1) == 0, k
            traj.append((m.trial_disp().copy(), m.load_factor))
        c = m.counters()
        runs.append((traj, c))
        m.close()
    (ta, ca), (tb, cb) = runs
    assert ca["band_bw"] > 0 and ca["band_reuses"] > 0 and cb["band_reuses"] == 0, (ca, cb)
    for (ua, la), (ub, lb) in zip(ta, tb):
        assert np.array_equal(ua, ub) and la == lb
