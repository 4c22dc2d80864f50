"""GPU parity of the nodal block inverses (k_block_inverse): the PCG that they
precondition against the same iteration in numpy with numpy's inverses.  Node
blocks of every size up to the DOFs per node, node counts that leave the
last workgroup part empty, rows longer than one sweep of the search."""
import numpy as np
import pytest

from xara_amd import meshes
from xara_amd.model import Model

pytestmark = pytest.mark.gpu


def pcg(A, blocks, b, rtol):
    def precond(r):
        z = np.zeros_like(r)
        for e, Bi in blocks:
            z[e] = Bi @ r[e]
        return z

    x, r = np.zeros_like(b), b.copy()
    z = precond(r)
    p, rz, it = z.copy(), r @ z, 0
    while it < 10000:
        q = A @ p
        alpha = rz / (p @ q)
        x, r, it = x + alpha * p, r - alpha * q, it + 1
        if np.linalg.norm(r) <= rtol * np.linalg.norm(b):
            break
        z = precond(r)
        rzn = r @ z
        p, rz = z + rzn / rz * p, rzn
    return x, it


# small: the solve in one workgroup, which a band narrower than 64 would take
# to the band factor instead
@pytest.mark.parametrize("case, small", [(("quad", 7, 6), False), (("brick", 4), False), (("brick", 4), True),
                                         (("frame2", 5, 3), False), (("frame3", 3, 2, 3), False)])
def test_block_jacobi_iterations_match_numpy(case, small):
    print(f"case: block inverse {case} small={small}", flush=True)
    kind, *size = case
    rng = np.random.default_rng(3)
    if kind == "quad":
        mesh = meshes.quad_strip(*size)
        m, n = Model(2, 2), len(mesh["crds"])
        meshes.build_quad_strip(m, mesh)
    elif kind == "brick":
        mesh = meshes.brick_cube(size[0])
        m, n = Model(3, 3), len(mesh["crds"])
        meshes.build_brick_cube(m, mesh)
    elif kind == "frame2":
        mesh = meshes.rc_frame_2d(*size)
        m, n = Model(2, 3), len(mesh["crds"])
        conn, _ = meshes.frame_elements(mesh)
        meshes.build_rc_frame_per_element(m, mesh, meshes.default_theta(len(conn)))
    else:
        mesh = meshes.rc_frame_3d(*size)
        m, n = Model(3, 6), len(mesh["crds"])
        meshes.build_rc_frame_3d(m, mesh)
    ndf = {"quad": 2, "brick": 3, "frame2": 3, "frame3": 6}[kind]
    for tag in range(n - 6, n):  # blocks of every size among the last nodes
        m.fix(tag, *(int(v) for v in rng.integers(0, 2, ndf)))
    m.system("GpuBlockPCG", 1e-8, 10000)
    m.cg_config(16, True, True, small=small, wide=False)
    m.setup()
    m.set_trial_disp(np.zeros((n, ndf)))
    m.update()
    vals = m.form_tangent()
    rp, ci = m.csr_pattern()
    A = np.zeros((m.neq, m.neq))
    A[np.repeat(np.arange(m.neq), np.diff(rp)), ci] = vals
    eq = np.asarray(m.node_eqns()).reshape(-1, ndf)
    sets = [e[e >= 0] for e in eq]
    assert len({len(e) for e in sets}) > ndf // 2
    blocks = [(e, np.linalg.inv(A[np.ix_(e, e)])) for e in sets if len(e)]
    b = rng.normal(size=m.neq)
    x, it = pcg(A, blocks, b, 1e-8)
    c0 = m.counters()
    X = m.solve(b)
    c1 = m.counters()
    assert not small or c1["band_bw"] < 0
    # rounding moves the residual of a converging iteration by a few per cent
    # of itself at most: the same count to one in twenty
    assert abs((c1["cg_iters"] - c0["cg_iters"]) - it) <= 1 + it // 20
    # both stop at |r| <= 1e-8 |b|: solutions apart by that times 2 |A^-1|
    Ai = np.linalg.norm(np.linalg.inv(A), 2)
    assert np.linalg.norm(X - x) <= 2e-8 * Ai * np.linalg.norm(b)
    m.close()
