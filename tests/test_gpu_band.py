"""GPU parity of the one-workgroup band factor and its PCG (k_band_gather,
k_band_factor_w, k_band_factor, k_pcg_band) against the CPU oracle's direct
solve at half bandwidths on either side of every kernel variant's limit (15,
23, 31, 39 and 44 columns, the shifting window above; sweeps in groups of 16
up to 48), with the tiled factor off so that the band factor takes them all;
and the allocation-free solve, whose factor lies in memory that holds
another solve's values, bit for bit."""
import numpy as np
import pytest

from tests import _oracle
from xara_amd import _lib, meshes
from xara_amd.model import Model

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


def noalloc(m, B):
    X = np.zeros(m.neq)
    assert m._b.solve_noalloc(m._h, B.ctypes.data_as(_lib.P_D), X.ctypes.data_as(_lib.P_D)) == 0
    return X


# (elements along and across the strip, half bandwidth 2 ny + 5)
STRIPS = [(33, 1, 7), (13, 5, 15), (21, 6, 17), (23, 9, 23), (25, 10, 25), (27, 13, 31), (29, 14, 33), (35, 17, 39),
          (37, 18, 41), (39, 19, 43), (41, 20, 45), (43, 21, 47), (45, 22, 49), (59, 29, 63)]


@pytest.mark.parametrize("nx,ny,bw", STRIPS)
def test_band_solve_matches_oracle(nx, ny, bw):
    print(f"case: band solve {nx} x {ny}, half bandwidth {bw}", flush=True)
    mesh = meshes.quad_strip(nx, ny, ly=8.0)
    U = np.random.default_rng(2).normal(0, 1e-3, mesh["crds"].shape)
    g, o = Model(2, 2), _oracle.oracle_model(2, 2)
    for m in (g, o):
        meshes.build_quad_strip(m, mesh)
        m.system("GpuBlockPCG", 1e-13, 1000)
        if m is g:
            m.cg_config(wide=False)
        m.setup()
        m.set_trial_disp(U)
        m.update()
        m.form_tangent(values=False)
    assert g.preconditioner() == "band" and g.counters()["band_bw"] == bw
    # leave another system's values in the memory of the allocation-free solve
    other = Model(3, 3)
    meshes.build_brick_cube(other, meshes.brick_cube(12))
    other.setup()
    other.form_tangent(values=False)
    noalloc(other, np.random.default_rng(5).normal(size=other.neq))
    other.close()
    # residual: the iteration's own stop test (1e-13 |b|) and the rounding of
    # the product it is formed with, eps sum |A| |x| per row; solutions to
    # the condition number times the rounding, below the parity bar of 1e-9
    rp, ci = o.csr_pattern()
    absA = np.abs(o.form_tangent())
    row = np.repeat(np.arange(o.neq), np.diff(rp))
    for seed in range(2):
        B = np.random.default_rng(seed).normal(size=g.neq)
        c0 = g.counters()
        X = g.solve(B)
        assert g.counters()["cg_iters"] - c0["cg_iters"] <= 2
        noise = np.bincount(row, absA * np.abs(X)[ci], o.neq)
        assert np.linalg.norm(o.spmv(X) - B) <= 1e-13 * np.linalg.norm(B) + 4 * EPS * np.linalg.norm(noise)
        assert relerr(X, o.solve(B)) <= 1e-9
        assert np.array_equal(X, noalloc(g, B))
    for m in (g, o):
        m.close()
