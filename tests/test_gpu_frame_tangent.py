"""GPU parity of the 3D frame tangent (16 lanes per element, 16 elements per
workgroup) against the oracle: element counts that fill a workgroup, leave
one part empty and need several."""
import numpy as np
import pytest

from tests import _oracle
from xara_amd import meshes
from xara_amd.model import Model

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("size", [(1, 1, 1), (1, 1, 2), (2, 1, 1), (2, 1, 3), (3, 2, 4)], ids=str)
def test_frame_tangent_3d(size):
    print(f"case: 3D frame tangent {size}", flush=True)
    fr = meshes.rc_frame_3d(*size)
    g, o = Model(3, 6), _oracle.oracle_model(3, 6)
    for m in (g, o):
        meshes.build_rc_frame_3d(m, fr)
        m.setup()
    U = np.random.default_rng(4).normal(0, 1e-2, (len(fr["crds"]), 6))
    U[:, 3:] *= 1e-4
    # unstrained: the same section stiffnesses; an entry sums at most 8
    # elements of 5 sections, each a product of three matrices: 100 roundings
    # of the largest entry at most.  Strained: fiber states to the parity bar.
    for disp, tol in ((0 * U, 100 * EPS), (U, 1e-9)):
        K = []
        for m in (g, o):
            m.set_trial_disp(disp)
            m.update()
            K.append(m.form_tangent())
        assert np.max(np.abs(K[0] - K[1])) <= tol * np.max(np.abs(K[1]))
