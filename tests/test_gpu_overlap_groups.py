"""Which atoms share a Legendre sum of S: in a long cell the metric's entries
differ by orders of magnitude, and each counts on its own scale.

Tolerance as in test_gpu_parity.py: relative Frobenius error <= 1e-13."""
import numpy as np
import pytest

from hybridhsdla_amd import tiny_system
from hybridhsdla_amd.system import KPoint
from oracle import pyoracle as po
from tests.helpers import rel_fro_lower

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 2])
def test_long_cell(ctx, axis):
    """Axes of 6, 6 and 60000 bohr; the second atom's matrix differs in one axis
    by 1e-8 of that axis' own length, which on the long axis is 1e-16 of the
    metric's largest entry.  Plane waves along the long axis, where that length
    decides the cosines.  The atoms lie in the plane z = 0, so the phases of large
    K are exact."""
    s, kp = tiny_system(natoms=2, lmax=(5,), a_cell=6.0, seed=4)
    b = 2 * np.pi / 6.0 * np.array([1.0, 1.0, 1e-4])
    s.bmat = np.diag(b).reshape(-1, order="F").copy()
    s.omega = 36.0 * 6e4
    s.pos[:, 2] = 0.0
    for a in range(2):
        m = np.diag(b)
        m[axis, axis] *= 1.0 + 1e-8 * a
        s.rotmat[a] = m.reshape(-1, order="F")
    rng = np.random.default_rng(2)
    g = np.stack([rng.integers(-1, 2, 120), rng.integers(-1, 2, 120), rng.integers(-8000, 8000, 120)], axis=1)
    g = np.unique(g, axis=0).astype(np.int32)
    sub = KPoint(k=np.array([0.1, 0.2, 0.3]), g=np.ascontiguousarray(g), kmax=10.0)
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, sub)
    Hr, Sr = po.reference_hs(s, sub)
    print(f"axis {axis}: H {rel_fro_lower(H, Hr):.2e} S {rel_fro_lower(S, Sr):.2e}", flush=True)
    assert rel_fro_lower(H, Hr) <= 1e-13 and rel_fro_lower(S, Sr) <= 1e-13
    h.close()
