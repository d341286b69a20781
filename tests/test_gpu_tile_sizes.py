"""H tiles of 32 x 64 and 64 x 64 of the FP64 path from a system, for one k-point
and for several, and the tiles of the contraction of given coefficients over many
tile rows: every tile gives the bits of the others.  An element depends on its two
plane waves alone, so small calls (tiles of 16 x 32 and 32 x 32) are the
reference, and the oracle for one of them.

On 256 CUs a call takes 32 x 64 tiles where it has 768 to 1535 lower tiles of
64 x 64 (one k-point: 2433 to 3456 plane waves), 64 x 64 from there on.

Tolerance as in test_gpu_parity.py: relative Frobenius error of the lower
triangle <= 1e-13."""
import numpy as np
import pytest

from hybridhsdla_amd import tiny_system
from hybridhsdla_amd.system import KPoint
from oracle import pyoracle as po
from tests.helpers import rel_fro_lower

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

TOL = 1e-13


def _subset(kp, idx):
    return KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[np.asarray(idx, dtype=np.int64)]), kmax=kp.kmax)


def _system(natoms, lmax, ng):
    s, kp = tiny_system(natoms=natoms, lmax=lmax, a_cell=17.0, ng_target=ng + 60, seed=18, rotate=True)
    assert kp.ng >= ng
    return s, kp


def _lower64(ng):
    n = (ng + 63) // 64
    return n * (n + 1) // 2


def _check_subsets(ctx, h, s, kp, H, S, sizes):
    for m in sizes:
        idx = np.sort(np.random.default_rng(m).permutation(kp.ng)[:m])
        Hs, Ss = ctx.create_HS2(h, _subset(kp, idx))
        assert np.array_equal(Hs, H[np.ix_(idx, idx)]) and np.array_equal(Ss, S[np.ix_(idx, idx)]), m
    Hr, Sr = po.reference_hs(s, _subset(kp, idx))
    assert rel_fro_lower(Hs, Hr) <= TOL and rel_fro_lower(Ss, Sr) <= TOL


# 2433 and 3456: the first and last of 32 x 64 tiles; 3457: the first of 64 x 64;
# (0, 1): atoms of one k-step, several of which end in a stage
@pytest.mark.parametrize("ng,lmax,natoms", [(2433, (3, 5, 2), 6), (2803, (0, 1), 5), (2803, (4, 3), 4),
                                            (3456, (2, 3), 3), (3457, (0, 2, 3), 5)])
def test_one_k_point(ctx, ng, lmax, natoms):
    s, kp = _system(natoms, lmax, ng)
    kp = _subset(kp, np.arange(ng))
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    print(f"ng {ng}: {_lower64(ng) / n_cu:.2f} tiles of 64 x 64 per CU", flush=True)
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, kp)
    _check_subsets(ctx, h, s, kp, H, S, (1409, 500, 60))
    h.close()


@pytest.mark.parametrize("ngs", [(1900, 1500, 1100), (1100, 2803, 65, 1, 1900)])
def test_several_k_points(ctx, ngs):
    """32 x 64 tiles (936 of 64 x 64), 64 x 64 tiles (1630); each replayed."""
    s, kp = _system(5, (3, 0, 4), 2803)
    rng = np.random.default_rng(9)
    kps = [KPoint(k=kp.k + 0.01 * i, g=np.ascontiguousarray(kp.g[np.sort(rng.permutation(kp.ng)[:n])]), kmax=kp.kmax)
           for i, n in enumerate(ngs)]
    n_cu = torch.cuda.get_device_properties(0).multi_processor_count
    print(f"{ngs}: {sum(map(_lower64, ngs)) / n_cu:.2f} tiles of 64 x 64 per CU", flush=True)
    h = ctx.upload(s)
    for _ in range(2):
        res, _ = ctx.create_HS2_batched(h, kps)
        for (H, S), k in zip(res, kps):
            m = min(k.ng, 300)
            idx = np.sort(np.random.default_rng(k.ng).permutation(k.ng)[:m])
            Hs, Ss = ctx.create_HS2(h, _subset(k, idx))
            assert np.array_equal(Hs, H[np.ix_(idx, idx)]) and np.array_equal(Ss, S[np.ix_(idx, idx)]), k.ng
    h.close()


@pytest.mark.parametrize("pipelined,staged", [(9, 8), (10, 2), (11, 8), (12, 3), (13, 4), (14, 4)])
def test_contraction_pipelined_and_staged(ctx, pipelined, staged):
    """The LDS-DMA pipelined products and the register-staged ones of the same
    tile, from given coefficients: the same bits over several tiles and a depth
    of many stages, for the T application and the contraction."""
    s, kp = tiny_system(natoms=4, lmax=(4, 3, 5, 2), ng_target=700, seed=21)
    A, B = po.construct_ab(s, kp)
    args = (s.L, s.natoms, kp.ng, A, B, s.taa, s.tab, s.tbb, s.lmax, s.max_lmax, s.sqrt_u_norms())
    H1, S1 = ctx.create_HS2_stripped_v2(*args, tile=staged)
    H2, S2 = ctx.create_HS2_stripped_v2(*args, tile=pipelined)
    assert np.array_equal(H1, H2) and np.array_equal(S1, S2)
    Hr, Sr = po.reference_hs(s, kp)
    assert rel_fro_lower(H2, Hr) <= TOL and rel_fro_lower(S2, Sr) <= TOL
