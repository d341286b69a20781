"""FP64 H and S from a system: coefficients as a phase times real vectors that
atoms of one kind share, S by the addition theorem.  Against the oracle at the
edges of its tiles (16, 32, 64 plane waves), of its k-step and stage depths
(2 (lmax+1)^2 against multiples of 4 and 16) and of its atom chunks, and tile
against tile: an element depends on its two plane waves alone, so every size
gives the same bits.

Tolerance as in test_gpu_parity.py: relative Frobenius error of the lower
triangle <= 1e-13."""
import numpy as np
import pytest

from hybridhsdla_amd import make_config, tiny_system
from hybridhsdla_amd.system import KPoint
from oracle import pyoracle as po
from tests.helpers import rel_fro_lower

pytestmark = pytest.mark.gpu

TOL = 1e-13


def _subset(kp, idx):
    return KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[np.asarray(idx, dtype=np.int64)]), kmax=kp.kmax)


def _check(ctx, s, kp):
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, kp)
    Hr, Sr = po.reference_hs(s, kp)
    # scaled by the largest element: the squares of the norm test's 1e200 overflow
    eh, es = (rel_fro_lower(X / np.abs(R).max(), R / np.abs(R).max()) for X, R in ((H, Hr), (S, Sr)))
    print(f"ng {kp.ng} lmax {list(s.lmax)[:6]}: H {eh:.2e} S {es:.2e}", flush=True)
    assert eh <= TOL and es <= TOL
    h.close()
    return H, S


@pytest.mark.parametrize("lmax", [(1,), (0, 1), (2, 1, 0), (3,), (5, 4), (8, 7)])
@pytest.mark.parametrize("natoms", [1, 9, 17])
def test_depths_and_atom_counts(ctx, lmax, natoms):
    """Depths of one k-step (lmax 0) to many stages, one atom, and more atoms
    of a kind than a chunk of phases holds."""
    if max(lmax) < 1 or (natoms < len(lmax) and max(lmax[:natoms]) < 1):
        pytest.skip("max_lmax 0 is refused")
    s, kp = tiny_system(natoms=natoms, lmax=lmax, a_cell=9.0, ng_target=90, seed=31)
    if s.lmax.max() < 1:
        pytest.skip("max_lmax 0 is refused")
    _check(ctx, s, kp)


def test_every_size_gives_the_same_bits(ctx):
    """Tiles of 16, 32 and 64 and the patch orders: principal submatrices of a
    1500-plane-wave call equal calls on subsets bit for bit."""
    s, kps = make_config(1, ng=1500, natoms=6)
    kp = kps[0]
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, kp)
    rng = np.random.default_rng(3)
    for n in (1, 15, 17, 31, 33, 63, 65, 480, 1023, 1409):
        idx = np.sort(rng.permutation(kp.ng)[:n])
        Hs, Ss = ctx.create_HS2(h, _subset(kp, idx))
        assert np.array_equal(Hs, H[np.ix_(idx, idx)]) and np.array_equal(Ss, S[np.ix_(idx, idx)]), n
    idx = np.sort(rng.permutation(kp.ng)[:70])
    Hr, Sr = po.reference_hs(s, _subset(kp, idx))
    assert rel_fro_lower(H[np.ix_(idx, idx)], Hr) <= TOL and rel_fro_lower(S[np.ix_(idx, idx)], Sr) <= TOL
    h.close()


def test_larger_triangle_with_patches(ctx):
    """Tiles of 64 in patches of 4 x 4 (25 tile rows and more)."""
    s, kp = tiny_system(natoms=2, lmax=(3, 2), a_cell=14.0, ng_target=1700, seed=8)
    _check(ctx, s, kp)


def test_opposite_and_equal_directions(ctx):
    """G and -G at the Gamma point: parallel, antiparallel and zero vectors."""
    s, kp = tiny_system(natoms=3, lmax=(6, 5), kpt=(0.0, 0.0, 0.0), ng_target=120, seed=12)
    assert np.any(np.all(kp.g == 0, axis=1))
    _check(ctx, s, kp)


@pytest.mark.parametrize("norm", [0.0, 1e-200, 1e200])
def test_norms_outside_folding(ctx, norm):
    """Norms that cannot be folded into the general operands need no other
    form here (the overlap weights carry them)."""
    s, kp = tiny_system(natoms=3, lmax=(3, 2, 4), ng_target=100, seed=9)
    s.match[1, 1, 4] = norm
    _check(ctx, s, kp)


def test_one_of_the_two_matrices(ctx):
    from hybridhsdla_amd.api import HSGEN_SKIP_H, HSGEN_SKIP_S
    s, kp = tiny_system(natoms=3, lmax=(3, 2, 4), ng_target=150, seed=5)
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, kp)
    H1, S1 = ctx.create_HS2(h, kp, flags=HSGEN_SKIP_S)
    H2, S2 = ctx.create_HS2(h, kp, flags=HSGEN_SKIP_H)
    assert np.array_equal(H, H1) and not S1.any() and np.array_equal(S, S2) and not H2.any()
    h.close()


@pytest.mark.parametrize("ng", [65, 129, 300])
def test_general_contraction_tiles_give_the_same_bits(ctx, ng):
    """The contraction of given coefficients keeps its tile configurations:
    every one gives the bits of the default."""
    s, kp = tiny_system(natoms=3, lmax=(3, 5, 2), ng_target=300, seed=6)
    sub = _subset(kp, np.arange(min(ng, kp.ng)))
    A, B = po.construct_ab(s, sub)
    args = (s.L, s.natoms, sub.ng, A, B, s.taa, s.tab, s.tbb, s.lmax, s.max_lmax, s.sqrt_u_norms())
    H0, S0 = ctx.create_HS2_stripped_v2(*args)
    Hr, Sr = po.reference_hs(s, sub)
    assert rel_fro_lower(H0, Hr) <= TOL and rel_fro_lower(S0, Sr) <= TOL
    for tile in range(1, 15):
        H, S = ctx.create_HS2_stripped_v2(*args, tile=tile)
        assert np.array_equal(H, H0) and np.array_equal(S, S0), tile


def _hexagonal(seed, natoms, turn):
    """A hexagonal cell whose atoms, of two types, carry rotations by multiples
    of 60 degrees (equal cosines up to rounding) or, with another kind of turn,
    matrices that change the cosines."""
    s, kp = tiny_system(natoms=natoms, lmax=(6, 4), a_cell=8.0, ng_target=150, seed=seed)
    a1, a3 = 8.0, 9.0
    amat = np.array([[a1, -a1 / 2, 0.0], [0.0, a1 * np.sqrt(3) / 2, 0.0], [0.0, 0.0, a3]])
    b33 = 2 * np.pi * np.linalg.inv(amat).T
    s.bmat = np.asfortranarray(b33).reshape(-1, order="F").copy()
    s.omega = float(np.linalg.det(amat))
    for a in range(natoms):
        c, sn = np.cos(a * np.pi / 3), np.sin(a * np.pi / 3)
        r = np.array([[c, -sn, 0.0], [sn, c, 0.0], [0.0, 0.0, 1.0]])
        if turn == "sheared":
            r = r + 0.05 * a * np.array([[0.0, 1.0, 0.0], [0.0, 0.0, 1.0], [0.0, 0.0, 0.0]])
        s.rotmat[a] = (r @ b33).reshape(-1, order="F")
    return s, kp


@pytest.mark.parametrize("turn", ["rotated", "sheared"])
@pytest.mark.parametrize("natoms", [3, 12])
def test_rotations_with_equal_and_other_cosines(ctx, natoms, turn):
    """Atoms that differ in their rotations alone share one Legendre sum where
    the rotations leave the cosines between plane waves as they are."""
    s, kp = _hexagonal(40, natoms, turn)
    _check(ctx, s, kp)


@pytest.mark.parametrize("norm", [None, 0.0])
def test_split_precision_column_chunks(ctx, monkeypatch, norm):
    """W of split precision comes from the real vectors in column chunks: 64
    columns at a time give the bits of one chunk, folded or not, for one
    k-point and for several (whose padding columns the chunks cut)."""
    from hybridhsdla_amd.api import HSGEN_PREC_OZAKI_INT8
    s, kp = tiny_system(natoms=5, lmax=(3, 2, 4), ng_target=300, seed=9, rotate=True)
    if norm is not None:
        s.match[1, 1, 4] = norm
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, kp, precision=HSGEN_PREC_OZAKI_INT8, slices=13)
    Hr, Sr = po.reference_hs(s, kp)
    assert rel_fro_lower(H, Hr) <= 1e-12 and rel_fro_lower(S, Sr) <= 1e-12
    sub = _subset(kp, np.arange(0, kp.ng, 2))
    Hs, Ss = ctx.create_HS2(h, sub, precision=HSGEN_PREC_OZAKI_INT8, slices=13)
    monkeypatch.setenv("HSGEN_BATCH_BYTES", "1")
    H1, S1 = ctx.create_HS2(h, kp, precision=HSGEN_PREC_OZAKI_INT8, slices=13)
    assert np.array_equal(H, H1) and np.array_equal(S, S1)
    monkeypatch.setenv("HSGEN_BATCH_BYTES", "60000000")
    res, _ = ctx.create_HS2_batched(h, [kp, sub], precision=HSGEN_PREC_OZAKI_INT8, slices=13)
    for (Hb, Sb), (Ha, Sa) in zip(res, ((H, S), (Hs, Ss))):
        assert np.array_equal(Hb, Ha) and np.array_equal(Sb, Sa)
    h.close()


@pytest.mark.parametrize("ng,nk,tile", [(1900, 1, 14), (1200, 2, 14), (1900, 2, 15), (3000, 1, 51), (3500, 1, 15)])
def test_int8_tiles_by_rounds(ctx, ng, nk, tile):
    """INT8 tiles by whole rounds of one per CU: 128 x 128 where they make one,
    128 x 256 where they save rounds; the bits of the 256 x 192 tiles."""
    from hybridhsdla_amd.api import HSGEN_PREC_OZAKI_INT8
    s, kps = make_config(1, ng=ng, natoms=2)
    kps = [kps[0], _subset(kps[0], np.arange(kps[0].ng - 5))][:nk]
    h = ctx.upload(s)
    res, reps = ctx.create_HS2_batched(h, kps, precision=HSGEN_PREC_OZAKI_INT8, slices=12)
    ref, _ = ctx.create_HS2_batched(h, kps, precision=HSGEN_PREC_OZAKI_INT8, slices=12, tile=51)
    print(f"ng {kps[0].ng} x {nk}: tile {reps[0]['tile_used']}", flush=True)
    assert reps[0]["tile_used"] == tile
    for (Ha, Sa), (Hb, Sb) in zip(res, ref):
        assert np.array_equal(Ha, Hb) and np.array_equal(Sa, Sb)
    h.close()


@pytest.mark.parametrize("ng", [4095, 4096, 4097])
def test_short_and_long_g_lists(ctx, ng):
    """G lists of up to 4096 plane waves are read from pinned memory, longer
    ones copied: both end in the bits of a small call."""
    s, kp = tiny_system(natoms=1, lmax=(2,), a_cell=19.0, ng_target=4600, seed=14)
    assert kp.ng > ng
    h = ctx.upload(s)
    H, S = ctx.create_HS2(h, _subset(kp, np.arange(ng)))
    idx = np.r_[0:20, ng // 2:ng // 2 + 20, ng - 20:ng]
    Hs, Ss = ctx.create_HS2(h, _subset(kp, idx))
    assert np.array_equal(Hs, H[np.ix_(idx, idx)]) and np.array_equal(Ss, S[np.ix_(idx, idx)])
    h.close()


@pytest.mark.parametrize("lmax", [(1,), (2,), (4,), (9, 3)])
@pytest.mark.parametrize("ng", [33, 300, 1100])
def test_h_and_s_in_one_launch(ctx, ng, lmax):
    """H and S tiles of one launch equal those of two, and the parts of the
    reported time are there for every choice of matrices."""
    from hybridhsdla_amd.api import HSGEN_FILL_UPPER, HSGEN_SKIP_H, HSGEN_SKIP_S
    torch = pytest.importorskip("torch")
    s, kp = tiny_system(natoms=5, lmax=lmax, a_cell=13.0, ng_target=1300, seed=4)
    sub = _subset(kp, np.arange(min(ng, kp.ng)))
    h = ctx.upload(s)
    n = sub.ng
    out = {}
    for flags in (0, HSGEN_SKIP_H, HSGEN_SKIP_S, HSGEN_FILL_UPPER, HSGEN_SKIP_H | HSGEN_SKIP_S):
        H, S = (torch.zeros(n, n, dtype=torch.complex128, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        r = ctx.create_hs_device(h, sub, H.data_ptr(), S.data_ptr(), n, flags=flags)
        out[flags] = [X.cpu().numpy().T for X in (H, S)]
        assert r["ms_total"] > 0 and r["ms_abgen"] >= 0 and r["ms_tmul"] >= 0 and r["ms_contract"] >= 0
        assert r["ms_abgen"] + r["ms_tmul"] + r["ms_contract"] <= r["ms_total"] * (1 + 1e-6) + 1e-2
        assert (r["ms_tmul"] > 0) == (not flags & HSGEN_SKIP_H)
    H, S = out[0]
    assert np.array_equal(out[HSGEN_SKIP_S][0], H) and np.array_equal(out[HSGEN_SKIP_H][1], S)
    for X, F in zip((H, S), out[HSGEN_FILL_UPPER]):
        assert np.array_equal(np.tril(F), np.tril(X)) and np.array_equal(F, np.tril(F) + np.tril(F, -1).conj().T)
    assert rel_fro_lower(H, po.reference_hs(s, sub)[0]) <= TOL
    h.close()


@pytest.mark.parametrize("lmax,natoms", [((16, 3), 10), ((24,), 1), ((15, 16), 9)])
def test_more_than_sixteen_l_and_all_s_tiles(ctx, lmax, natoms):
    """Radial factors in two planes of 16 values of l, groups of more atoms than
    are staged at a time, S tiles of 16, 32 and 64."""
    s, kp = tiny_system(natoms=natoms, lmax=lmax, a_cell=19.0, ng_target=4300, seed=3)
    h = ctx.upload(s)
    n = 4200
    H, S = ctx.create_HS2(h, _subset(kp, np.arange(n)))
    for m in (40, 900):
        idx = np.sort(np.random.default_rng(m).permutation(n)[:m])
        Hs, Ss = ctx.create_HS2(h, _subset(kp, idx))
        assert np.array_equal(Hs, H[np.ix_(idx, idx)]) and np.array_equal(Ss, S[np.ix_(idx, idx)]), m
        if m == 40:
            Hr, Sr = po.reference_hs(s, _subset(kp, idx))
            assert rel_fro_lower(Hs, Hr) <= TOL and rel_fro_lower(Ss, Sr) <= TOL
    h.close()


@pytest.mark.parametrize("ng,cap", [(50, None), (64, None), (700, None), (700, 200000)])
@pytest.mark.parametrize("norm", [None, 0.0])
def test_split_sample_from_real_vectors(ctx, monkeypatch, ng, cap, norm):
    """The FP64 sample of split precision, over one and several column chunks:
    the error it reports is the split result's distance from FP64 on the sampled
    columns.  FP64's own rounding, 1e-14 at most, is 1e-3 of the 1e-11 that 9
    moduli leave."""
    from hybridhsdla_amd.api import HSGEN_PREC_OZAKI_INT8
    s, kp = tiny_system(natoms=10, lmax=(3, 5), a_cell=11.0, ng_target=720, seed=17)
    if norm is not None:
        s.match[1, 1, 4] = norm
    sub = _subset(kp, np.arange(ng))
    h = ctx.upload(s)
    H0, S0 = ctx.create_HS2(h, sub)
    if cap:
        monkeypatch.setenv("HSGEN_BATCH_BYTES", str(cap))
    H, S, rep = ctx.create_HS2(h, sub, precision=HSGEN_PREC_OZAKI_INT8, slices=9, report=True)
    nb = min(ng, 64)
    cols = [(2 * j + 1) * ng // (2 * nb) for j in range(nb)]
    for X, X0, e in ((H, H0, rep["err_smp_h"]), (S, S0, rep["err_smp_s"])):
        d = np.sqrt(sum(np.sum(np.abs(X[j:, j] - X0[j:, j]) ** 2) for j in cols) /
                    sum(np.sum(np.abs(X0[j:, j]) ** 2) for j in cols))
        print(f"sample {e:.4e} direct {d:.4e}", flush=True)
        assert d > 1e-12 and abs(e - d) <= 1e-2 * d
    h.close()
