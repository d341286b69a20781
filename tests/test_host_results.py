"""Matrices that the binding allocates for a call's results: what the library
does not write is zero, whatever the memory held before."""
import numpy as np
import pytest

from hybridhsdla_amd import api, tiny_system
from hybridhsdla_amd.system import KPoint

# 1448 plane waves are the last whose matrices (32 MiB) are left to the library to clear
ORDERS = [(400, 1500), (1500, 400), (1448, 1449, 30), (40, 30), (1449, 1449)]
FLAGS = [0, api.HSGEN_FILL_UPPER, api.HSGEN_SKIP_H, api.HSGEN_SKIP_S]


def _dirty_empty(monkeypatch):
    monkeypatch.setattr(api.np, "empty", lambda shape, dtype=float, order="C": np.full(shape, 5.0, dtype, order))


def _zero_where_unwritten(H, S, flags):
    for X, skipped in ((H, flags & api.HSGEN_SKIP_H), (S, flags & api.HSGEN_SKIP_S)):
        if skipped:
            assert not X.any()
        elif not flags & api.HSGEN_FILL_UPPER:
            assert not np.triu(X, 1).any()


class _Library:
    """hsgen_create_hs_batched as far as memory goes: ones where H and S are
    written, zeros above the diagonal where the flags ask for them."""

    def hsgen_create_hs_batched(self, ctx, sys, nk, kps, opts, H, S, ld, reps):
        flags = opts._obj.flags
        for i in range(nk):
            n = kps[i].ng
            for ptrs, skip in ((H, api.HSGEN_SKIP_H), (S, api.HSGEN_SKIP_S)):
                if flags & skip:
                    continue
                buf = (api.C.c_double * (2 * n * n)).from_address(ptrs[i])
                m = np.frombuffer(buf, dtype=np.complex128).reshape((n, n), order="F")
                m[np.tril_indices(n)] = 1.0
                if flags & api.HSGEN_FILL_UPPER:
                    m[:] = 1.0
                elif flags & api.HSGEN_CLEAR_UPPER:
                    m[np.triu_indices(n, 1)] = 0.0
        return 0


@pytest.mark.parametrize("flags", FLAGS)
@pytest.mark.parametrize("ngs", ORDERS)
def test_batched_binding(monkeypatch, ngs, flags):
    """One decision for all k-points of a call, in any order of their sizes."""
    _dirty_empty(monkeypatch)
    ctx = api.Context.__new__(api.Context)
    ctx.lib, ctx.handle = _Library(), None
    sysh = type("Handle", (), {"handle": None})()
    kps = [KPoint(k=np.zeros(3), g=np.zeros((n, 3), dtype=np.int32), kmax=1.0) for n in ngs]
    res, _ = ctx.create_HS2_batched(sysh, kps, flags=flags)
    assert [H.shape[0] for H, _ in res] == list(ngs)
    for H, S in res:
        _zero_where_unwritten(H, S, flags)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [api.HSGEN_PREC_FP64, api.HSGEN_PREC_OZAKI_INT8])
@pytest.mark.parametrize("ngs", ORDERS[:2])
def test_batched_results_of_both_kinds(ctx, monkeypatch, ngs, precision):
    s, kp = tiny_system(natoms=2, lmax=(3, 2), a_cell=13.0, ng_target=1520, seed=23)
    kps = [KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[:n]), kmax=kp.kmax) for n in ngs]
    h = ctx.upload(s)
    want = [ctx.create_HS2(h, k, precision=precision, H=np.zeros((k.ng, k.ng), complex, order="F"),
                           S=np.zeros((k.ng, k.ng), complex, order="F")) for k in kps]
    _dirty_empty(monkeypatch)
    res, _ = ctx.create_HS2_batched(h, kps, precision=precision)
    for pair, ref in zip(res, want):
        for X, W in zip(pair, ref):
            assert np.array_equal(X, W)
    h.close()
