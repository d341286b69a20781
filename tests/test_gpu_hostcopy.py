"""Results and inputs in host memory: the slots, groups and threads of the
copies.  Every byte equals the call on device memory, and what a call is to
leave alone stays as it was."""
import numpy as np
import pytest

from hybridhsdla_amd import tiny_system
from hybridhsdla_amd.api import HSGEN_FILL_UPPER, HSGEN_SKIP_H
from hybridhsdla_amd.system import KPoint

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _system(ng):
    s, kp = tiny_system(natoms=3, lmax=(3, 2), a_cell=15.0, ng_target=2300, seed=21)
    assert kp.ng >= ng
    return s, KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[:ng]), kmax=kp.kmax)


def _device(ctx, h, kp, flags=0):
    H, S = (torch.zeros(kp.ng, kp.ng, dtype=torch.complex128, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    ctx.create_hs_device(h, kp, H.data_ptr(), S.data_ptr(), kp.ng, flags=flags)
    return [X.cpu().numpy().T for X in (H, S)]


# 90 to 250: below one thread's share; 512: one slot exactly; 513, 700: a slot and
# more; 1449: fresh pages; 2200: more slots than the ring has
@pytest.mark.parametrize("ng", [1, 90, 250, 512, 513, 700, 1449, 2200])
@pytest.mark.parametrize("flags", [0, HSGEN_FILL_UPPER, HSGEN_SKIP_H])
def test_results(ctx, ng, flags):
    s, kp = _system(ng)
    h = ctx.upload(s)
    want = _device(ctx, h, kp, flags)
    got = ctx.create_HS2(h, kp, flags=flags)
    for X, W in zip(got, want):
        assert np.array_equal(X, W if flags & HSGEN_FILL_UPPER else np.tril(W))
    # the caller's own memory: nothing above the diagonal changes
    own = [np.full((ng, ng), 3.5 - 2j, order="F") for _ in range(2)]
    ctx.create_HS2(h, kp, flags=flags, H=own[0], S=own[1])
    for i, (X, W) in enumerate(zip(own, want)):
        if i == 0 and flags & HSGEN_SKIP_H:
            assert np.all(X == 3.5 - 2j)
        elif flags & HSGEN_FILL_UPPER:
            assert np.array_equal(X, W)
        else:
            assert np.array_equal(np.tril(X), np.tril(W)) and np.all(X[np.triu_indices(ng, 1)] == 3.5 - 2j)
    one = np.full((ng, ng), 7.0 + 0j, order="F")
    H, S = ctx.create_HS2(h, kp, flags=flags, S=one)
    assert S is one and np.array_equal(np.tril(S), np.tril(want[1])) and np.array_equal(np.tril(H), np.tril(want[0]))
    if not flags & HSGEN_FILL_UPPER:
        assert not np.triu(H, 1).any() and np.all(S[np.triu_indices(ng, 1)] == 7.0)
    h.close()


def test_leading_dimension(ctx):
    """Columns further apart than they are long."""
    import ctypes as C
    from hybridhsdla_amd import api
    s, kp = _system(900)
    h = ctx.upload(s)
    want = _device(ctx, h, kp)
    n, ld = kp.ng, 1017
    bufs = [np.full((ld, n), -1.0 + 1j, order="F") for _ in range(2)]
    ks, g = api._kpoint(kp)
    o, rep = api._opts(), api.HsgenReport()
    assert ctx.lib.hsgen_create_hs(ctx.handle, h.handle, C.byref(ks), C.byref(o), bufs[0].ctypes.data,
                                   bufs[1].ctypes.data, ld, C.byref(rep)) == 0
    for X, W in zip(bufs, want):
        assert np.array_equal(np.tril(X[:n]), np.tril(W)) and np.all(X[n:] == -1.0 + 1j)
        assert np.all(X[:n][np.triu_indices(n, 1)] == -1.0 + 1j)
    h.close()


@pytest.mark.parametrize("ng", [1, 300, 2200])
def test_coefficients_there_and_back(ctx, ng):
    """A and B to the host (62 MB at the largest), and from there into the
    contraction; two contexts give the same bytes."""
    from hybridhsdla_amd import Context
    s, kp = _system(ng)
    h = ctx.upload(s)
    A, B = ctx.construct_AB(h, kp)
    dA = torch.empty(A.size, dtype=torch.complex128, device="cuda")
    dB = torch.empty_like(dA)
    torch.cuda.synchronize()
    import ctypes as C
    from hybridhsdla_amd import api
    ks, g = api._kpoint(kp)
    assert ctx.lib.hsgen_construct_ab(ctx.handle, h.handle, C.byref(ks), dA.data_ptr(), dB.data_ptr()) == 0
    assert np.array_equal(A.reshape(-1, order="F"), dA.cpu().numpy())
    assert np.array_equal(B.reshape(-1, order="F"), dB.cpu().numpy())
    args = (s.L, s.natoms, kp.ng, A, B, s.taa, s.tab, s.tbb, s.lmax, s.max_lmax, s.sqrt_u_norms())
    H, S = ctx.create_HS2_stripped_v2(*args)
    other = Context(0)
    H2, S2 = other.create_HS2_stripped_v2(*args)
    other.close()
    assert np.array_equal(H, H2) and np.array_equal(S, S2) and not np.triu(H, 1).any()
    h.close()


def test_batched_results(ctx):
    """Matrices of several k-points in one list, all sizes of columns."""
    s, kp = _system(1100)
    kps = [KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[:n]), kmax=kp.kmax) for n in (1100, 1, 37, 820)]
    h = ctx.upload(s)
    res, _ = ctx.create_HS2_batched(h, kps)
    for (H, S), k in zip(res, kps):
        want = _device(ctx, h, k)
        assert np.array_equal(H, np.tril(want[0])) and np.array_equal(S, np.tril(want[1]))
    h.close()


def test_two_contexts_in_two_threads(ctx):
    """Contexts that share the GPU and a system, each with its own slots and
    threads, at the same time."""
    import threading
    from hybridhsdla_amd import Context
    s, kp = _system(1300)
    small = KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[:500]), kmax=kp.kmax)
    h = ctx.upload(s)
    want = [ctx.create_HS2(h, k) for k in (kp, small)]
    other = Context(0)
    bad = []

    def work(c):
        for _ in range(4):
            for k, w in zip((kp, small), want):
                got = c.create_HS2(h, k)
                if not all(np.array_equal(a, b) for a, b in zip(got, w)):
                    bad.append(k.ng)

    threads = [threading.Thread(target=work, args=(c,)) for c in (ctx, other)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads) and not bad
    other.close()
    h.close()
