"""The allocation-free entry point depends on the system alone, not on the calls
before it: it serves a fresh system, every tile id, and the calls that follow
larger ones.  Its H and S are hsgen_create_hs's bit for bit."""
import numpy as np
import pytest

from hybridhsdla_amd import make_config
from hybridhsdla_amd.system import KPoint

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _subset(kp, n):
    return KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[:n]), kmax=kp.kmax)


def _pair(n):
    return [torch.zeros((n, n), dtype=torch.complex128, device="cuda") for _ in range(2)]


def _call(f, h, kp, **opts):
    H, S = _pair(kp.ng)
    torch.cuda.synchronize()
    f(h, kp, H.data_ptr(), S.data_ptr(), kp.ng, **opts)
    return H, S


def _equal(a, b):
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("tile", [0, 8, 11, 12])
def test_fresh_system(ctx, tile):
    s, kps = make_config(0)
    h = ctx.upload(s)
    kp = _subset(kps[0], 300)
    got = _call(ctx.create_hs_noalloc, h, kp, tile=tile)
    assert _equal(got, _call(ctx.create_hs_device, h, kp))
    h.close()


def test_between_larger_calls(ctx):
    s, kps = make_config(1, ng=2600, natoms=4)
    h = ctx.upload(s)
    kp = _subset(kps[0], 200)
    want = _call(ctx.create_hs_device, h, kp)
    for n in (2600, 700):
        _call(ctx.create_hs_device, h, _subset(kps[0], n), tile=11)
        assert _equal(_call(ctx.create_hs_noalloc, h, kp), want)
    h.close()
