"""The allocation-free entry point at its size limit, where the operands of atoms
that share nothing pass its array: S over some of the atoms at a time, H from
some columns of W at a time, with the bits of hsgen_create_hs.  And what the array
takes of the GPU's memory."""
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from hybridhsdla_amd import tiny_system
from hybridhsdla_amd.api import HSGEN_FILL_UPPER, HSGEN_SKIP_H, HSGEN_SKIP_S, HsgenError
from hybridhsdla_amd.system import KPoint
from oracle import pyoracle as po
from tests.helpers import rel_fro_lower

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ROOT = Path(__file__).resolve().parent.parent


def _subset(kp, idx):
    return KPoint(k=kp.k, g=np.ascontiguousarray(kp.g[np.asarray(idx, dtype=np.int64)]), kmax=kp.kmax)


@pytest.fixture(scope="module")
def system():
    """1000 atoms of lmax 0 (one of lmax 1), each with radial data of its own:
    2.0 KB of Y and as much of W per plane wave; phases, radial factors, real
    vectors and W padded to k-steps of four take 144 KB."""
    s, kp = tiny_system(natoms=1000, lmax=(0, 1), a_cell=40.0, ng_target=7900, seed=2)
    s.lmax[:] = 0
    s.lmax[400] = 1
    one = [np.asfortranarray(t[:1, :1]) for t in (s.taa[0], s.tab[0], s.tbb[0])]
    four = [s.taa[1], s.tab[1], s.tbb[1]]
    for a in range(s.natoms):
        s.taa[a], s.tab[a], s.tbb[a] = four if a == 400 else one
    s.match[:] = s.match[1]
    s.match[:, :, 0] += 1e-3 * np.arange(s.natoms)[:, None]
    assert kp.ng >= 7800
    return s, kp


def _pair(n):
    return [torch.zeros((n, n), dtype=torch.complex128, device="cuda") for _ in range(2)]


# 3900 plane waves: 246 MiB of Y and W (536 of the call's own); 7800 with S alone
# 242 MiB of Y (358)
@pytest.mark.parametrize("ng,flags", [(3900, 0), (3900, HSGEN_SKIP_S | HSGEN_FILL_UPPER), (7800, HSGEN_SKIP_H),
                                      (7800, HSGEN_SKIP_H | HSGEN_SKIP_S)])
def test_at_the_limit(ctx, system, ng, flags):
    s, kp = system
    sub = _subset(kp, np.arange(ng))
    h = ctx.upload(s)
    want, got = _pair(ng), _pair(ng)
    torch.cuda.synchronize()
    ctx.create_hs_device(h, sub, want[0].data_ptr(), want[1].data_ptr(), ng, flags=flags)
    for _ in range(2):
        rep = ctx.create_hs_noalloc(h, sub, got[0].data_ptr(), got[1].data_ptr(), ng, flags=flags)
        assert rep["ng"] == ng and rep["ms_total"] >= 0
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    if not flags:
        idx = np.sort(np.random.default_rng(1).permutation(ng)[:60])
        ref = po.reference_hs(s, _subset(sub, idx))
        for X, R in zip(got, ref):
            assert rel_fro_lower(X.cpu().numpy().T[np.ix_(idx, idx)], R) <= 1e-13
    # a smaller call afterwards
    small = _subset(kp, np.arange(100))
    want, got = _pair(100), _pair(100)
    torch.cuda.synchronize()
    ctx.create_hs_device(h, small, want[0].data_ptr(), want[1].data_ptr(), 100)
    ctx.create_hs_noalloc(h, small, got[0].data_ptr(), got[1].data_ptr(), 100)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    h.close()


def test_past_the_limit(ctx, system):
    """What the limit of 256 MiB of Y and W refuses stays refused."""
    s, kp = system
    sub = _subset(kp, np.arange(4300))
    h = ctx.upload(s)
    H, S = _pair(4300)
    with pytest.raises(HsgenError) as e:
        ctx.create_hs_noalloc(h, sub, H.data_ptr(), S.data_ptr(), 4300)
    assert e.value.status == -1 and "scratch" in str(e.value)
    h.close()


def test_memory_of_the_library():
    """A process that loads the library and makes a context gives up the array of
    257 MiB and the runtime's own (code objects, queues), in all under 400 MiB."""
    code = ("import torch; torch.cuda.init(); torch.zeros(1, device='cuda'); torch.cuda.synchronize()\n"
            "free = torch.cuda.mem_get_info()[0]\n"
            "from hybridhsdla_amd.api import Context\n"
            "c = Context(0)\n"
            "print((free - torch.cuda.mem_get_info()[0]) >> 20)\n")
    res = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stderr
    mib = int(res.stdout.split()[-1])
    print(f"{mib} MiB", flush=True)
    assert 256 <= mib <= 400
