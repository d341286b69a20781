"""The threads that copy results to the host sleep while the GPU computes them."""
import ctypes as C
import time

import numpy as np
import pytest

from hybridhsdla_amd import api

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_no_thread_spins_while_the_gpu_computes(ctx):
    """A contraction of given coefficients into host matrices: 0.2 s of products,
    then 576 MB to copy.  The calling thread polls throughout (1 x the time), the
    HIP runtime may (1 x), eight threads copy for about a tenth of it (1 x); threads
    that wait for the copy by spinning would add 7 to 8 x."""
    natoms, lmax, ng = 256, 8, 6000
    L = (lmax + 1) ** 2
    gen = torch.Generator(device="cuda").manual_seed(5)
    A, B = (torch.randn((ng, natoms * L), dtype=torch.complex128, device="cuda", generator=gen) for _ in range(2))
    t = np.asfortranarray(np.eye(L, dtype=np.complex128))
    ptr = (C.c_void_p * natoms)(*[t.ctypes.data] * natoms)
    size = np.full(natoms, L, dtype=np.int32)
    lm = np.full(natoms, lmax, dtype=np.int32)
    un = np.full(natoms * (lmax + 1), 0.3)
    H, S = (np.full((ng, ng), 1.0 + 0j, order="F") for _ in range(2))
    o, rep = api._opts(), api.HsgenReport()
    torch.cuda.synchronize()
    for _ in range(2):
        cpu, wall = time.process_time(), time.perf_counter()
        assert ctx.lib.hsgen_contract_hs(ctx.handle, L, natoms, ng, A.data_ptr(), B.data_ptr(), size.ctypes.data, ptr,
                                         ptr, ptr, lm.ctypes.data, lmax, un.ctypes.data, C.byref(o), H.ctypes.data,
                                         S.ctypes.data, ng, C.byref(rep)) == 0
        cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    print(f"wall {wall:.3f} s, all threads {cpu:.3f} s", flush=True)
    assert wall > 0.1 and cpu <= 4.0 * wall
    assert np.all(np.triu(H, 1) == np.triu(np.ones_like(H), 1))
    ctx.release_workspace()
