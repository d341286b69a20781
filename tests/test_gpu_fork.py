"""A forked process that drops the context and the system it inherits: neither is
its to release, and the parent's work on."""
import os
import signal
import time

import numpy as np
import pytest

from hybridhsdla_amd import tiny_system

pytestmark = pytest.mark.gpu


def test_child_drops_what_it_inherits(ctx):
    from hybridhsdla_amd import Context
    s, kp = tiny_system(natoms=3, lmax=(3, 2), a_cell=12.0, ng_target=700, seed=2)
    c = Context(0)
    h = c.upload(s)
    H, S = c.create_HS2(h, kp)          # 8 MB and more: the copying threads are there
    pid = os.fork()
    if pid == 0:
        h.close()
        c.close()
        os._exit(0)
    for _ in range(200):
        done, status = os.waitpid(pid, os.WNOHANG)
        if done:
            break
        time.sleep(0.05)
    else:
        os.kill(pid, signal.SIGKILL)
        os.waitpid(pid, 0)
        pytest.fail("the child did not end")
    assert os.WIFEXITED(status) and os.WEXITSTATUS(status) == 0
    H2, S2 = c.create_HS2(h, kp)
    assert np.array_equal(H, H2) and np.array_equal(S, S2)
    h.close()
    c.close()
