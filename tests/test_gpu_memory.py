"""Device memory that a context holds after its calls."""
import numpy as np
import pytest

from hybridhsdla_amd import make_config
from hybridhsdla_amd.api import HSGEN_PREC_FP64, HSGEN_PREC_OZAKI_INT8
from hybridhsdla_amd.system import KPoint

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

MIB = 1 << 20


def _used():
    free, total = torch.cuda.mem_get_info()
    return total - free


def _workload(ng):
    """32 atoms of lmax 10: 7744 rows, so W at 2400 plane waves is 290 MiB and more."""
    s, kps = make_config(1, ng=ng)
    return s, KPoint(k=kps[0].k, g=np.ascontiguousarray(kps[0].g[:ng]), kmax=kps[0].kmax)


def _matrices(n):
    return [torch.zeros(n, n, dtype=torch.complex128, device="cuda") for _ in range(2)]


def _held(ctx, h, kp, out, precisions):
    """Bytes that the calls leave in use, beside what the first call ever sets up."""
    ctx.release_workspace()
    before = _used()
    for p in precisions:
        ctx.create_hs_device(h, kp, out[0].data_ptr(), out[1].data_ptr(), kp.ng, precision=p, slices=10 if p else 0)
    return _used() - before


def test_fp64_and_split_precision_share_their_memory(ctx):
    """One set of operands serves both, in either order."""
    s, kp = _workload(2400)
    h = ctx.upload(s)
    out = _matrices(kp.ng)
    _held(ctx, h, kp, out, [HSGEN_PREC_OZAKI_INT8, HSGEN_PREC_FP64])     # code objects, tables of the system
    split = _held(ctx, h, kp, out, [HSGEN_PREC_OZAKI_INT8])
    fp64 = _held(ctx, h, kp, out, [HSGEN_PREC_FP64])
    assert fp64 > 250 * MIB and split > 550 * MIB
    for order in ([HSGEN_PREC_OZAKI_INT8, HSGEN_PREC_FP64], [HSGEN_PREC_FP64, HSGEN_PREC_OZAKI_INT8]):
        both = _held(ctx, h, kp, out, order)
        print(f"fp64 {fp64 / MIB:.0f} split {split / MIB:.0f} both {both / MIB:.0f} MiB", flush=True)
        # the largest of each buffer: within the allocator's granularity
        assert both <= max(fp64, split) + 32 * MIB
    h.close()


def test_real_vectors_of_split_precision_take_no_memory_of_their_own(ctx):
    """Atoms that share nothing have real vectors a quarter the size of Y and W:
    they lie where the residues will."""
    s, kp = _workload(2400)
    out = _matrices(kp.ng)
    held = []
    for own in (False, True):
        if own:
            s.match = s.match.copy()
            s.match[:, :, 0] += 1e-3 * np.arange(s.natoms)[:, None]
        h = ctx.upload(s)
        _held(ctx, h, kp, out, [HSGEN_PREC_OZAKI_INT8])
        held.append(_held(ctx, h, kp, out, [HSGEN_PREC_OZAKI_INT8]))
        h.close()
    print(f"shared {held[0] / MIB:.0f} own {held[1] / MIB:.0f} MiB", flush=True)
    assert abs(held[1] - held[0]) <= 32 * MIB


def test_sample_of_a_system_takes_no_products_memory(ctx):
    """Twelve k-points of 64 plane waves, 128 columns each in 128 x 128 tiles:
    Y, W and the residues of ten moduli (of Y and of W) are what the
    call keeps.  Gathered columns for a sample from the operands would be 190 MB."""
    s, kp = _workload(100)
    h = ctx.upload(s)
    kps = [KPoint(k=kp.k + 0.001 * i, g=kp.g[:64], kmax=kp.kmax) for i in range(12)]
    out = [_matrices(64) for _ in kps]
    outputs = [(H.data_ptr(), S.data_ptr(), 64) for H, S in out]

    def held():
        ctx.release_workspace()
        before = _used()
        ctx.create_HS2_batched(h, kps, precision=HSGEN_PREC_OZAKI_INT8, slices=10, tile=14, outputs=outputs)
        return _used() - before

    held()
    rows, cols = 2 * 121 * 32, 12 * 128
    kept = held()
    want = 2 * 16 * rows * cols + 10 * 2 * 2 * rows * cols
    print(f"kept {kept / MIB:.0f} of {want / MIB:.0f} MiB", flush=True)
    assert kept <= 1.02 * want + 64 * MIB
    h.close()
