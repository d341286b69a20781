// hsgen_create_hs_noalloc: hsgen_create_hs in FP64 with no device allocation,
// for callers that cannot call hipMalloc (code under HIP graph capture, tight
// serving loops, harnesses that forbid it).
//
// Every workspace of the call (the G list when it is host memory, the phases,
// radial factors, real vectors and W of sphere.h) lives in `scratch`, one
// file-scope device array that each GPU the library runs on holds until the
// process ends.  In host code the array's name is only a host-side stand-in:
// the address of each GPU's copy comes from hipGetSymbolAddress, taken once
// per device when a context is created on it (noalloc_setup, called by
// hsgen_init with the device current), and only that address is handed to
// kernels and copies.
//
// What is served is set by the size of the general operands (Y and W, or Z,
// Zs and W, and their work lists) against HSGEN_NOALLOC_SCRATCH_BYTES.  The
// call's own operands need less for the l cutoffs in use, but up to 9/4 as
// much where atoms have lmax 0 and each is of a kind of its own (144 bytes per
// plane wave: phase 16, radial factors 32, y and W of two rows padded to the
// MFMA depth of four 32 and 64; general operands 64), and 3/2 for S alone.
// Those calls go in parts: S over some groups of atoms at a time, then H from
// some columns of W at a time (phases and y 48 bytes, the rest for W).
//
// The call copies nothing from host memory except a host G list (a short one is
// read from pinned memory).  Every value
// that reaches H or S is written earlier in the same call, so nothing needs
// clearing between calls.  Calls on one GPU share its array and the last
// call's contents stay there: calls that overlap on one GPU, from any
// contexts, race.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "hsgen_host.h"

namespace hsgen {

constexpr size_t kScratchLimit = HSGEN_NOALLOC_SCRATCH_BYTES;      // of the general operands
constexpr size_t kScratchBytes = kScratchLimit + ((size_t)1 << 20);   // the array
constexpr int kScratchDevices = 64;

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

std::mutex g_scratch_mu;
void* g_scratch_ptr[kScratchDevices] = {};   // per device: the address of that GPU's `scratch`

// Lower tiles of tile row bi of an ng x ng problem: the bj with
// bj * cbn < (bi + 1) * cbm.
inline int lower_row_tiles(int bi, int ntc, int cbm, int cbn)
{
    return std::min(ntc, (int)(((int64_t)(bi + 1) * cbm + cbn - 1) / cbn));
}

void* scratch_of(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return (device >= 0 && device < kScratchDevices) ? g_scratch_ptr[device] : nullptr;
}

}  // namespace

// Once per device, with the device current: the address of its `scratch`.
hsgen_status noalloc_setup(hsgen_ctx* ctx)
{
    if (ctx->device < 0 || ctx->device >= kScratchDevices) return HSGEN_OK;   // entry point reports it
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[ctx->device]) return HSGEN_OK;
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        (void)hipGetLastError();
        return fail(ctx, HSGEN_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", ctx->device,
                    hipGetErrorString(e));
    }
    g_scratch_ptr[ctx->device] = ptr;
    return HSGEN_OK;
}

}  // namespace hsgen

using namespace hsgen;

extern "C" hsgen_status hsgen_create_hs_noalloc(hsgen_ctx* ctx, const hsgen_sys* s, const hsgen_kpoint* kp,
                                                const hsgen_opts* opts, double* H, double* S, int64_t ld,
                                                hsgen_report* rep)
{
    if (!ctx || !s) return fail(ctx, HSGEN_ERR_ARG, "null argument");
    hsgen_status st = check_kpoint(ctx, kp);
    if (st) return st;
    hsgen_opts o{};
    if (opts) o = *opts;
    if (o.precision != HSGEN_PREC_FP64)
        return fail(ctx, HSGEN_ERR_UNSUPPORTED, "the allocation-free entry point computes in FP64 only");
    const int ng = kp->ng;
    if (ld < std::max(ng, 1)) return fail(ctx, HSGEN_ERR_ARG, "ld %lld < ng %d", (long long)ld, ng);
    const bool do_h = !(o.flags & HSGEN_SKIP_H), do_s = !(o.flags & HSGEN_SKIP_S);
    if ((do_h && !H) || (do_s && !S)) return fail(ctx, HSGEN_ERR_ARG, "null output matrix");
    if ((do_h && !is_device_ptr(H)) || (do_s && !is_device_ptr(S)))
        return fail(ctx, HSGEN_ERR_ARG, "the allocation-free entry point needs H and S in device memory");
    if (rep) std::memset(rep, 0, sizeof *rep);
    if (ng == 0) return HSGEN_OK;
    HIPCHK(hipSetDevice(ctx->device));
    if (!s->real_vectors) return fail(ctx, HSGEN_ERR_ARG, "K %d is beyond the allocation-free entry point", s->kdim);
    char* base = (char*)scratch_of(ctx->device);
    if (!base) return fail(ctx, HSGEN_ERR_UNSUPPORTED, "no scratch array on device %d", ctx->device);
    o.tile = pick_tile(ctx, o, ng, s->kdim);
    Geometry geo = geometry(o.tile, s->kdim, ng);
    geo.fold = s->fold;
    const int tc = tapp_cfg(geo);
    const ZgemmLaunchCfg tcc = zgemm_cfg(tc);
    // the general operands and their work lists, which set the limit
    const int na = s->natoms;
    const int ntn = (int)((geo.gp + tcc.bn - 1) / tcc.bn);
    int64_t n_tmul = 0;
    if (do_h)
        for (int a = 0; a < na; ++a) n_tmul += (int64_t)((2 * s->atoms[a].nlm + tcc.bm - 1) / tcc.bm) * ntn;
    const int ntr = (ng + geo.t.bm - 1) / geo.t.bm, ntc = (ng + geo.t.bn - 1) / geo.t.bn;
    int64_t n_hs = 0;
    for (int bi = 0; bi < ntr; ++bi) n_hs += lower_row_tiles(bi, ntc, geo.t.bm, geo.t.bn);
    n_hs *= (int)do_s + (int)do_h;
    if (n_tmul + n_hs > INT32_MAX) return fail(ctx, HSGEN_ERR_ARG, "too many tiles");
    const bool gdev = is_device_ptr(kp->g);
    size_t off = 0;
    auto take = [&](size_t bytes) {   // 256-byte aligned pieces
        const size_t at = off;
        off = (size_t)roundup((int64_t)(off + bytes), 256);
        return at;
    };
    if (!gdev) take(sizeof(int32_t) * 3 * (size_t)ng);
    take(sizeof(GemmProblem) * (size_t)(na + 2));
    take(sizeof(TileWork) * (size_t)(n_tmul + n_hs));
    take(sizeof(int32_t) * (size_t)(na + 1));
    const size_t zbytes = sizeof(double2) * (size_t)geo.ldz * (size_t)geo.gp;
    for (int i = 0; i < (geo.fold ? 1 : 2) + (int)do_h; ++i) take(zbytes);
    if (off > kScratchLimit)
        return fail(ctx, HSGEN_ERR_ARG,
                    "N_G %d with K %d needs %zu bytes of scratch; the allocation-free entry point has %zu "
                    "(use hsgen_create_hs)",
                    ng, s->kdim, off, kScratchLimit);
    // the call's own layout
    SphereLayout l = sphere_layout(ctx, s, {ng}, do_h);
    off = 0;
    const size_t o_g = gdev ? 0 : take(sizeof(int32_t) * 3 * (size_t)ng);
    const size_t o_ph = take(l.b_ph), o_rs = take(l.b_rs), o_y = take(l.b_y), o_w = take(l.b_w);
    if (off > kScratchBytes && (o_ph >= kScratchBytes || !sphere_parts(s, l, do_h, do_s, kScratchBytes - o_ph)))
        return fail(ctx, HSGEN_ERR_ARG, "N_G %d with K %d needs %zu bytes of scratch; the array has %zu", ng, s->kdim, off,
                    kScratchBytes);
    SphereArgs p = sphere_args(s, l, base + o_ph, base + o_rs, do_h ? base + o_y : nullptr, do_h ? base + o_w : nullptr);
    p.one = sphere_ks(l, {kp}, {nullptr}, {(double2*)H}, {(double2*)S}, {ld}, {ld})[0];
    st = sphere_g(ctx, kp, gdev ? nullptr : (int32_t*)(base + o_g), p.one);
    if (st) return st;
    return sphere_run(ctx, s, l, p, o.flags, geo.cfg, rep);
}
