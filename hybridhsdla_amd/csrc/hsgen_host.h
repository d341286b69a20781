// Host-side state and helpers shared by the hsgen C-ABI translation units:
//   context.hip     contexts, device-resident systems, workspace
//   hostcopy.hip    copies from and to host memory (threads: hostpool.cpp)
//   fp64_path.hip   tiling, the single-k and batched FP64 paths, construct_ab,
//                   create_hs, create_hs_batched, contract_hs
//   split_path.hip  split precision (Ozaki scheme II on INT8 MFMA), single-k
//                   and batched
//   tune_eig.hip    the tile autotuner and the generalized eigensolve
//   noalloc.hip     the allocation-free FP64 entry point
//   sphere_path.hip FP64 H and S from a system (kernels: sphere.hip, whose
//                   operands sphere.h describes)
//
// Operand layout of the other paths (split precision, the contraction of
// given coefficients) in HBM, per k-point (complex128, column-major, ld = ldz).
// Folded (every ||u_dot_l||^2 > 0, the usual case):
//   Y  = [A_1; N_1^1/2 B_1; A_2; ...]   rows 2*off_a .. 2*off_a + 2*nlm_a - 1
//   W  = [M'_1 Y_1; M'_2 Y_2; ...]      M'_a = D_a^-1/2 M_a D_a^-1/2
// so that   S = Y^H Y   and   H = Y^H W   (only i >= j stored); otherwise
//   Z  = [A_1; B_1; A_2; B_2; ...]
//   Zs = [A_1; N_1 B_1; ...]            N_a = diag(||u_dot_l||^2)
//   W  = [M_1 Z_1; M_2 Z_2; ...]        M_a = [[T_aa, T_ab], [T_ab^H, T_bb]]
// so that   S = Z^H Zs   and   H = Z^H W.  Y lives where Z does (ctx->Z).
// ldz = roundup(2K, BK) + BK, columns padded to the tile size; every padding
// element is zero so the kernels need no bounds checks along k.
#pragma once

#include <unistd.h>

#include <atomic>
#include <complex>
#include <cstdarg>
#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include <rocblas/rocblas.h>

#include "../../include/hsgen.h"
#include "hostpool.h"
#include "hsgen_internal.h"
#include "sphere.h"

namespace hsgen {

constexpr int kDefaultTile = 11;
// FP64 tile for problems too small to fill the GPU with 128 x 128 tiles:
// fewer than kSmallWaves tiles of 128 x 128 per CU (S and H lower tiles of
// all k-points of the call) take the 64 x 64 tile, whose workgroups are a
// quarter of the work and two of which a CU holds at once
constexpr int kSmallTile = 12;
constexpr int kSmallWaves = 6;
// INT8 configurations of 128 x 128 and 128 x 256 tiles for smaller calls
// (pick_tile), BF16: 256 x 128 below kBf16SomeTiles S and H lower tiles of 256 x 192
// (all k-points)
constexpr int kInt8SmallCfg = 14, kInt8MidCfg = 15, kBf16SmallCfg = 62;
constexpr int kBf16SomeTiles = 160;
constexpr int kFallbackTile = 8;   // register-staged, 64-bit addressing
constexpr int kIgemmCfg = 51;      // default INT8 kernel configuration (256 x 192 tiles)
constexpr int kBf16Cfg = 61;       // default BF16 kernel configuration (256 x 192 tiles)
constexpr int kSampleTile = 12;    // FP64 tile of the split-precision sample: 64 x 64, so 64 columns
constexpr int kPinnedG = 4096;     // plane waves of a G list that is read from pinned host memory
constexpr size_t kPinStamps = 64;
constexpr int kRingSlots = 6;       // pinned slots of a host copy
constexpr size_t kMaxOzGraphs = 16; // cached split-precision launch-segment sets per context

struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
};

// Columns to copy between device and host memory; sizes and strides in bytes.
// Device addresses and strides are multiples of 16, so are sizes of several
// columns; a run's size is a multiple of 8.
struct HostCopy {
    char* dev;
    char* host;
    size_t rows, cols, ldd, ldh;
    bool lower;        // of column j only the 16-byte rows from j on
    bool clear;        // and zeros into the host's rows above them
};
inline HostCopy copy_run(void* dev, const void* host, size_t bytes)
{
    return {(char*)dev, (char*)host, bytes, 1, bytes, bytes, false, false};
}
// an n x n matrix, its lower triangle or (HSGEN_FILL_UPPER) all of it
inline HostCopy copy_matrix(const double2* dev, int n, double* host, int64_t ld, int flags)
{
    const size_t e = sizeof(double2);
    return {(char*)dev, (char*)host, e * n, (size_t)n, e * n, e * ld, !(flags & HSGEN_FILL_UPPER),
            (flags & HSGEN_CLEAR_UPPER) != 0};
}

// Maps the pages of a call's host results in the background until they are
// copied or the object goes.
class Prefault {
public:
    Prefault(hsgen_ctx* ctx, const std::vector<HostCopy>& list);
    ~Prefault();
    void stop() { stop_.store(true, std::memory_order_relaxed); }

private:
    hsgen_ctx* ctx_;
    HostPool* pool_ = nullptr;
    std::vector<std::pair<char*, size_t>> ranges_;
    std::atomic<size_t> next_{0};
    std::atomic<bool> stop_{false};
};

}  // namespace hsgen

struct hsgen_ctx {
    int device = 0;
    pid_t pid = getpid();                            // of the process whose GPU resources these are
    hipStream_t stream = nullptr;
    hipStream_t stream2 = nullptr;                   // S beside the T application and H
    hipEvent_t ev[8] = {};
    std::string err;
    // workspace
    hsgen::DevBuf Z, Zs, W, Htmp, Stmp, A, B, g, probs, work, pack, m_in, M, lists;
    // split precision (oz_res: before the residues, the real vectors that W is formed from)
    hsgen::DevBuf oz_e, oz_res, oz_out, oz_probs, oz_work, oz_smp, oz_fprob;
    hipEvent_t oz_ev[2 * hsgen::kMaxModuli] = {};   // INT8 GEMM start/stop per residue group
    int n_cu = 0;                                    // compute units
    // batched k-points: one captured graph per batch, replayed while the
    // call signature is unchanged
    struct BatchGraph {
        std::vector<int64_t> sig;
        hipGraphExec_t exec = nullptr;
        hsgen::DevBuf g, ks;
    };
    std::vector<BatchGraph> bgraphs;
    hsgen::DevBuf btmp;                              // device H, S of host-output k-points
    // batched split precision: captured launch segments of one evaluation
    // (per residue group its residue pass and its INT8 launches, then the
    // recombination) with their own problem and tile lists, replayed while
    // their key (modulus count, k-points, outputs, workspace) is unchanged
    struct OzGraph {
        std::vector<int64_t> key;
        hsgen::DevBuf probs, work, fprob;
        std::vector<hipGraphExec_t> seg;
    };
    std::list<OzGraph> ozgraphs;                     // oldest first, at most kMaxOzGraphs
    // autotuned tile configurations: (precision, size buckets) -> config id
    std::map<std::vector<int>, int> tuned;
    // generalized eigensolver
    rocblas_handle blas = nullptr;
    hsgen::DevBuf eig_a, eig_b, eig_d;
    // pinned buffer and its device address: kernel starts (kPinStamps bytes), then
    // a short G list (kPinnedG plane waves)
    void* pin = nullptr;
    void* pin_dev = nullptr;
    double ms_per_tick = 1e-5;                       // of the GPU's wall clock
    // pinned slots of copies from and to pageable memory
    char* ring = nullptr;
    void* ring_dev = nullptr;
    uint64_t ring_seq = 0;
    hsgen::DevBuf ring_left;
    std::unique_ptr<hsgen::HostPool> pool;
    hsgen::Prefault* prefault = nullptr;
};

struct hsgen_sys {
    uint64_t serial = 0;               // unique per created system
    int natoms = 0, max_lmax = 0, nl = 0, L = 0, kdim = 0;
    double omega = 0.0, vol_prefac = 0.0;
    double bmat[9];
    std::vector<hsgen::AtomDev> atoms; // host copy
    std::vector<int64_t> m_off;        // per atom: offset of M_a in d_M (complex units)
    std::vector<int32_t> m_ld;         // per atom: leading dim of M_a
    std::vector<int32_t> m_cols;       // per atom: padded column count
    int m_bk = 0, m_bm = 0;            // tile geometry M was padded for
    // M is built by the first call that reads it (calls on contexts that share
    // the system may be the first together)
    std::mutex m_mu;
    int64_t sum_nlm2 = 0;              // sum_a nlm_a^2
    // folded operands: Y = [A_a; sqrt(N_a) B_a] per atom (S = Y^H Y,
    // H = Y^H M' Y) when every N_l = ||u_dot_l||^2 is positive; otherwise
    // Z and Zs = [A_a; N_a B_a] (S = Z^H Zs, H = Z^H M Z)
    bool fold = false;
    std::vector<double> h_sqrtn;       // [natoms][nl] sqrt(N_l), 0 for l > lmax
    hsgen::AtomDev* d_atoms = nullptr;
    hsgen::RadDev* d_rad = nullptr;
    double* d_ynorm = nullptr;
    double2* d_M = nullptr;
    // host copies of the T blocks, so that M can be rebuilt for another tile
    // geometry
    std::vector<std::vector<std::complex<double>>> h_taa, h_tab, h_tbb;
    std::vector<int> h_owner;          // per atom: the atom whose copies hold its T
    // FP64 path (sphere.h): one allocation, d_sphere
    void* d_sphere = nullptr;
    double2* d_mt = nullptr;
    hsgen::KindDev* d_kinds = nullptr;
    hsgen::OverlapGroup* d_groups = nullptr;
    int32_t* d_order = nullptr;
    hsgen::SphereStage* d_stages = nullptr;
    int64_t* d_mtoff = nullptr;
    std::vector<int32_t> h_order;      // atoms in kind order
    std::vector<hsgen::OverlapGroup> h_groups;
    std::vector<int32_t> h_group_kind; // first kind of each, and the end
    // split precision (built by its first call): matrices, their offsets per
    // atom in kind order, rows of W
    void* d_split = nullptr;
    int64_t* d_split_off = nullptr;
    int32_t* d_split_rows = nullptr;
    int nkinds = 0, ngroups = 0, nksteps = 0, ldr = 0, rt32 = 0;
    int64_t ldy = 0, ldw = 0;
    bool real_vectors = true;          // calls take the path of sphere.h, else the general operands
    // first atom of each rotation class and of each rmt class (AtomDev::cls)
    std::vector<int32_t> rot_rep, rmt_rep;
};

namespace hsgen {

// Record the error text on the context and return the status.
hsgen_status fail(hsgen_ctx* ctx, hsgen_status s, const char* fmt, ...);

#define HIPCHK(call)                                                                  \
    do {                                                                              \
        hipError_t e_ = (call);                                                       \
        if (e_ != hipSuccess)                                                         \
            return ::hsgen::fail(ctx, HSGEN_ERR_HIP, "%s failed: %s (%s:%d)", #call,  \
                                 hipGetErrorString(e_), __FILE__, __LINE__);          \
    } while (0)

inline int64_t roundup(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// ---- context.hip ----
// Grow a workspace buffer to at least `bytes` (contents not kept).
hsgen_status ensure(hsgen_ctx* ctx, DevBuf& b, size_t bytes, bool zero_new);
void release(DevBuf& b);
bool is_device_ptr(const void* p);
// M_a blocks of every atom padded for tile geometry (bk, bm), deduplicated by
// T pointer triple, built at s->d_M: in `into`, or (null) in an allocation of
// the system's own.  in: further copies to the device that the call needs.
hsgen_status upload_M(hsgen_ctx* ctx, hsgen_sys* s, const int32_t* nlm, const double* const* taa,
                      const double* const* tab, const double* const* tbb, const double* rsc, int bk, int bm, DevBuf* into,
                      std::vector<HostCopy> in);
// Folded operands unless HSGEN_FOLD=0 (environment; tests and comparisons).
bool fold_enabled();
// N_l usable for folding (positive, 1/sqrt(N) far from overflow).
bool fold_ok(double n);
hsgen_status ensure_M(hsgen_ctx* ctx, hsgen_sys* s, int bk, int bm);
hsgen_status check_kpoint(hsgen_ctx* ctx, const hsgen_kpoint* kp);
hsgen_status upload_g(hsgen_ctx* ctx, const hsgen_kpoint* kp);
// Copies of a call, started on `stream` and complete on return (to the device:
// the host side is; calls with different streams order their slots' use).
// computed: to the host, what is copied is there already.
hsgen_status host_copy(hsgen_ctx* ctx, const std::vector<HostCopy>& list, bool to_host, hipStream_t stream,
                       bool computed = true);

// ---- fp64_path.hip ----
struct Geometry {
    int cfg;
    ZgemmLaunchCfg t;
    int64_t kpad;   // kdepth of the S/H contraction = roundup(2K, BK)
    int64_t ldz;    // kpad + BK
    int64_t gp;     // padded column count
    bool fold;      // operands Y (in Z) and W: S = Y^H Y; else Z, Zs, W
};

// FP64 operand arrays per column set: Y, W (folded) or Z, Zs, W.
inline int n_operands(const Geometry& g) { return g.fold ? 2 : 3; }
// The right operand of S: Zs, or Y itself (in ctx->Z) when folded.
inline double2* zs_ptr(hsgen_ctx* ctx, const Geometry& g) { return (double2*)(g.fold ? ctx->Z.p : ctx->Zs.p); }

// Split precision (INT8 or BF16 MFMA on the same residues).
inline bool is_split(int precision)
{
    return precision == HSGEN_PREC_OZAKI_INT8 || precision == HSGEN_PREC_OZAKI_BF16;
}
inline bool valid_precision(int precision) { return precision == HSGEN_PREC_FP64 || is_split(precision); }
// The split-precision kernel configuration of a call: opts.tile when it names
// one for the precision's MFMA type, else the precision's default.
int split_cfg(int precision, int tile);
// Column padding of split-precision operands: a multiple of both tile sides.
int64_t split_col_align(int precision, int tile);
Geometry geometry(int tile, int kdim, int ng, int64_t col_align = 1);
void add_hs_problems(std::vector<GemmProblem>& probs, std::vector<TileWork>& work, const Geometry& geo, int ng,
                     const double2* Z, const double2* Zs, const double2* W, double2* H, double2* S, int64_t ld,
                     int flags);
void xcd_permute(std::vector<TileWork>& work);
AbgenParams abgen_params(const hsgen_sys* s, const hsgen_kpoint* kp, const int32_t* dg);
int tapp_cfg(const Geometry& geo);
void add_tmul_problems(std::vector<GemmProblem>& probs, std::vector<TileWork>& work, const hsgen_sys* s,
                       const Geometry& geo, const ZgemmLaunchCfg& tc, int64_t ncols, const double2* Z, double2* W);
hsgen_status run_grouped(hsgen_ctx* ctx, int cfg, std::vector<GemmProblem>& probs, std::vector<TileWork>& work);
hsgen_status finish_hs(hsgen_ctx* ctx, hsgen_sys* s, const Geometry& geo, int ng, const hsgen_opts& o, double* H,
                       double* S, int64_t ld, hsgen_report* rep, double ms_front,
                       const hsgen_kpoint* kp = nullptr);

// create_hs on the general operands (split precision; the autotuner's FP64 runs)
hsgen_status create_hs_general(hsgen_ctx* ctx, hsgen_sys* s, const hsgen_kpoint* kp, const hsgen_opts& o, double* H,
                               double* S, int64_t ld, hsgen_report* rep);

// ---- sphere_path.hip ----
struct SphereLayout {
    int64_t gtot = 0;                       // operand columns, 64 per tile column of every k-point
    int64_t ngcols = 0, nsquares = 0, nstiles = 0;
    int htile = 64, ttile = 64, stile = 64;
    size_t b_ph = 0, b_rs = 0, b_y = 0, b_w = 0;   // bytes of the operand arrays
    // a call in parts (sphere_parts), or empty and 0
    std::vector<int> sparts;                // first groups of S's parts, and the end
    int64_t wcols = 0;                      // columns of W at a time
};
// Operands of a call: phases, radial factors, real vectors, W.
struct SphereOperands {
    void *ph, *rs, *y, *w;
};
hsgen_status sphere_setup(hsgen_ctx* ctx, hsgen_sys* s, const RadDev* rad);
hsgen_status sphere_operands(hsgen_ctx* ctx, const SphereLayout& l, bool do_h, SphereOperands& o);
SphereLayout sphere_layout(const hsgen_ctx* ctx, const hsgen_sys* s, const std::vector<int>& ngs, bool do_h);
// Lays a call of one k-point out for `bytes` of memory that do not hold its
// operands at once (all of it from SphereArgs::ph on); false if it cannot be.
bool sphere_parts(const hsgen_sys* s, SphereLayout& l, bool do_h, bool do_s, size_t bytes);
SphereArgs sphere_args(const hsgen_sys* s, const SphereLayout& l, void* ph, void* rs, void* y, void* w);
std::vector<SphereK> sphere_ks(const SphereLayout& l, const std::vector<const hsgen_kpoint*>& kps,
                               const std::vector<const int32_t*>& gs, const std::vector<double2*>& H,
                               const std::vector<double2*>& S, const std::vector<int64_t>& ldH,
                               const std::vector<int64_t>& ldS);
hsgen_status sphere_g(hsgen_ctx* ctx, const hsgen_kpoint* kp, int32_t* dev, SphereK& k);
hipError_t sphere_launch(const SphereArgs& p, const SphereLayout& l, const hsgen_sys* s, bool do_h, bool do_s,
                         hipEvent_t stop, hipStream_t st);
hsgen_status sphere_run(hsgen_ctx* ctx, const hsgen_sys* s, const SphereLayout& l, SphereArgs& p, int flags, int tile,
                        hsgen_report* rep);
hsgen_status sphere_split_setup(hsgen_ctx* ctx, hsgen_sys* s);
hsgen_status sphere_split_w(hsgen_ctx* ctx, hsgen_sys* s, const std::vector<SphereK>& ks, const SphereK* ks_dev,
                            int64_t ncols, double2* W, int64_t ldw, const std::vector<int32_t>* cols, bool do_s);
// Bytes of the operands per plane wave (reports).
inline double sphere_gen_bytes(const hsgen_sys* s)
{
    return 16.0 * s->natoms + 16.0 * s->ldr + 8.0 * s->ldy;
}

// ---- split_path.hip ----
struct OzResult {
    int nmod = 0;
    double est_h = 0.0, est_s = 0.0;     // modelled error, exact norms
    double smp_h = 0.0, smp_s = 0.0;     // measured error on the FP64 sample block
    double ms_igemm = 0.0;
};

// One k-point of a split-precision run: columns [col0, col0 + ng) of the
// resident Z, Zs, W (each k-point's columns padded to a multiple of both INT8
// tile sides) and its device outputs.
struct OzK {
    int ng = 0;
    int64_t col0 = 0;
    int64_t ncols = 0;      // padded column count (ng rounded up to the INT8 tile multiple)
    double2* dH = nullptr;
    int64_t ldH = 0;
    double2* dS = nullptr;
    int64_t ldS = 0;
};

// The FP64 sample of a call: nb evenly spaced columns of S and H of every
// k-point, all rows, leading dimension ng, in the context's sample buffer.
struct OzSample {
    std::vector<int> nb;
    std::vector<int32_t> cols;                 // the columns, relative to their k-point
    std::vector<size_t> soff, off, gath;       // per k-point: first of cols, of S and H, of the gathered operands
    size_t nbt = 0, total = 0, gath_total = 0;
    int nsplit = 1;
    double2* S = nullptr;
    double2* H = nullptr;
    double2* gath_s = nullptr;
    double2* gath_h = nullptr;
    double2* parts = nullptr;
    // kSampleCols columns per k-point, the last again past nb
    std::vector<int32_t> padded() const;
};
// operands: whether run_ozaki forms it from the operands (with memory for their
// gathered columns and the depth chunks' products), or sphere_split_w does.
hsgen_status oz_sample(hsgen_ctx* ctx, const Geometry& geo, const std::vector<OzK>& ks, bool operands, OzSample& smp);

// capture: the INT8 launch sequence of each modulus count runs as cached
// hipGraphs (the batched path), else eagerly.  sample: null, or the call's
// sample, computed already.
hsgen_status run_ozaki(hsgen_ctx* ctx, const Geometry& geo, const std::vector<OzK>& ks, int flags, int icfg,
                       int nmod_req, double target, std::vector<OzResult>& res, bool capture, const OzSample* sample);
void destroy_oz_graph(hsgen_ctx::OzGraph& g);
hsgen_status batched_split(hsgen_ctx* ctx, hsgen_sys* s, int nk, const hsgen_kpoint* kps, const hsgen_opts& o,
                           double* const* H, double* const* S, const int64_t* ld, hsgen_report* rep);

// ---- noalloc.hip ----
// Look up this context's device's scratch array once (the device current).
hsgen_status noalloc_setup(hsgen_ctx* ctx);

// ---- tune_eig.hip ----
// Size buckets of the autotuning table: half-octaves of G and K.
std::vector<int> tune_key(int precision, int ng, int kdim);
// Tile configuration for a call: the caller's, else the autotuned one for
// this size, else 0 (the built-in default).
// The tile of a call: opts.tile if set, else the autotuned one for the size,
// else the default by size over the call's k-points (kps[0 .. nk-1], or one
// k-point of ng when kps is null).
int pick_tile(const hsgen_ctx* ctx, const hsgen_opts& o, int ng, int kdim, const hsgen_kpoint* kps = nullptr,
              int nk = 0);
// FP64 tile by size: kSmallTile when the S and H lower tiles of 128 x 128 of
// all the k-points number fewer than kSmallWaves per CU, else 0 (the default)
int fp64_tile_by_size(const hsgen_ctx* ctx, int ng, const hsgen_kpoint* kps = nullptr, int nk = 0);

}  // namespace hsgen
