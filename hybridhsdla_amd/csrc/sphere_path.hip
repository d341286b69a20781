// Host side of the FP64 path from a system description (sphere.h, sphere.hip):
// tables of a system, operand layout of a call and its launch sequence
//   generator (phases, radial factors, real vectors) -> T application -> H, S
// shared by hsgen_create_hs, hsgen_create_hs_batched and
// hsgen_create_hs_noalloc.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>

#include "hsgen_host.h"

namespace hsgen {

namespace {

// The bits that make two atoms one kind, or, without the rotation, candidates
// for one overlap group.
std::string kind_key(const hsgen_sys* s, int a, const RadDev* rad, bool rot)
{
    const AtomDev& at = s->atoms[a];
    std::string k((const char*)&at.lmax, sizeof at.lmax);
    k.append((const char*)&at.rmt, sizeof at.rmt);
    if (rot) k.append((const char*)at.rot, sizeof at.rot);
    k.append((const char*)(rad + (size_t)a * s->nl), sizeof(RadDev) * (size_t)(at.lmax + 1));
    return k;
}

// Two rotations give the same cosines between plane waves: their R R^T (of
// kb = R^T K) agree to the rounding of the products, 4 units of each entry's own
// scale |R_i| |R_j| (in a long cell the axes' differ by orders of magnitude).
bool same_cosines(const double* r, const double* q)
{
    double g[2][9];
    for (int w = 0; w < 2; ++w) {
        const double* m = w ? q : r;
        for (int i = 0; i < 3; ++i)
            for (int j = 0; j < 3; ++j)
                g[w][3 * i + j] = m[i] * m[j] + m[3 + i] * m[3 + j] + m[6 + i] * m[6 + j];
    }
    for (int i = 0; i < 9; ++i) {
        const double scale = std::sqrt(g[0][i / 3 * 4]) * std::sqrt(g[0][i % 3 * 4]);
        if (!(std::fabs(g[0][i] - g[1][i]) <= 4.0 * 2.220446049250313e-16 * scale)) return false;   // NaN too
    }
    return true;
}

// Rotation class of an atom (AtomDev::cls holds 16 bits of it).
int rot_class(const hsgen_sys* s, int a)
{
    int c = s->atoms[a].cls & 0xffff;
    while (std::memcmp(s->atoms[s->rot_rep[c]].rot, s->atoms[a].rot, sizeof s->atoms[a].rot)) c += 0x10000;
    return c;
}

int64_t lower(int64_t n) { return n * (n + 1) / 2; }

}  // namespace

namespace {

int64_t mt_size(int64_t nlm) { return roundup(2 * nlm, 4) * roundup(2 * nlm, 16); }

// Device memory of a set-up step.
struct Tmp {
    void* p = nullptr;
    ~Tmp() { if (p) (void)hipFree(p); }
};

// grid.y is at most 65535
constexpr size_t kJobsPerLaunch = 32768;

// T-application tiles of 32 x 64 once they give every CU eight: us, 32 and
// 32 x 64: N_G 235 12 / 15, 600 17 / 17, 1000 157 / 139, 6002 847 / 808.
int tapp_tile(const hsgen_ctx* ctx, const hsgen_sys* s, int64_t gtot)
{
    return (int64_t)s->rt32 * (gtot / 64) >= 8 * (int64_t)std::max(ctx->n_cu, 1) ? 64 : 32;
}

// Real vectors of split precision's T application at a time.
constexpr int64_t kSplitChunkBytes = (int64_t)512 << 20;

}  // namespace

// Kinds, their tables and the T blocks in real harmonics.  rad: the radial
// data as uploaded to s->d_rad.
hsgen_status sphere_setup(hsgen_ctx* ctx, hsgen_sys* s, const RadDev* rad)
{
    const int na = s->natoms;
    // classes of rotations with the same cosines
    std::vector<int> cos_rep, cos_of_rot(s->rot_rep.size());
    for (size_t c = 0; c < s->rot_rep.size(); ++c) {
        const double* rot = s->atoms[s->rot_rep[c]].rot;
        size_t k = 0;
        while (k < cos_rep.size() && !same_cosines(s->atoms[cos_rep[k]].rot, rot)) ++k;
        if (k == cos_rep.size()) cos_rep.push_back(s->rot_rep[c]);
        cos_of_rot[c] = (int)k;
    }
    // kinds, sorted by cosine class, then by overlap group
    struct Kind {
        int cos, group;
        std::vector<int> atoms;
    };
    std::map<std::string, int> id;
    std::map<std::pair<int, std::string>, int> gid;
    std::vector<Kind> members;
    for (int a = 0; a < na; ++a) {
        const auto it = id.emplace(kind_key(s, a, rad, true), (int)members.size());
        if (it.second) {
            const int c = cos_of_rot[rot_class(s, a)];
            const auto g = gid.emplace(std::make_pair(c, kind_key(s, a, rad, false)), (int)gid.size());
            members.push_back(Kind{c, g.first->second, {}});
        }
        members[it.first->second].atoms.push_back(a);
    }
    std::stable_sort(members.begin(), members.end(), [](const Kind& x, const Kind& y) {
        return std::make_pair(x.cos, x.group) < std::make_pair(y.cos, y.group);
    });
    std::vector<OverlapGroup> groups;
    std::vector<KindDev> kinds(members.size());
    std::vector<int32_t> order;
    std::vector<int32_t> steps;
    int64_t ry = 0, rw = 0, rr = 0, rt32 = 0;
    for (size_t i = 0; i < members.size(); ++i) {
        KindDev& k = kinds[i];
        const AtomDev& at = s->atoms[members[i].atoms[0]];
        std::memset(&k, 0, sizeof k);
        k.lmax = at.lmax;
        k.nlm = at.nlm;
        k.r4 = (int32_t)roundup(2 * at.nlm, 4);
        k.rep = members[i].atoms[0];
        k.yoff = (int32_t)ry;
        k.woff = (int32_t)rw;
        k.ldm = (int32_t)roundup(2 * at.nlm, 16);
        k.rt32 = (int32_t)rt32;
        k.first = (int32_t)order.size();
        k.count = (int32_t)members[i].atoms.size();
        k.rmt = at.rmt;
        std::memcpy(k.rot, at.rot, sizeof k.rot);
        k.rsoff = -1;
        if (i == 0 || members[i].group != members[i - 1].group) {
            k.rsoff = (int32_t)rr;
            OverlapGroup g;
            std::memset(&g, 0, sizeof g);
            g.lmax = at.lmax;
            g.rep = k.rep;
            g.rsoff = k.rsoff;
            g.first = k.first;
            g.newdir = i == 0 || members[i].cos != members[i - 1].cos;
            std::memcpy(g.rot, s->atoms[cos_rep[members[i].cos]].rot, sizeof g.rot);
            groups.push_back(g);
            s->h_group_kind.push_back((int32_t)i);
            rr += 2 * (at.lmax + 1);
        }
        groups.back().count += k.count;
        for (int a : members[i].atoms) {
            order.push_back(a);
            for (int r = 0; r < k.r4; r += 4) steps.push_back(k.yoff + r + (r + 4 == k.r4));
        }
        ry += k.r4;
        rw += (int64_t)k.count * k.r4;
        rt32 += ((int64_t)k.count * k.r4 + 31) / 32;
    }
    if (rw > INT32_MAX - 64) return fail(ctx, HSGEN_ERR_UNSUPPORTED, "contraction depth too large");
    s->nksteps = (int)steps.size();
    std::vector<SphereStage> stages((steps.size() + 3) / 4);
    int atoms = 0;
    for (size_t i = 0; i < stages.size(); ++i) {
        SphereStage& g = stages[i];
        std::memset(&g, 0, sizeof g);
        g.atom = -1;
        for (int q = 0; q < 4; ++q) {
            const size_t k = 4 * i + q;
            // past the depth: any row, no end
            int32_t e = k < steps.size() ? steps[k] : 0;
            if (e & 1) {
                if (g.atom >= 0) e |= 2;
                else g.atom = atoms;
                ++atoms;
            }
            g.step[q] = e;
        }
    }
    s->nkinds = (int)kinds.size();
    s->h_order = order;
    s->ngroups = (int)groups.size();
    s->h_groups = groups;
    s->h_group_kind.push_back(s->nkinds);
    s->ldr = (int)rr;
    s->rt32 = (int)rt32;
    // whole stages of 16 rows can be read at the end of a column, from any
    // kind's first row; the odd multiple of 16 spreads the columns over the
    // memory channels
    s->ldy = (roundup(ry, 16) + 16) | 16;
    s->ldw = roundup(rw, 16) | 16;
    // the products address 4 columns of W and 8 of y with 32-bit offsets; longer
    // columns (44 million rows of coefficients) take the general operands
    const char* env = std::getenv("HSGEN_REAL_VECTORS");      // 0: general operands (tests and comparisons)
    s->real_vectors = 64 * s->ldw < (int64_t(1) << 32) && 64 * s->ldy < (int64_t(1) << 32) && !(env && env[0] == '0');
    // T blocks in real harmonics, one per distinct T (h_owner)
    std::vector<int64_t> off(na, 0);
    int64_t total = 0;
    std::vector<int> owners;
    for (int a = 0; a < na; ++a) {
        if (s->h_owner[a] != a) continue;
        off[a] = total;
        total += mt_size(s->atoms[a].nlm);
        owners.push_back(a);
    }
    std::vector<int64_t> mtoff(na);
    for (int i = 0; i < na; ++i) mtoff[i] = off[s->h_owner[order[i]]];
    auto up = [](size_t b) { return (size_t)roundup((int64_t)b, 256); };
    const size_t b_mt = up(sizeof(double2) * (size_t)total), b_k = up(sizeof(KindDev) * kinds.size()),
                 b_g = up(sizeof(OverlapGroup) * groups.size()),
                 b_o = up(sizeof(int32_t) * order.size()), b_s = up(sizeof(SphereStage) * stages.size()),
                 b_m = up(sizeof(int64_t) * mtoff.size());
    HIPCHK(hipMalloc(&s->d_sphere, b_mt + b_k + b_g + b_o + b_s + b_m));
    char* p = (char*)s->d_sphere;
    s->d_mt = (double2*)p;
    s->d_kinds = (KindDev*)(p += b_mt);
    s->d_groups = (OverlapGroup*)(p += b_k);
    s->d_order = (int32_t*)(p += b_g);
    s->d_stages = (SphereStage*)(p += b_o);
    s->d_mtoff = (int64_t*)(p += b_s);
    // the tables in one copy
    std::vector<char> tables(b_k + b_g + b_o + b_s + b_m);
    auto put = [&](const void* dev, const void* src, size_t n) {
        std::memcpy(tables.data() + ((const char*)dev - (const char*)s->d_kinds), src, n);
    };
    put(s->d_kinds, kinds.data(), sizeof(KindDev) * kinds.size());
    put(s->d_groups, groups.data(), sizeof(OverlapGroup) * groups.size());
    put(s->d_order, order.data(), sizeof(int32_t) * order.size());
    put(s->d_stages, stages.data(), sizeof(SphereStage) * stages.size());
    put(s->d_mtoff, mtoff.data(), sizeof(int64_t) * mtoff.size());
    HIPCHK(hipMemcpyAsync(s->d_kinds, tables.data(), tables.size(), hipMemcpyHostToDevice, ctx->stream));
    // the raw blocks and the jobs, only until the matrices are built: in one
    // copy, large ones through the pinned slots
    int64_t raw = 0, most = 0;
    for (int a : owners) {
        raw += 3 * (int64_t)s->atoms[a].nlm * s->atoms[a].nlm;
        most = std::max(most, mt_size(s->atoms[a].nlm));
    }
    const size_t b_raw = sizeof(double2) * (size_t)raw, b_jobs = sizeof(MtJob) * owners.size();
    Tmp t_raw;
    HIPCHK(hipMalloc(&t_raw.p, b_raw + b_jobs));
    double2* d = (double2*)t_raw.p;
    std::vector<MtJob> jobs;
    std::vector<HostCopy> in;
    for (int a : owners) {
        const int64_t n = s->atoms[a].nlm, n2 = n * n;
        const std::vector<std::complex<double>>* src[3] = {&s->h_taa[a], &s->h_tab[a], &s->h_tbb[a]};
        for (int b = 0; b < 3; ++b) in.push_back(copy_run(d + b * n2, src[b]->data(), sizeof(double2) * (size_t)n2));
        jobs.push_back(MtJob{d, d + n2, d + 2 * n2, off[a], (int32_t)n, (int32_t)roundup(2 * n, 4),
                             (int32_t)roundup(2 * n, 16), 0});
        d += 3 * n2;
    }
    in.push_back(copy_run(d, jobs.data(), b_jobs));
    std::vector<char> small;
    if (b_raw + b_jobs < ((size_t)4 << 20)) {
        small.resize(b_raw + b_jobs);
        for (const HostCopy& c : in) std::memcpy(small.data() + (c.dev - (char*)t_raw.p), c.host, c.rows);
        HIPCHK(hipMemcpyAsync(t_raw.p, small.data(), small.size(), hipMemcpyHostToDevice, ctx->stream));
    } else {
        const hsgen_status st = host_copy(ctx, in, false, ctx->stream);
        if (st) return st;
    }
    for (size_t j0 = 0; j0 < jobs.size(); j0 += kJobsPerLaunch)
        HIPCHK(launch_build_mt((const MtJob*)d + j0, (int)std::min(kJobsPerLaunch, jobs.size() - j0), most, s->d_mt,
                               ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return HSGEN_OK;
}

// The matrices of split precision's T application, one per distinct (T,
// divisors of the B rows), and the rows of its W, in atom order without padding.
hsgen_status sphere_split_setup(hsgen_ctx* ctx, hsgen_sys* s)
{
    std::lock_guard<std::mutex> lk(s->m_mu);
    if (s->d_split) return HSGEN_OK;
    const int na = s->natoms, nl = s->nl;
    const std::vector<double> ones(nl, 1.0);
    std::map<std::pair<int, std::vector<double>>, int64_t> seen;
    std::vector<int64_t> src(na), off(na), mtoff;
    std::vector<SplitMtJob> jobs;
    std::vector<double> sq;
    std::vector<int32_t> rows;
    int64_t total = 0, most = 0, mt = 0;
    for (int a = 0; a < na; ++a) {           // Mt in the order sphere_setup lays it out
        if (s->h_owner[a] != a) continue;
        src[a] = mt;
        mt += mt_size(s->atoms[a].nlm);
    }
    for (int a = 0; a < na; ++a) {
        const double* d = s->fold ? s->h_sqrtn.data() + (size_t)a * nl : ones.data();
        const auto it = seen.emplace(std::make_pair(s->h_owner[a], std::vector<double>(d, d + nl)), total);
        off[a] = it.first->second;
        if (!it.second) continue;
        const int n = s->atoms[a].nlm;
        jobs.push_back(SplitMtJob{src[s->h_owner[a]], total, n, (int32_t)roundup(2 * n, 4), (int32_t)roundup(2 * n, 16),
                                  (int32_t)sq.size()});
        sq.insert(sq.end(), d, d + nl);
        total += mt_size(n);
        most = std::max(most, mt_size(n));
    }
    for (int a : s->h_order) {
        const int n2 = 2 * s->atoms[a].nlm;
        mtoff.push_back(off[a]);
        for (int r = 0; r < (int)roundup(n2, 4); ++r) rows.push_back(r < n2 ? 2 * s->atoms[a].off + r : -1);
    }
    const size_t b_mt = (size_t)roundup((int64_t)(sizeof(double2) * (size_t)total), 256),
                 b_m = (size_t)roundup((int64_t)(sizeof(int64_t) * mtoff.size()), 256);
    Tmp keep, t_jobs, t_sq;
    HIPCHK(hipMalloc(&keep.p, b_mt + b_m + sizeof(int32_t) * rows.size()));
    HIPCHK(hipMalloc(&t_jobs.p, sizeof(SplitMtJob) * jobs.size()));
    HIPCHK(hipMalloc(&t_sq.p, sizeof(double) * sq.size()));
    char* p = (char*)keep.p;
    HIPCHK(hipMemcpyAsync(p + b_mt, mtoff.data(), sizeof(int64_t) * mtoff.size(), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(p + b_mt + b_m, rows.data(), sizeof(int32_t) * rows.size(), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(t_jobs.p, jobs.data(), sizeof(SplitMtJob) * jobs.size(), hipMemcpyHostToDevice, ctx->stream));
    HIPCHK(hipMemcpyAsync(t_sq.p, sq.data(), sizeof(double) * sq.size(), hipMemcpyHostToDevice, ctx->stream));
    for (size_t j0 = 0; j0 < jobs.size(); j0 += kJobsPerLaunch)
        HIPCHK(launch_split_mt((const SplitMtJob*)t_jobs.p + j0, (int)std::min(kJobsPerLaunch, jobs.size() - j0), most,
                               (const double*)t_sq.p, s->d_mt, (double2*)p, ctx->stream));
    HIPCHK(hipStreamSynchronize(ctx->stream));
    s->d_split_off = (int64_t*)(p + b_mt);
    s->d_split_rows = (int32_t*)(p + b_mt + b_m);
    s->d_split = keep.p;
    keep.p = nullptr;
    return HSGEN_OK;
}

// W of split precision (rows 2 off_a .. of every column, leading dimension ldw)
// over the ncols padded columns of the k-points ks (k, g, ng, col0 set;
// ks_dev: their device copy).  Column chunks bound the real vectors' memory,
// which with the sample's operands lies where the residues will.
// cols: null, or per k-point kSampleCols columns (past its plane waves the last
// again) whose H and, with do_s, S go to the k-points' H and S, in FP64: H from
// W of the sampled columns and the chunk's real vectors, S by the addition
// theorem.  Sample of 32 atoms at N_G 6002 0.39 ms, of 4 k-points of 1900 plane
// waves 0.65 ms; the products of the operands took 1.03 and 1.32.
hsgen_status sphere_split_w(hsgen_ctx* ctx, hsgen_sys* s, const std::vector<SphereK>& ks, const SphereK* ks_dev,
                            int64_t ncols, double2* W, int64_t ldw, const std::vector<int32_t>* cols, bool do_s)
{
    hsgen_status st = sphere_split_setup(ctx, s);
    if (st) return st;
    int64_t bytes = kSplitChunkBytes;
    if (const char* e = std::getenv("HSGEN_BATCH_BYTES"))   // cap (tuning and tests)
        if (std::strtoull(e, nullptr, 10) > 0) bytes = std::min<int64_t>(bytes, std::strtoll(e, nullptr, 10));
    const int64_t per = 8 * s->ldy + 16 * (int64_t)s->natoms + (cols ? 16 * (int64_t)s->ldr : 0);
    const int64_t chunk = std::min(ncols, std::max<int64_t>(kSphereCols, bytes / per / kSphereCols * kSphereCols));
    auto up = [](size_t b) { return (size_t)roundup((int64_t)b, 256); };
    const int nk = (int)ks.size();
    const int64_t nsmp = cols ? (int64_t)kSampleCols * nk : 0;
    // the chunk's operands and the sample's, in the residues' buffer
    const size_t b_ph = up(sizeof(double2) * (size_t)(chunk * s->natoms)),
                 b_rs = cols ? up(sizeof(double2) * (size_t)(chunk * s->ldr)) : 0,
                 b_y = up(sizeof(double) * (size_t)(chunk * s->ldy));
    const size_t s_k = up(sizeof(SphereK) * nk), s_c = up(sizeof(int32_t) * nsmp), s_g = up(3 * sizeof(int32_t) * nsmp),
                 s_ph = up(sizeof(double2) * nsmp * s->natoms), s_rs = up(sizeof(double2) * nsmp * s->ldr),
                 s_y = up(sizeof(double) * nsmp * s->ldy), s_w = up(sizeof(double2) * nsmp * s->ldw);
    st = ensure(ctx, ctx->oz_res, b_ph + b_rs + b_y + (cols ? s_k + s_c + s_g + s_ph + s_rs + s_y + s_w : 0), false);
    if (st) return st;
    char* const d_ph = (char*)ctx->oz_res.p;
    char* const d_rs = d_ph + b_ph;
    char* const d_y = d_rs + b_rs;
    SphereArgs smp;
    std::vector<SphereK> sk;
    std::vector<char> tables;
    if (cols) {
        // the sampled columns as k-points of their own: operands and W
        SphereLayout l;
        l.gtot = nsmp;
        char* p = d_y + b_y;
        int32_t* g = (int32_t*)(p + s_k + s_c);
        for (int i = 0; i < nk; ++i) {
            SphereK k = ks[i];
            k.ng = std::min(ks[i].ng, kSampleCols);
            k.g = g + 3 * kSampleCols * i;
            k.gd = const_cast<int32_t*>(k.g);
            k.col0 = (int64_t)kSampleCols * i;
            k.gcol0 = (int32_t)l.ngcols;
            l.ngcols += k.ng;
            sk.push_back(k);
        }
        tables.resize(s_k + s_c);
        std::memcpy(tables.data(), sk.data(), sizeof(SphereK) * nk);
        std::memcpy(tables.data() + s_k, cols->data(), sizeof(int32_t) * l.gtot);
        HIPCHK(hipMemcpyAsync(p, tables.data(), tables.size(), hipMemcpyHostToDevice, ctx->stream));
        char* a = p + s_k + s_c + s_g;
        smp = sphere_args(s, l, a, a + s_ph, a + s_ph + s_rs, a + s_ph + s_rs + s_y);
        smp.nk = nk;
        smp.one = ks[0];
        smp.many = ks_dev;
        HIPCHK(launch_sample_g(smp, (const int32_t*)(p + s_k), g, ctx->stream));
        smp.one = sk[0];
        smp.many = (const SphereK*)p;
        HIPCHK(launch_sphere_gen(smp, nullptr, ctx->stream));
        HIPCHK(launch_sphere_tapp(smp, 32, s->rt32, nullptr, ctx->stream));
        smp.smp_g = g;
    }
    for (int64_t c0 = 0; c0 < ncols; c0 += chunk) {
        SphereLayout l;
        l.gtot = std::min(chunk, ncols - c0);
        l.ngcols = l.gtot;
        SphereArgs p = sphere_args(s, l, d_ph, cols ? d_rs : nullptr, d_y, W + c0 * ldw);
        p.mt = (const double2*)s->d_split;
        p.mtoff = s->d_split_off;
        p.rowdst = s->d_split_rows;
        p.cbase = c0;
        p.ldw = ldw;
        p.nk = (int32_t)ks.size();
        p.one = ks[0];
        p.many = ks_dev;
        HIPCHK(launch_sphere_gen(p, nullptr, ctx->stream));
        HIPCHK(launch_sphere_tapp(p, tapp_tile(ctx, s, l.gtot), s->rt32, nullptr, ctx->stream));
        if (cols) {
            p.smp_W = smp.W;
            p.smp_ldw = smp.ldw;
            p.smp_ph = smp.ph;
            p.smp_rs = smp.rs;
            p.smp_g = smp.smp_g;
            p.smp_gtot = smp.gtot;
            HIPCHK(launch_sample(p, true, do_s, ctx->stream));
        }
    }
    // the host tables must outlive their copy
    if (cols) HIPCHK(hipStreamSynchronize(ctx->stream));
    return HSGEN_OK;
}

// Operand layout of a call over k-points of ngs[] plane waves (each > 0).
SphereLayout sphere_layout(const hsgen_ctx* ctx, const hsgen_sys* s, const std::vector<int>& ngs, bool do_h)
{
    SphereLayout l;
    const int ncu = std::max(ctx->n_cu, 1);
    int64_t t64 = 0;
    for (int ng : ngs) {
        t64 += lower((ng + 63) / 64);
        l.gtot += roundup(ng, kSphereCols);
    }
    // H tiles by the 64 x 64 ones per CU: smaller tiles share a small triangle
    // more evenly, larger ones read less.  Measured, us (32 atoms, lmax 10; N_G,
    // tiles of 32, 32 x 64, 64): 1000 410 / 534 / 541, 2003 1046 / 1265 / 1468,
    // 3001 (24 atoms, lmax 8-12) 1846 / 1720 / 1864, 4000 4231 / 3946 / 3854,
    // 6002 9583 / 8625 / 8566.
    l.htile = t64 < 3 * (int64_t)ncu ? 32 : t64 < 6 * (int64_t)ncu ? 48 : 64;
    // Where 16 x 32 tiles leave every CU at most one, H is one chain of MFMAs per
    // wave: real and imaginary parts then go to waves of their own.  Calls, us: 2
    // atoms of lmax 8 at N_G 235 49 -> 47, 16 of lmax 12 at 100 190 -> 166, 64 of
    // lmax 8 at 100 317 -> 268; with two tiles per CU (600) both take the same.
    int64_t t32 = 0;
    for (int ng : ngs) t32 += lower((ng + 31) / 32);
    if (2 * t32 <= ncu) l.htile = 16;
    l.ttile = tapp_tile(ctx, s, l.gtot);
    l.stile = overlap_tile_size(t64, ncu);
    const int hc = l.htile <= 32 ? 32 : 64;
    for (int ng : ngs) {
        l.nsquares += lower((ng + hc - 1) / hc);
        l.nstiles += lower((ng + l.stile - 1) / l.stile);
        l.ngcols += ng;
    }
    const size_t g = (size_t)l.gtot;
    l.b_ph = sizeof(double2) * g * (size_t)s->natoms;
    l.b_rs = sizeof(double2) * g * (size_t)s->ldr;
    l.b_y = do_h ? sizeof(double) * g * (size_t)s->ldy : 0;
    l.b_w = do_h ? sizeof(double2) * g * (size_t)s->ldw : 0;
    return l;
}

// The operands of a call in the buffers that the general ones have too (a
// context that uses both holds one set): W in W, the others in Z.
hsgen_status sphere_operands(hsgen_ctx* ctx, const SphereLayout& l, bool do_h, SphereOperands& o)
{
    auto up = [](size_t b) { return (size_t)roundup((int64_t)b, 256); };
    hsgen_status st = ensure(ctx, ctx->Z, up(l.b_ph) + up(l.b_rs) + l.b_y, false);
    if (st) return st;
    if (do_h && (st = ensure(ctx, ctx->W, l.b_w, false))) return st;
    o.ph = ctx->Z.p;
    o.rs = (char*)o.ph + up(l.b_ph);
    o.y = do_h ? (char*)o.rs + up(l.b_rs) : nullptr;
    o.w = do_h ? ctx->W.p : nullptr;
    return HSGEN_OK;
}

SphereArgs sphere_args(const hsgen_sys* s, const SphereLayout& l, void* ph, void* rs, void* y, void* w)
{
    SphereArgs p;
    std::memset(&p, 0, sizeof p);
    p.kinds = s->d_kinds;
    p.groups = s->d_groups;
    p.atoms = s->d_atoms;
    p.order = s->d_order;
    p.rad = s->d_rad;
    p.ynorm = s->d_ynorm;
    std::memcpy(p.bmat, s->bmat, sizeof p.bmat);
    p.vol_prefac = s->vol_prefac;
    p.natoms = s->natoms;
    p.nkinds = s->nkinds;
    p.ngroups = s->ngroups;
    p.max_lmax = s->max_lmax;
    p.nl = s->nl;
    p.L = s->L;
    p.chunk = sphere_chunk(s->nl, s->L);
    p.nk = 1;
    p.ngcols = (int32_t)l.ngcols;
    p.gtot = l.gtot;
    p.tcols = (int32_t)l.gtot;
    p.ph = (double2*)ph;
    p.rs = (double2*)rs;
    p.ldr = s->ldr;
    p.y = (double*)y;
    p.W = (double2*)w;
    p.ldy = s->ldy;
    p.ldw = s->ldw;
    p.mt = s->d_mt;
    p.mtoff = s->d_mtoff;
    p.stages = s->d_stages;
    p.nksteps = s->nksteps;
    p.nsquares = (int32_t)l.nsquares;
    return p;
}

// The k-points of a call in layout order; gs, H, S device pointers.
std::vector<SphereK> sphere_ks(const SphereLayout& l, const std::vector<const hsgen_kpoint*>& kps,
                               const std::vector<const int32_t*>& gs, const std::vector<double2*>& H,
                               const std::vector<double2*>& S, const std::vector<int64_t>& ldH,
                               const std::vector<int64_t>& ldS)
{
    std::vector<SphereK> ks(kps.size());
    const int hc = l.htile <= 32 ? 32 : 64;
    int64_t col = 0, g = 0, st = 0, hp = 0;
    for (size_t i = 0; i < kps.size(); ++i) {
        SphereK& k = ks[i];
        std::memset(&k, 0, sizeof k);
        for (int q = 0; q < 3; ++q) k.k[q] = kps[i]->k[q];
        k.g = gs[i];
        k.gd = const_cast<int32_t*>(gs[i]);
        k.H = H[i];
        k.S = S[i];
        k.ldH = ldH[i];
        k.ldS = ldS[i];
        k.col0 = col;
        k.ng = kps[i]->ng;
        k.gcol0 = (int32_t)g;
        k.stile0 = (int32_t)st;
        k.hsquare0 = (int32_t)hp;
        col += roundup(k.ng, kSphereCols);
        g += k.ng;
        st += lower((k.ng + l.stile - 1) / l.stile);
        hp += lower((k.ng + hc - 1) / hc);
    }
    return ks;
}

// The G list of a one-k-point call: device memory as it is; a short host list
// goes into the context's pinned buffer, which the generator reads and copies
// to dev (a copy on the stream costs 12 us); a longer one is copied to dev.
// dev: room for the list in device memory, or null to take ctx->g.
hsgen_status sphere_g(hsgen_ctx* ctx, const hsgen_kpoint* kp, int32_t* dev, SphereK& k)
{
    if (is_device_ptr(kp->g)) {
        k.g = kp->g;
        k.gd = const_cast<int32_t*>(kp->g);
        return HSGEN_OK;
    }
    const size_t bytes = sizeof(int32_t) * 3 * (size_t)kp->ng;
    if (!dev) {
        const hsgen_status st = ensure(ctx, ctx->g, bytes, false);
        if (st) return st;
        dev = (int32_t*)ctx->g.p;
    }
    k.gd = dev;
    if (kp->ng <= kPinnedG) {
        std::memcpy((char*)ctx->pin + kPinStamps, kp->g, bytes);
        k.g = (const int32_t*)((char*)ctx->pin_dev + kPinStamps);
    } else {
        HIPCHK(hipMemcpyAsync(dev, kp->g, bytes, hipMemcpyHostToDevice, ctx->stream));
        k.g = dev;
    }
    return HSGEN_OK;
}

// Bytes of the phases and radial factors of groups g0 .. g1 - 1.
static size_t part_bytes(const hsgen_sys* s, const SphereLayout& l, int g0, int g1)
{
    const int atoms = (g1 < s->ngroups ? s->h_groups[g1].first : s->natoms) - s->h_groups[g0].first;
    const int rows = (g1 < s->ngroups ? s->h_groups[g1].rsoff : s->ldr) - s->h_groups[g0].rsoff;
    return sizeof(double2) * (size_t)l.gtot * ((size_t)atoms + rows);
}

bool sphere_parts(const hsgen_sys* s, SphereLayout& l, bool do_h, bool do_s, size_t bytes)
{
    for (int g0 = 0; do_s && g0 < s->ngroups;) {
        int g1 = g0 + 1;
        while (g1 < s->ngroups && part_bytes(s, l, g0, g1 + 1) <= bytes) ++g1;
        if (part_bytes(s, l, g0, g1) > bytes) return false;
        l.sparts.push_back(g0);
        g0 = g1;
    }
    l.sparts.push_back(s->ngroups);
    const size_t column = sizeof(double2) * (size_t)s->ldw;
    if (l.b_ph + l.b_y >= bytes) return !do_h;
    l.wcols = std::min(l.gtot, (int64_t)((bytes - l.b_ph - l.b_y) / column) / kSphereCols * kSphereCols);
    return !do_h || l.wcols > 0;
}

// The launches of one k-point in parts: S over its groups in turn, then H from
// W a few columns at a time, in the same memory.  The same kernels in the same
// order of sums, so the same bits.
static hipError_t sphere_launch_parts(const SphereArgs& p, const SphereLayout& l, const hsgen_sys* s, bool do_h, bool do_s,
                                      hipEvent_t stop, hipStream_t st)
{
    if (!do_h && !do_s) return stop ? hipEventRecord(stop, st) : hipSuccess;
    hipError_t e = hipSuccess;
    const int nparts = do_s ? (int)l.sparts.size() - 1 : 0;
    for (int i = 0; i < nparts; ++i) {
        const int g0 = l.sparts[i], g1 = l.sparts[i + 1];
        const int first = s->h_groups[g0].first, rs0 = s->h_groups[g0].rsoff;
        SphereArgs q = p;
        q.y = nullptr;
        q.groups += g0;
        q.ngroups = g1 - g0;
        q.kinds += s->h_group_kind[g0];
        q.nkinds = s->h_group_kind[g1] - s->h_group_kind[g0];
        q.order += first;
        q.natoms = (g1 < s->ngroups ? s->h_groups[g1].first : s->natoms) - first;
        q.ldr = (g1 < s->ngroups ? s->h_groups[g1].rsoff : s->ldr) - rs0;
        // rows of the whole call: the part's begin at rs0, its atoms at `first`
        q.rs = (double2*)((uintptr_t)(p.ph + (int64_t)q.natoms * l.gtot) - sizeof(double2) * (size_t)rs0);
        if ((e = launch_sphere_gen(q, nullptr, st)) != hipSuccess) return e;
        q.ph = (double2*)((uintptr_t)p.ph - sizeof(double2) * (size_t)first * (size_t)l.gtot);
        q.sadd = i > 0;
        e = launch_overlap_part(q, i + 1 < nparts || do_h ? nullptr : stop, st);
        if (e != hipSuccess) return e;
    }
    if (!do_h) return e;
    SphereArgs q = p;
    q.rs = nullptr;
    q.y = (double*)((char*)p.ph + l.b_ph);
    double2* const w = (double2*)((char*)q.y + l.b_y);
    e = launch_sphere_gen(q, nullptr, st);
    for (int64_t c0 = 0; c0 < l.gtot && e == hipSuccess; c0 += l.wcols) {
        const int64_t n = std::min(l.wcols, l.gtot - c0);
        SphereArgs t = q;
        t.tcols = (int32_t)n;
        t.y += c0 * p.ldy;
        t.ph += c0;
        t.W = w;
        if ((e = launch_sphere_tapp(t, l.ttile, s->rt32, nullptr, st)) != hipSuccess) return e;
        t = q;
        t.W = (double2*)((uintptr_t)w - sizeof(double2) * (size_t)(c0 * p.ldw));   // addressed by the call's columns
        t.hcol0 = (int32_t)c0;
        t.hcol1 = (int32_t)(c0 + n);
        e = launch_sphere_h_part(t, c0 + n < l.gtot ? nullptr : stop, st);
    }
    return e;
}

// The launches of one call.  stop: null, or an event that takes the end of the
// last of them.
hipError_t sphere_launch(const SphereArgs& p, const SphereLayout& l, const hsgen_sys* s, bool do_h, bool do_s,
                         hipEvent_t stop, hipStream_t st)
{
    if (!l.sparts.empty()) return sphere_launch_parts(p, l, s, do_h, do_s, stop, st);
    const hipEvent_t none = nullptr, last = stop;
    hipError_t e = launch_sphere_gen(p, do_h || do_s ? none : last, st);
    if (e == hipSuccess && do_h) e = launch_sphere_tapp(p, l.ttile, s->rt32, none, st);
    if (e != hipSuccess) return e;
    if (do_h && do_s && l.htile <= 32 && l.stile <= (l.htile == 16 ? 16 : 32))
        return launch_sphere_hs(p, l.htile, l.stile, l.nstiles, last, st);
    if (do_h) e = launch_sphere_h(p, l.htile, do_s ? none : last, st);
    if (e == hipSuccess && do_s) e = launch_overlap(p, l.stile, l.nstiles, last, st);
    return e;
}

// A one-k-point call on device matrices: launches, wait, report.
hsgen_status sphere_run(hsgen_ctx* ctx, const hsgen_sys* s, const SphereLayout& l, SphereArgs& p, int flags, int tile,
                        hsgen_report* rep)
{
    const bool do_h = !(flags & HSGEN_SKIP_H), do_s = !(flags & HSGEN_SKIP_S);
    const SphereK& k = p.one;
    p.stamp = rep ? (uint64_t*)ctx->pin_dev : nullptr;
    if (rep) HIPCHK(hipEventRecord(ctx->ev[0], ctx->stream));
    const hipError_t le = sphere_launch(p, l, s, do_h, do_s, ctx->ev[1], ctx->stream);
    if (le != hipSuccess) {
        (void)hipStreamSynchronize(ctx->stream);    // nothing reads the pinned buffer after the call
        HIPCHK(le);
    }
    hipEvent_t end = ctx->ev[1];
    if (flags & HSGEN_FILL_UPPER) {
        if (do_h) HIPCHK(launch_fill_upper(k.H, k.ldH, k.ng, ctx->stream));
        if (do_s) HIPCHK(launch_fill_upper(k.S, k.ldS, k.ng, ctx->stream));
        end = ctx->ev[2];
        HIPCHK(hipEventRecord(end, ctx->stream));
    }
    HIPCHK(hipEventSynchronize(end));
    if (!rep) return HSGEN_OK;
    // the whole by events, the kernels' starts by the wall clock: a call of 50 us
    // took 14 us more with events around each kernel
    float total = 0;
    HIPCHK(hipEventElapsedTime(&total, ctx->ev[0], end));
    const volatile uint64_t* t = (const volatile uint64_t*)ctx->pin;
    auto ms = [&](int from, int to) { return (double)(int64_t)(t[to] - t[from]) * ctx->ms_per_tick; };
    rep->ms_total = total;
    rep->ms_abgen = do_h ? ms(0, 1) : do_s ? ms(0, 3) : total;
    rep->ms_tmul = do_h ? ms(1, 2) : 0.0;
    rep->ms_contract = do_h || do_s ? std::max(0.0, total - rep->ms_abgen - rep->ms_tmul) : 0.0;
    rep->ng = k.ng;
    rep->kdim = s->kdim;
    rep->flops_alg = 16.0 * (double)k.ng * k.ng * s->kdim + 32.0 * (double)k.ng * (double)s->sum_nlm2;
    rep->bytes_abgen = sphere_gen_bytes(s) * k.ng;
    rep->tile_used = tile;
    return HSGEN_OK;
}

}  // namespace hsgen
