// FP64 kernels of the path from a system description to H and S that use the
// form of the matching coefficients: a phase per atom times real numbers that
// atoms of one kind share (sphere.h).
#include <algorithm>
#include <type_traits>

#include <hip/hip_ext.h>

#include "sphere.h"
#include "sphere_dev.h"

namespace hsgen {

namespace {

// Launch, with the event that the call waits for attached to the kernel itself.
template <class... A>
hipError_t launch(void (*k)(A...), dim3 grid, int threads, size_t lds, hipEvent_t stop, hipStream_t st, A... args)
{
    if (grid.x == 0) return hipSuccess;
    if (lds > 64 * 1024) {
        // per launch: the attribute is per device
        const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    if (stop)
        hipExtLaunchKernelGGL(k, grid, dim3(threads), lds, st, nullptr, stop, 0, args...);
    else
        hipLaunchKernelGGL(k, grid, dim3(threads), lds, st, args...);
    return hipGetLastError();
}

// The kernel's start, by its first workgroup, for the report: events between
// the kernels of a call cost 5 us each.
__device__ __forceinline__ void stamp(const SphereArgs& p, int which)
{
    if (p.stamp && blockIdx.x == 0 && threadIdx.x == 0) p.stamp[which] = (uint64_t)wall_clock64();
}

// Largest i in [0, n) with key(i) <= v; key ascending, key(0) <= v.
template <class Key>
__device__ __forceinline__ int find_last(int n, int v, Key key)
{
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (key(mid) <= v) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Row of the lower triangle that element t of its row-by-row list is in.
__device__ __forceinline__ int tri_row(int t)
{
    int r = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((int64_t)(r + 1) * (r + 2) / 2 <= t) ++r;
    while ((int64_t)r * (r + 1) / 2 > t) --r;
    return r;
}

struct Reciprocals {
    double v[kMaxLmax + 1];
};
constexpr Reciprocals reciprocals()
{
    Reciprocals r{};
    for (int i = 1; i <= kMaxLmax; ++i) r.v[i] = 1.0 / i;
    return r;
}
__constant__ const Reciprocals kReciprocal = reciprocals();

// Real harmonics of one m >= 0 by the ylm4 recurrences (ylm4.f:194-217):
// Y_l0, and for m > 0 Re and Im of Y_lm at l(l+1)+m and l(l+1)-m, so that
// conj(Y_lm) = re - i im and conj(Y_l,-m) = (-1)^m (re + i im).
__device__ inline void ylm_real(int m, int lmax, const DirAngles& dir, const double* __restrict__ ynorm, double* yl)
{
    double cm = 1.0, sm = 0.0;
    if (m >= 1) {
        double cmm1 = 1.0, smm1 = 0.0;
        cm = dir.cph;
        sm = dir.sph;
        const double cph2 = dir.cph + dir.cph;
        for (int mm = 2; mm <= m; ++mm) {
            const double cn = cph2 * cm - cmm1;
            const double sn = cph2 * sm - smm1;
            cmm1 = cm;
            smm1 = sm;
            cm = cn;
            sm = sn;
        }
    }
    double fac = 1.0;
    for (int mm = 0; mm < m; ++mm) {
        fac = -(mm + mm - 1) * fac;
        fac = fac * dir.sth;
    }
    fac = -(m + m - 1) * fac;
    double pl2 = 0.0, pl1 = fac;
    for (int l = m; l <= lmax; ++l) {
        double pv;
        if (l == m) pv = fac;
        else if (l == m + 1) pv = (m + m + 1) * dir.cth * fac;
        else {
            // divided by l - m: the product with its reciprocal, corrected
            const double num = (l + l - 1) * dir.cth * pl1 - (l + m - 1) * pl2;
            const double rec = kReciprocal.v[l - m];
            pv = num * rec;
            pv = __builtin_fma(__builtin_fma(-(double)(l - m), pv, num), rec, pv);
        }
        if (l > m) {
            pl2 = pl1;
            pl1 = pv;
        }
        const int lm0 = l * (l + 1);
        const double v = ynorm[lm0 + m] * pv;
        if (m == 0) {
            yl[lm0] = v;
        } else {
            yl[lm0 + m] = v * cm;
            yl[lm0 - m] = v * sm;
        }
    }
}

// a b - c d without the rounding of c d, which counts where they cancel.
__device__ __forceinline__ double product_difference(double a, double b, double c, double d)
{
    const double cd = c * d;
    return __builtin_fma(a, b, -cd) - __builtin_fma(c, d, -cd);
}

}  // namespace

// ---------------------------------------------------------------------------
// Generator: one workgroup per plane wave.  Phases of all atoms, then per
// chunk of kinds the Bessel values and the direction (one lane per kind), the
// real radial factors a_l, b_l (A and B without phase and harmonic), the real
// harmonics (one lane per kind and m) and, with y, the real vectors
// [a_l Y_lm; b_l Y_lm].
// ---------------------------------------------------------------------------
template <bool kSplit>
__global__ __launch_bounds__(256) void k_sphere_gen(SphereArgs p)
{
    extern __shared__ double smem[];
    stamp(p, 0);
    const int tid = threadIdx.x;
    const int nl = p.nl;
    const int L = p.L;
    double* s_bes = smem;                              // [chunk][2 nl]  fj, dfj
    double2* s_ab = (double2*)(s_bes + p.chunk * 2 * nl);   // [chunk][nl] (a_l, b_l)
    double* s_y = (double*)(s_ab + p.chunk * nl);      // [chunk][L]     real harmonics
    DirAngles* s_dir = (DirAngles*)(s_y + p.chunk * L);     // [chunk]
    unsigned char* s_l = (unsigned char*)(s_dir + p.chunk); // [L]       l of lm
    // the k-point and the plane wave: every column of the chunk, padding as
    // zeros (kSplit), or the plane waves of all k-points
    const int c = kSplit ? (int)p.cbase + (int)blockIdx.x : (int)blockIdx.x;
    int ki = 0;
    if (p.nk > 1)
        ki = find_last(p.nk, c, [&](int i) { return kSplit ? (int)p.many[i].col0 : p.many[i].gcol0; });
    const SphereK k = p.nk > 1 ? p.many[ki] : p.one;
    const int gi = c - (kSplit ? (int)k.col0 : k.gcol0);
    const int64_t col = kSplit ? blockIdx.x : k.col0 + gi;
    if (kSplit && gi >= k.ng) {
        for (int64_t r = tid; r < p.ldy; r += blockDim.x) p.y[col * p.ldy + r] = 0.0;
        for (int a = tid; a < p.natoms; a += blockDim.x) p.ph[(int64_t)a * p.gtot + col] = make_double2(0.0, 0.0);
        return;
    }
    const int g0 = k.g[3 * gi + 0], g1 = k.g[3 * gi + 1], g2 = k.g[3 * gi + 2];
    if (!kSplit && k.gd != k.g && tid < 3) k.gd[3 * gi + tid] = tid == 0 ? g0 : tid == 1 ? g1 : g2;
    const double K0 = k.k[0] + g0;
    const double K1 = k.k[1] + g1;
    const double K2 = k.k[2] + g2;
    const double c0 = p.bmat[0] * K0 + p.bmat[3] * K1 + p.bmat[6] * K2;
    const double c1 = p.bmat[1] * K0 + p.bmat[4] * K1 + p.bmat[7] * K2;
    const double c2 = p.bmat[2] * K0 + p.bmat[5] * K1 + p.bmat[8] * K2;
    const double Knorm = sqrt(c0 * c0 + c1 * c1 + c2 * c2);

    for (int lm = tid; lm < L; lm += blockDim.x) s_l[lm] = (unsigned char)l_of_lm(lm);
    // phases e^{i 2 pi K.tau}; the lanes with the Bessel recurrences come last
    for (int a = blockDim.x - 1 - tid; a < p.natoms; a += blockDim.x) {
        const AtomDev& at = p.atoms[p.order[a]];
        // the fraction of K.tau, term by term: its rounding, not that of the whole
        const double kq[6] = {(double)g0, (double)g1, (double)g2, k.k[0], k.k[1], k.k[2]};
        double f = 0.0, rest = 0.0;
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const double v = kq[q] * at.pos[q % 3];
            rest += __builtin_fma(kq[q], at.pos[q % 3], -v);
            f += v - rint(v);
        }
        f += rest;
        double ps, pc;
        sincospi(2.0 * (f - rint(f)), &ps, &pc);
        p.ph[(int64_t)a * p.gtot + col] = make_double2(pc, ps);
    }
    for (int k0 = 0; k0 < p.nkinds; k0 += p.chunk) {
        const int nk = min(p.chunk, p.nkinds - k0);
        if (tid < nk) {
            double* fj = s_bes + tid * 2 * nl;
            bessel_lds(p.max_lmax, p.kinds[k0 + tid].rmt * Knorm, fj, fj + nl);
        } else if (p.y && tid >= 64 && tid - 64 < nk) {
            s_dir[tid - 64] = dir_angles(p.kinds[k0 + tid - 64].rot, K0, K1, K2);
        }
        __syncthreads();
        for (int q = tid; q < nk * nl; q += blockDim.x) {
            const int t = q / nl;
            const int l = q - t * nl;
            const KindDev& kd = p.kinds[k0 + t];
            if (l > kd.lmax) continue;
            const double* fj = s_bes + t * 2 * nl;
            const double* dfj = fj + nl;
            const RadDev m = p.rad[(int64_t)kd.rep * nl + l];
            const double pref = p.vol_prefac * m.inv_wronk;
            const double au = product_difference(m.dE_u * Knorm, dfj[l], m.dE_u_dr, fj[l]);
            const double bu = product_difference(m.u_dr, fj[l], m.u * Knorm, dfj[l]);
            const double2 ab = make_double2(pref * au, pref * bu);
            s_ab[t * nl + l] = ab;
            if (p.rs && kd.rsoff >= 0) {
                // as they are, and with the weights of S
                double2* r = p.rs + col * p.ldr + kd.rsoff + l;
                const double wl = (2 * l + 1) / (4.0 * kPi);
                const double wb = wl * m.dE_u_norm;
                r[0] = ab;
                r[kd.lmax + 1] = make_double2(wl * ab.x, wb * ab.y);
            }
        }
        if (p.y) {
            // from the other end: the first waves have the radial factors
            for (int q = blockDim.x - 1 - tid; q < nk * nl; q += blockDim.x) {
                const int t = q / nl;
                const int m = q - t * nl;
                if (m <= p.kinds[k0 + t].lmax) ylm_real(m, p.kinds[k0 + t].lmax, s_dir[t], p.ynorm, s_y + t * L);
            }
            __syncthreads();
            double* yc = p.y + col * p.ldy;
            for (int t = 0; t < nk; ++t) {
                const KindDev& kd = p.kinds[k0 + t];
                for (int r = tid; r < kd.r4; r += blockDim.x) {
                    double v = 0.0;
                    if (r < kd.nlm) v = s_ab[t * nl + s_l[r]].x * s_y[t * L + r];
                    else if (r < 2 * kd.nlm) v = s_ab[t * nl + s_l[r - kd.nlm]].y * s_y[t * L + r - kd.nlm];
                    yc[kd.yoff + r] = v;
                }
            }
        }
        __syncthreads();
    }
}

static size_t sphere_gen_lds(int chunk, int nl, int L)
{
    return sizeof(double) * (size_t)chunk * (2 * nl + 2 * nl + L) + sizeof(DirAngles) * (size_t)chunk + (size_t)L;
}

// Kinds per pass of the generator: as many as 32 KiB of LDS hold, at most 16
// (5 workgroups per CU; 16 kinds of lmax 12 take 28 KiB).
int sphere_chunk(int nl, int L)
{
    int chunk = 16;
    while (chunk > 1 && sphere_gen_lds(chunk, nl, L) > 32 * 1024) chunk /= 2;
    return chunk;
}

hipError_t launch_sphere_gen(const SphereArgs& p, hipEvent_t stop, hipStream_t st)
{
    const size_t lds = sphere_gen_lds(p.chunk, p.nl, p.L);
    return launch(p.rowdst ? k_sphere_gen<true> : k_sphere_gen<false>, dim3(p.ngcols), 256, lds, stop, st, p);
}

// ---------------------------------------------------------------------------
// S by the addition theorem.  One workgroup per lower tile of 16 M x 16 M,
// M x MJ elements per thread (rows tx + 16 m: stores of 16 consecutive rows).
// Per group, per element: the Legendre sum (6 FP64 operations per l) and 4 fused
// operations per atom, against 8 (2 L) per atom of the contraction S = Y^H Y it
// replaces.  Vector FP64 takes a third of its time, the start and end of a tile
// (one workgroup of 64 x 64 per CU) most of the rest: a group's radial factors
// and phases go straight into LDS while the group before is summed, and the
// factors of the next l are read ahead.  Measured: 5.5 ms at N_G 12007 (128
// atoms of 8 kinds, lmax 12; 6.0 with the loads in front of each group), where
// the contraction took about 350 ms; 0.52 (0.59) ms at 6002 (32 atoms, 4 kinds,
// lmax 10).  Atoms whose rotations leave the cosines as they are share a group:
// at N_G 3001 24 atoms of 3 types and 22 rotations took 0.83 ms as 24 sums, 0.12
// ms as 3.
//
// P_l comes from t = 1 - |cos| = |n -+ n'|^2 / 2, formed from the difference
// (sum, where the cosine is negative) of the unit vectors, by
//   D_l+1 = D_l - (2l+1) t P_l,  P_l+1 = P_l + D_l+1 / (l+1):
// near parallel and antiparallel vectors, where P_l varies fastest, t keeps
// its relative accuracy, which a cosine would lose.  Odd l carry the sign.
// ---------------------------------------------------------------------------
namespace {

typedef double v2d __attribute__((ext_vector_type(2)));

// s_waitcnt immediate: at most n vector-memory operations outstanding and, with
// lgkm, no LDS or scalar ones (vmcnt bits [3:0] and [15:14], expcnt [6:4],
// lgkmcnt [11:8]).
constexpr int wait_vm(int n, bool lgkm)
{
    return (n & 15) | (7 << 4) | ((lgkm ? 0 : 15) << 8) | ((n >> 4) << 14);
}

struct LegendreCoef {
    double v[kMaxLmax + 1];
};
constexpr LegendreCoef legendre_coef()
{
    LegendreCoef c{};
    for (int l = 0; l <= kMaxLmax; ++l) c.v[l] = 1.0 / (double)(l + 1);
    return c;
}
__constant__ const LegendreCoef kLegendre = legendre_coef();

// 1 KiB into LDS: lane i's 16 bytes at dst + 16 i
__device__ __forceinline__ void load_lds(const void* src, char* dst)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

}  // namespace

// Wave-uniform values the compiler is to keep in scalar registers.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <int M, int MJ>
struct OverlapTile {
    static constexpr int T = 16 * M, TY = T / MJ, NT = 16 * TY, NW = NT / 64;
    static constexpr int kAtoms = M == 2 ? 4 : 8;        // whose phases are staged at a time
    static constexpr int kPlane = T * 256;               // 16 values of l of T columns
    static constexpr int kPhases = 2 * kAtoms * T * 16;  // of the rows, of the columns
    // two buffers of each; planes: of 16 values of l
    static constexpr int lds(int planes) { return 4 * planes * kPlane + 2 * kPhases; }
};

// kSample: the sampled columns of S, all rows of a chunk's columns.
// kAdd: S of some of the groups, added (p.sadd) to that of the ones before.
template <int M, int MJ, bool kAhead, bool kSample, bool kAdd = false>
__device__ __forceinline__ void overlap_tile(const SphereArgs& p, int blk, char* lds)
{
    // one rounding per written operation: every tile gives the same bits
#pragma clang fp contract(off)
    using Ov = OverlapTile<M, MJ>;
    constexpr int T = Ov::T, TY = Ov::TY, NW = Ov::NW, kAtoms = Ov::kAtoms;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = uni(tid >> 6);
    const int tx = tid & 15, ty = tid >> 4;
    const SphereK* kp = &p.one;
    int I0, J0;                           // first row, first column (sampled: among the samples)
    int64_t ci, cj;                       // their columns of the operands
    if constexpr (kSample) {
        constexpr int kRow = kSampleCols / T;
        const int tc = blk / kRow;
        const int c = (int)p.cbase + tc * T;
        const int ki = p.nk > 1 ? find_last(p.nk, c, [&](int i) { return (int)p.many[i].col0; }) : 0;
        if (p.nk > 1) kp = p.many + ki;
        I0 = c - (int)kp->col0;
        J0 = (blk - tc * kRow) * T;
        if (I0 >= kp->ng || J0 >= min(kp->ng, kSampleCols)) return;
        ci = tc * T;
        cj = ki * kSampleCols + J0;
    } else {
        if (p.nk > 1) kp = p.many + find_last(p.nk, blk, [&](int i) { return p.many[i].stile0; });
        const int tile = blk - kp->stile0;
        const int bi = tri_row(tile);
        const int bj = tile - (int)((int64_t)bi * (bi + 1) / 2);
        I0 = bi * T;
        J0 = bj * T;
        ci = kp->col0 + I0;
        cj = kp->col0 + J0;
    }
    const int ng = kp->ng;
    // the columns' operands
    const double2* const rs_j = kSample ? p.smp_rs : p.rs;
    const double2* const ph_j = kSample ? p.smp_ph : p.ph;
    const int64_t gtot_j = kSample ? p.smp_gtot : p.gtot;
    const int planes = (p.nl + 15) / 16;
    char* const ph0 = lds + 4 * planes * Ov::kPlane;
    // constant address space: the groups come by scalar loads
    typedef __attribute__((address_space(4))) const OverlapGroup* cgroups;
    const cgroups groups = (cgroups)(const void*)p.groups;

    // Radial factors of group kk (rows: as they are, columns: weighted):
    // [buffer][side][plane][T][16], value l of column c at l ^ (c % 16) so that
    // 16 columns hit distinct banks; past the last l that one again.
    auto load_radial = [&](int kk, int buf) {
        const auto& kd = groups[kk];
        const int nlk = kd.lmax + 1;
        for (int w = wave; w < 2 * planes * (T / 4); w += NW) {
            const int part = w / (T / 4), c0 = 4 * (w % (T / 4));
            const int side = part >= planes, plane = part - side * planes;
            const int c = c0 + (lane >> 4), l = plane * 16 + ((lane & 15) ^ (c & 15));
            const double2* src = (side ? rs_j + (cj + c) * p.ldr : p.rs + (ci + c) * p.ldr) + kd.rsoff + side * nlk +
                                 min(l, nlk - 1);
            load_lds(src, lds + (buf * 2 * planes + part) * Ov::kPlane + c0 * 256);
        }
    };
    // Phases of kAtoms atoms from `first` on, n of them: [buffer][side][atom][T]
    auto load_phases = [&](int first, int n, int buf) {
        for (int w = wave; w < 2 * kAtoms * T / 64; w += NW) {
            const int e = w * 64 + lane;
            const int side = w * 64 >= kAtoms * T;
            const int a = min(e / T % kAtoms, n - 1), c = e % T;
            load_lds((side ? ph_j + (int64_t)(first + a) * gtot_j + cj : p.ph + (int64_t)(first + a) * p.gtot + ci) + c, ph0 + buf * Ov::kPhases + w * 1024);
        }
    };

    double sr[M][MJ], si[M][MJ], t[M][MJ], sg[M][MJ], rad[M][MJ], fr[M][MJ], fi[M][MJ];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int n = 0; n < MJ; ++n) {
            sr[m][n] = 0.0;
            si[m][n] = 0.0;
            t[m][n] = 0.0;
            sg[m][n] = 1.0;
            if constexpr (kAdd) {
                const int i = I0 + tx + 16 * m, j = J0 + ty + TY * n;
                if (p.sadd && i < ng && i >= j) {
                    const double2 v = kp->S[(int64_t)j * kp->ldS + i];
                    sr[m][n] = v.x;
                    si[m][n] = v.y;
                }
            }
        }
    // 1 / (l + 1) in lane l: read from there, not by a load that a step would wait for
    const double inv_l = kLegendre.v[min(lane, kMaxLmax)];
    const int inv_lo = __double2loint(inv_l), inv_hi = __double2hiint(inv_l);
    // Steps: per group its atoms, kAtoms at a time.  The loads of the next step
    // are in flight during a step; its buffers were last read before the
    // barrier that begins this one.
    load_radial(0, 0);
    load_phases(groups[0].first, min(kAtoms, groups[0].count), 0);
    int pb = 0;                           // buffer of the step's phases
    for (int kk = 0; kk < p.ngroups; ++kk) {
        const auto& kd = groups[kk];
        const int nlk = kd.lmax + 1, count = kd.count, rb = kk & 1;
        if ((kAdd && kk == 0) || kd.newdir) {
            // unit vectors [side][3][T] where the next group's radial factors will be
            double* s_n = (double*)(lds + (rb ^ 1) * 2 * planes * Ov::kPlane);
            __syncthreads();
            if (tid < 2 * T) {
                const int side = tid / T, c = tid - side * T;
                const int32_t* g = kSample ? kp->g : kp->gd;
                if (kSample && side) g = p.smp_g + 3 * (cj - J0 + min(J0 + c, min(ng, kSampleCols) - 1));
                else g += 3 * min((side ? J0 : I0) + c, ng - 1);
                double rot[9];
#pragma unroll
                for (int q = 0; q < 9; ++q) rot[q] = kd.rot[q];
                const DirAngles d = dir_angles(rot, kp->k[0] + g[0], kp->k[1] + g[1], kp->k[2] + g[2]);
                double* s = s_n + side * 3 * T + c;
                s[0] = d.sth * d.cph;
                s[T] = d.sth * d.sph;
                s[2 * T] = d.cth;
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int n = 0; n < MJ; ++n) {
                    const double* a = s_n + tx + 16 * m;
                    const double* b = s_n + 3 * T + ty + TY * n;
                    const double dot = __builtin_fma(a[2 * T], b[2 * T], __builtin_fma(a[T], b[T], a[0] * b[0]));
                    sg[m][n] = dot < 0.0 ? -1.0 : 1.0;
                    const double x = __builtin_fma(-sg[m][n], b[0], a[0]);
                    const double y = __builtin_fma(-sg[m][n], b[T], a[T]);
                    const double z = __builtin_fma(-sg[m][n], b[2 * T], a[2 * T]);
                    t[m][n] = 0.5 * __builtin_fma(z, z, __builtin_fma(y, y, x * x));
                }
        }
        for (int a0 = 0; a0 < count; a0 += kAtoms, pb ^= 1) {
            // this wave's loads of the step landed and its reads of the last
            // one are done; after the barrier every wave's
            __builtin_amdgcn_s_waitcnt(wait_vm(0, true));
            asm volatile("s_barrier" ::: "memory");
            if (a0 + kAtoms < count) {
                load_phases(kd.first + a0 + kAtoms, min(kAtoms, count - a0 - kAtoms), pb ^ 1);
            } else if (kk + 1 < p.ngroups) {
                load_radial(kk + 1, rb ^ 1);
                load_phases(groups[kk + 1].first, min(kAtoms, groups[kk + 1].count), pb ^ 1);
            }
            if (a0 == 0) {
                // sum over l, even and odd apart
                double P[M][MJ], d[M][MJ], od[M][MJ];
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int n = 0; n < MJ; ++n) {
                        P[m][n] = 1.0;
                        d[m][n] = 0.0;
                        rad[m][n] = 0.0;
                        od[m][n] = 0.0;
                        fr[m][n] = 0.0;
                        fi[m][n] = 0.0;
                    }
                const char* ri0 = lds + rb * 2 * planes * Ov::kPlane;
                struct Factors {
                    v2d ri[M], rj[MJ];
                };
                auto read = [&](int l, Factors& f) {
                    const char* base = ri0 + (l >> 4) * Ov::kPlane;
#pragma unroll
                    for (int m = 0; m < M; ++m)
                        f.ri[m] = *(const v2d*)&base[(tx + 16 * m) * 256 + ((l & 15) ^ tx) * 16];
#pragma unroll
                    for (int n = 0; n < MJ; ++n)
                        f.rj[n] = *(const v2d*)&base[planes * Ov::kPlane + (ty + TY * n) * 256 + ((l & 15) ^ (ty & 15)) * 16];
                };
                auto step = [&](int l, const Factors& f, double(&acc)[M][MJ]) {
                    const double cb = -(double)(2 * l + 1);
                    const double inv = __hiloint2double(__builtin_amdgcn_readlane(inv_hi, l), __builtin_amdgcn_readlane(inv_lo, l));
#pragma unroll
                    for (int m = 0; m < M; ++m)
#pragma unroll
                        for (int n = 0; n < MJ; ++n) {
                            const double w = __builtin_fma(f.ri[m].y, f.rj[n].y, f.ri[m].x * f.rj[n].x);
                            acc[m][n] = __builtin_fma(w, P[m][n], acc[m][n]);
                            d[m][n] = __builtin_fma(cb, t[m][n] * P[m][n], d[m][n]);
                            P[m][n] = __builtin_fma(d[m][n], inv, P[m][n]);
                        }
                };
                // kAhead: the factors of the next l are read ahead of a step
                Factors even, odd;
                if (kAhead) read(0, even);
                for (int l = 0; l < nlk; l += 2) {
                    if (kAhead) read(min(l + 1, nlk - 1), odd);
                    else read(l, even);
                    if (kAhead) __builtin_amdgcn_sched_barrier(0);
                    step(l, even, rad);
                    if (l + 1 >= nlk) break;
                    if (kAhead) read(min(l + 2, nlk - 1), even);
                    else read(l + 1, odd);
                    if (kAhead) __builtin_amdgcn_sched_barrier(0);
                    step(l + 1, odd, od);
                }
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int n = 0; n < MJ; ++n) rad[m][n] = __builtin_fma(sg[m][n], od[m][n], rad[m][n]);
            }
            // structure factor of the group's atoms
            const int na = min(kAtoms, count - a0);
            const char* pi0 = ph0 + pb * Ov::kPhases;
            auto read_phases = [&](int a, v2d* u, v2d* v) {
#pragma unroll
                for (int m = 0; m < M; ++m) u[m] = *(const v2d*)&pi0[(a * T + tx + 16 * m) * 16];
#pragma unroll
                for (int n = 0; n < MJ; ++n) v[n] = *(const v2d*)&pi0[((kAtoms + a) * T + ty + TY * n) * 16];
            };
            auto add_atom = [&](const v2d* u, const v2d* v) {
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int n = 0; n < MJ; ++n) {
                        fr[m][n] = __builtin_fma(u[m].y, v[n].y, __builtin_fma(u[m].x, v[n].x, fr[m][n]));
                        fi[m][n] = __builtin_fma(-u[m].y, v[n].x, __builtin_fma(u[m].x, v[n].y, fi[m][n]));
                    }
            };
            v2d u0[M], v0[MJ], u1[M], v1[MJ];
            if (kAhead) read_phases(0, u0, v0);
            for (int a = 0; a < na; a += 2) {
                if (kAhead) read_phases(min(a + 1, na - 1), u1, v1);
                else read_phases(a, u0, v0);
                if (kAhead) __builtin_amdgcn_sched_barrier(0);
                add_atom(u0, v0);
                if (a + 1 >= na) break;
                if (kAhead) read_phases(min(a + 2, na - 1), u0, v0);
                else read_phases(a + 1, u1, v1);
                if (kAhead) __builtin_amdgcn_sched_barrier(0);
                add_atom(u1, v1);
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int n = 0; n < MJ; ++n) {
                sr[m][n] = __builtin_fma(fr[m][n], rad[m][n], sr[m][n]);
                si[m][n] = __builtin_fma(fi[m][n], rad[m][n], si[m][n]);
            }
    }
#pragma unroll
    for (int n = 0; n < MJ; ++n)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int i = I0 + tx + 16 * m, j = J0 + ty + TY * n;
            if constexpr (kSample) {
                if (i < ng && j < min(ng, kSampleCols)) kp->S[(int64_t)j * kp->ldS + i] = make_double2(sr[m][n], si[m][n]);
            } else {
                if (i < ng && i >= j) kp->S[(int64_t)j * kp->ldS + i] = make_double2(sr[m][n], i == j ? 0.0 : si[m][n]);
            }
        }
}

template <int M, int MJ>
__global__ __launch_bounds__(256 * M / MJ) void k_overlap(SphereArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    stamp(p, 3);
    overlap_tile<M, MJ, true, false>(p, (int)blockIdx.x, lds);
}

__global__ __launch_bounds__(256) void k_overlap_sample(SphereArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    overlap_tile<2, 2, true, true>(p, (int)blockIdx.x, lds);
}

__global__ __launch_bounds__(256) void k_overlap_part(SphereArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    stamp(p, 3);
    overlap_tile<2, 2, true, false, true>(p, (int)blockIdx.x, lds);
}

int overlap_tile_size(int64_t tiles64, int n_cu)
{
    // 64 x 64 tiles, one workgroup per CU, once every CU has eight; 32 x 32 once
    // those give two, else 16 x 16: a smaller tile reads its columns more often but
    // spreads a small triangle over more CUs.  H and S at N_G 3001 with S in tiles
    // of 64 and 32: 1846, 1824 us; 6002: 9126, 9110; 12007: 190.4, 191.2 ms; a batch
    // of 12 of 1900 plane waves 16.38, 16.39 ms.
    if (tiles64 >= 8 * (int64_t)n_cu) return 64;
    return 4 * tiles64 >= 2 * (int64_t)n_cu ? 32 : 16;
}

template <int M, int MJ>
static hipError_t launch_overlap_tile(const SphereArgs& p, int64_t ntiles, hipEvent_t stop, hipStream_t st)
{
    using Ov = OverlapTile<M, MJ>;
    const size_t lds = Ov::lds((p.nl + 15) / 16);
    return launch(k_overlap<M, MJ>, dim3((unsigned)ntiles), Ov::NT, lds, stop, st, p);
}

hipError_t launch_overlap(const SphereArgs& p, int tile, int64_t ntiles, hipEvent_t stop, hipStream_t st)
{
    if (ntiles <= 0) return hipSuccess;
    if (tile == 64) return launch_overlap_tile<4, 2>(p, ntiles, stop, st);
    if (tile == 32) return launch_overlap_tile<2, 2>(p, ntiles, stop, st);
    return launch_overlap_tile<1, 1>(p, ntiles, stop, st);
}

hipError_t launch_overlap_part(const SphereArgs& p, hipEvent_t stop, hipStream_t st)
{
    const int64_t n = (p.one.ng + 31) / 32;
    return launch(k_overlap_part, dim3((unsigned)(n * (n + 1) / 2)), 256, (size_t)OverlapTile<2, 2>::lds((p.nl + 15) / 16),
                  stop, st, p);
}

// ---------------------------------------------------------------------------
// T in real harmonics: Mt = D^H M D of one atom's M = [[T_aa, T_ab],
// [T_ab^H, T_bb]] (T_aa, T_bb from their lower triangles), rows contiguous:
// Mt[r * ldm + k] = (D^H M D)_rk, zero for r or k past 2 nlm.  D maps real to
// complex harmonics with entries 1 and +-i, so an element is a sum of at most
// four elements of M.
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ double2 t_elem(const double2* taa, const double2* tab, const double2* tbb, int n, int r,
                                          int c)
{
    const bool rb = r >= n, cb = c >= n;
    const int i = rb ? r - n : r, j = cb ? c - n : c;
    double2 v;
    if (rb == cb) {
        const double2* t = rb ? tbb : taa;
        if (i >= j) {
            v = t[i + (int64_t)n * j];
        } else {
            v = t[j + (int64_t)n * i];
            v.y = -v.y;
        }
        if (i == j) v.y = 0.0;
    } else if (cb) {
        v = tab[i + (int64_t)n * j];
    } else {
        v = tab[j + (int64_t)n * i];
        v.y = -v.y;
    }
    return v;
}

}  // namespace

// Bound by latency: 7 MB of M for 16 atoms of lmax 8 take 12 us, where a loop on
// the host with the copy of its result took 1.9 ms.
__global__ __launch_bounds__(256) void k_build_m(const MJob* __restrict__ jobs, double2* __restrict__ m)
{
#pragma clang fp contract(off)
    const MJob jb = jobs[blockIdx.y];
    const int n = jb.nlm;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c = (int)(e / jb.ld), r = (int)(e - (int64_t)c * jb.ld);
    if (c >= jb.cols) return;
    double2 v = make_double2(0.0, 0.0);
    if (r < 2 * n && c < 2 * n) {
        v = t_elem(jb.taa, jb.tab, jb.tbb, n, r, c);
        if (jb.rsc && (r >= n || c >= n)) {
            const double d = (r >= n ? jb.rsc[l_of_lm(r - n)] : 1.0) * (c >= n ? jb.rsc[l_of_lm(c - n)] : 1.0);
            v.x /= d;
            v.y /= d;
        }
    }
    m[jb.off + e] = v;
}

hipError_t launch_build_m(const MJob* jobs, int njobs, int64_t max_elems, double2* m, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_build_m, dim3((unsigned)((max_elems + 255) / 256), njobs), dim3(256), 0, st, jobs, m);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_build_mt(const MtJob* __restrict__ jobs, double2* __restrict__ mt)
{
#pragma clang fp contract(off)
    const MtJob jb = jobs[blockIdx.y];
    const int n = jb.nlm, n2 = 2 * n;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int r = (int)(e / jb.ldm), k = (int)(e - (int64_t)r * jb.ldm);
    if (r >= jb.rows) return;
    double2 out = make_double2(0.0, 0.0);
    if (r < n2 && k < n2) {
        // D column of x = (l, +-m): entries at (l, m) and (l, -m)
        auto terms = [&](int x, int idx[2], double2 co[2]) {
            const int blk = x >= n ? n : 0;
            const int lm = x - blk;
            const int l = l_of_lm(lm);
            const int m = lm - l * (l + 1);
            if (m == 0) {
                idx[0] = x;
                co[0] = make_double2(1.0, 0.0);
                return 1;
            }
            const int am = m > 0 ? m : -m;
            const double s = (am & 1) ? -1.0 : 1.0;
            idx[0] = blk + l * (l + 1) + am;
            idx[1] = blk + l * (l + 1) - am;
            // cos: (1, s); sin: (-i, s i)
            co[0] = m > 0 ? make_double2(1.0, 0.0) : make_double2(0.0, -1.0);
            co[1] = m > 0 ? make_double2(s, 0.0) : make_double2(0.0, s);
            return 2;
        };
        int ir[2], ik[2];
        double2 cr[2], ck[2];
        const int nr = terms(r, ir, cr), nk = terms(k, ik, ck);
        for (int a = 0; a < nr; ++a)
            for (int b = 0; b < nk; ++b) {
                const double2 v = t_elem(jb.taa, jb.tab, jb.tbb, n, ir[a], ik[b]);
                // conj(cr) ck is a power of i
                const double fr = cr[a].x * ck[b].x + cr[a].y * ck[b].y;
                const double fi = cr[a].x * ck[b].y - cr[a].y * ck[b].x;
                if (fr != 0.0) {
                    out.x += fr * v.x;
                    out.y += fr * v.y;
                } else {
                    out.x -= fi * v.y;
                    out.y += fi * v.x;
                }
            }
    }
    mt[jb.off + e] = out;
}

hipError_t launch_build_mt(const MtJob* jobs, int njobs, int64_t max_elems, double2* mt, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_build_mt, dim3((unsigned)((max_elems + 255) / 256), njobs), dim3(256), 0, st, jobs, mt);
    return hipGetLastError();
}

// Split precision's W has complex rows: E M D = E D diag(1, 1/2) Mt, where
// D^H D = diag(1 for m = 0, else 2) and E divides the B rows by sq (sqrt(N_l)
// of folded operands, or 1).
__global__ __launch_bounds__(256) void k_split_mt(const SplitMtJob* __restrict__ jobs, const double* __restrict__ sq,
                                                  const double2* __restrict__ mt, double2* __restrict__ out)
{
#pragma clang fp contract(off)
    const SplitMtJob jb = jobs[blockIdx.y];
    const int n = jb.nlm;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int r = (int)(e / jb.ldm), k = (int)(e - (int64_t)r * jb.ldm);
    if (r >= jb.rows) return;
    double2 v = make_double2(0.0, 0.0);
    if (r < 2 * n) {
        const int blk = r >= n ? n : 0;
        const int l = l_of_lm(r - blk);
        const int m = r - blk - l * (l + 1);
        const int am = m < 0 ? -m : m;
        const double2* src = mt + jb.src + (int64_t)(blk + l * (l + 1)) * jb.ldm + k;
        const double2 c = src[(int64_t)am * jb.ldm];
        v = c;
        if (m != 0) {
            const double2 s = src[-(int64_t)am * jb.ldm];
            // (l, m): (c - i s) / 2; (l, -m): (-1)^m (c + i s) / 2
            v = m > 0 ? make_double2(0.5 * (c.x + s.y), 0.5 * (c.y - s.x))
                      : make_double2(0.5 * (c.x - s.y), 0.5 * (c.y + s.x));
            if (m < 0 && (am & 1)) v = make_double2(-v.x, -v.y);
        }
        if (blk) {
            const double d = sq[jb.sq + l];
            v.x /= d;
            v.y /= d;
        }
    }
    out[jb.dst + e] = v;
}

hipError_t launch_split_mt(const SplitMtJob* jobs, int njobs, int64_t max_elems, const double* sq, const double2* mt,
                           double2* out, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_split_mt, dim3((unsigned)((max_elems + 255) / 256), njobs), dim3(256), 0, st, jobs, sq, mt, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Complex-by-real products on v_mfma_f64_16x16x4.
//
// One tile is BR x BC: rows are columns of a complex operand X, columns are
// columns of a real operand y, both contiguous along the depth:
//   T[r][c] = sum_k X[k, r] y[k, c]       two real MFMAs per 16 x 16 x 4.
// kH: X = W of the tile's H columns j, y of the tile's H rows i.  The depth
//   runs over all atoms; where an atom ends (a k-step of 4, marked in the
//   k-step table) T is multiplied by conj(ph_a(i)) into the result C and
//   cleared: 4 fused operations per element and atom on the vector pipe next
//   to 4 (2 L_a) on the matrix pipe.  The table also gives the row of y of
//   each k-step, so atoms of one kind read the same y.
// !kH (T application): X = rows of Mt of one kind's atoms side by side, y of
//   the kind; W = ph_a(g) T is stored.
//
// Bound by FP64 MFMA.  Waves own 16 x 32 of the tile (16 x 16 of the 32 x 32
// tile): T and C take 64 VGPRs, so four waves per SIMD fit (two workgroups of
// 64 x 64 per CU, whose barriers do not wait for each other).  The operands go
// from global memory straight into a two-stage LDS ring (16 rows per stage);
// X's columns are 16 chunks of 16 bytes, chunk q stored at q ^ (column % 16),
// y's 8 chunks, chunk q at q ^ (column / 2 % 8): 16 lanes that read one row
// hit distinct banks.  The fragments of the next k-step are read before the
// MFMAs of the current one, across the stage barrier too; a stage also brings
// the phases of an atom that ends in it, so that no flush waits for memory;
// LDS addresses are constants per lane and load bases scalar, which leaves the
// vector pipe to the MFMAs.  Rings of 3 and 4 stages, 64 x 128 tiles and waves
// of 32 x 32 measured no faster for these tiles at any size from 235 to 25000
// plane waves.
// The 32 x 32 tiles of H serve triangles that leave CUs idle, with two to four
// waves per SIMD: there the latency of a stage counts.  A deeper ring, the
// fragments of a whole stage read while the one before is multiplied, table
// entries two barriers ahead: H and S together 20.8 us (two stages without:
// 26.9) at N_G 600, 12.5 (13.7) at 235, 1075 (1121) at 2003; four stages and
// three workgroups per CU 21.3, 12.7 and 1112.  The T application, with depths of
// 10 to 20 stages, loses with a third stage what it loses in workgroups.
// Rate of the H tiles: 0.86 of the FP64 peak at N_G 12009, 16000 and 24995 (0.84
// on the slowest board), 0.85 at 10025, 0.82 at 6002 (32 atoms, lmax 10).
// Measured (whole call, complex-by-complex contraction of S and H before, now):
// 714 -> 202 ms at N_G 12007 (128 atoms, lmax 12), 33.5 -> 10.0 ms at 6002 and
// 5.41 -> 1.37 ms at 2003 (32 atoms, lmax 10), with S and all else since.
// ---------------------------------------------------------------------------
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef int i8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(4))) const i8* ctab;

// Columns of a group in the T application's order: an XCD's eighth of a
// group's y (340 rows at lmax 12) is 1.4 MB of its 4 MB L2.  T application in
// one group, in groups of 8192, 4096, 2048: 13.2, 12.7, 12.4, 12.4 ms at N_G 12007;
// a batch of 22800 columns (whole) 17.00, 16.87, 16.75, 16.83 ms; nothing
// changes up to 4096 columns.  An eighth of the tiles of contiguous columns per
// XCD instead: 351 -> 370 us at N_G 3001.
constexpr int kSphereColumns = 4096;

// Stages in LDS of the 32 x 32 tiles of H: three of 13 KB let four workgroups
// share a CU, as 128 VGPRs do.
constexpr int kSphereSmall = 3;

// Atoms that end in a stage before its k-step ks.
__device__ __forceinline__ int ends_before(i8 e, int ks)
{
    return (ks > 0 ? e[0] & 1 : 0) + (ks > 1 ? e[1] & 1 : 0) + (ks > 2 ? e[2] & 1 : 0);
}

}  // namespace

// BR x BC tile (rows: X columns, columns: y columns), waves of 16 RB x 16 CB,
// NS stages in LDS.  PARTS 2: one wave the real, one the imaginary part.
template <int BR, int BC, int RB, int CB, int NS, int PARTS = 1>
struct SphereTile {
    static constexpr int kWR = BR / (16 * RB);    // waves along the rows
    static constexpr int kWC = BC / (16 * CB);
    static constexpr int kWaves = kWR * kWC * PARTS;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kXBytes = BR * 256;      // one stage of X, of y
    static constexpr int kYBytes = BC * 128;
    static constexpr int kPhBytes = 256 * CB;     // a wave's phases of an atom that ends in a stage
    static constexpr int kStage = kXBytes + kYBytes + kWaves * kPhBytes;
    static constexpr int kSwap = PARTS == 2 ? 2 * kWaves * RB * CB * 2048 : 0;   // T that the parts exchange
    static constexpr int kLds = NS * kStage + kSwap;
    static constexpr int kXLoads = kXBytes / 1024 / kWaves;   // 1 KiB wave loads per wave and stage
    static constexpr int kYLoads = kYBytes / 1024 / kWaves;
    static_assert(kXLoads * kWaves * 1024 == kXBytes && kYLoads * kWaves * 1024 == kYBytes,
                  "a stage splits evenly over the waves");
    static_assert(BC % BR == 0, "patches are square in plane waves");
};

template <class F, int... I>
__device__ __forceinline__ void stages(const F& f, int s, std::integer_sequence<int, I...>)
{
    f(s, std::integral_constant<int, I>{}...);
}

__device__ __forceinline__ int64_t uni(int64_t v)
{
    return (int64_t)(((uint64_t)(uint32_t)uni((int)(v >> 32)) << 32) | (uint32_t)uni((int)v));
}

// What a product computes: W (T application), the lower triangle of H, the
// sampled columns of H, or the triangle's columns hcol0 .. hcol1 - 1.
enum SphereMode { kTApp, kLowerH, kSampleH, kPartH };

template <int BR, int BC, int RB, int CB, int NS, int kMode, int PARTS = 1>
__device__ __forceinline__ void sphere_gemm_tile(const SphereArgs& p, int blk, char* lds)
{
#pragma clang fp contract(off)
    constexpr bool kH = kMode != kTApp;
    using Tl = SphereTile<BR, BC, RB, CB, NS, PARTS>;
    constexpr int NX = Tl::kXLoads, NY = Tl::kYLoads;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % Tl::kWR, wc = wave / Tl::kWR % Tl::kWC;
    const int part = PARTS == 2 ? wave / (Tl::kWR * Tl::kWC) : 0;

    // ---- the tile ----
    const SphereK* kp = &p.one;
    const KindDev* kd = nullptr;
    int R0, C0;             // first row (X column), first column (y column) of the tile
    int nsteps;             // k-steps of 4
    int i0 = 0, xcol = 0;   // samples: H row of the tile's first y column, first of the k-point's X columns
    if constexpr (kMode == kSampleH) {
        // tiles of the chunk's columns in turn, per tile the sampled ones
        constexpr int kRow = kSampleCols / BR;
        const int tc = blk / kRow;
        C0 = uni(tc * BC);
        R0 = uni((blk - tc * kRow) * BR);
        const int c = (int)p.cbase + C0;
        const int ki = p.nk > 1 ? find_last(p.nk, c, [&](int i) { return (int)p.many[i].col0; }) : 0;
        if (p.nk > 1) kp = p.many + ki;
        i0 = uni(c - (int)kp->col0);
        xcol = uni(ki * kSampleCols);
        if (i0 >= kp->ng || R0 >= min(kp->ng, kSampleCols)) return;
        nsteps = p.nksteps;
    } else if constexpr (kH) {
        // Workgroups go to the 8 XCDs in turn.  The lower squares of BC of all
        // k-points, in patches of P x P squares, are cut into 8 equal
        // parts, one per XCD: the tiles in flight on one L2 share their
        // panels, and every XCD has the same work.
        constexpr int kRat = BC / BR;
        constexpr int P = kSpherePatch;
        const int n = p.nsquares * kRat;
        const int x = blk % 8, at = blk / 8;
        const int t0 = (int)((int64_t)n * x / 8), t1 = (int)((int64_t)n * (x + 1) / 8);
        if (at >= t1 - t0) return;
        const int sq = (t0 + at) / kRat;
        if (p.nk > 1) kp = p.many + find_last(p.nk, sq, [&](int i) { return p.many[i].hsquare0; });
        const int t = sq - kp->hsquare0;
        const int nt = (kp->ng + BC - 1) / BC;
        const int pi = tri_row(t) / P;                        // patch row
        int u = t - (int)((int64_t)(pi * P) * (pi * P + 1) / 2);
        const int h = min(P, nt - pi * P);                    // its rows
        int bi, bj;
        if (u < pi * P * h) {
            const int pj = u / (P * h);
            u -= pj * P * h;
            bi = u % h;
            bj = pj * P + u / h;
        } else {
            u -= pi * P * h;
            bi = tri_row(u);
            bj = pi * P + u - bi * (bi + 1) / 2;
        }
        C0 = uni((pi * P + bi) * BC);
        R0 = uni(bj * BC + (t0 + at) % kRat * BR);
        if (R0 >= kp->ng) return;
        if (kMode == kPartH && (R0 < p.hcol0 || R0 >= p.hcol1)) return;
        nsteps = p.nksteps;
    } else {
        // Columns in groups of P tiles; per group the tiles of rows of all
        // kinds in turn, per row tile the group's columns, which go to the XCDs
        // in turn: what an XCD reads of the group's y stays in its L2 while the
        // rows pass.
        constexpr int P = kSphereColumns / BC;
        const int ntc = p.tcols / BC;
        const int cg = (int)(blk / ((int64_t)P * p.rtiles));
        const int u = (int)(blk - (int64_t)cg * P * p.rtiles);
        const int h = min(P, ntc - cg * P);                   // the group's columns
        const int tr = u / h;
        const int kk = find_last(p.nkinds, tr, [&](int i) { return p.kinds[i].rt32; });
        kd = p.kinds + kk;
        R0 = uni((tr - kd->rt32) * BR);
        C0 = uni((cg * P + u - tr * h) * BC);
        nsteps = uni(kd->r4 / 4);
    }
    const int64_t col0 = kMode == kLowerH || kMode == kPartH ? uni(kp->col0) : 0;
    const double2* const X = kMode == kSampleH ? p.smp_W + (int64_t)xcol * p.smp_ldw : p.W + col0 * p.ldw;
    const int64_t ldx = kMode == kSampleH ? p.smp_ldw : p.ldw;
    const int nst = uni((nsteps + 3) / 4);

    // ---- loads ----
    // A wave load of X fills 4 columns of 16 chunks, one of y 8 columns of 8.
    // Bases are wave-uniform, lanes add 32-bit offsets; only Mt, whose rows
    // change blocks between atoms, takes a pointer per lane.
    const char* xbase[NX];
    uint32_t xoff[NX];
    const char* xptr[NX];
#pragma unroll
    for (int r = 0; r < NX; ++r) {
        const int c0 = (wave * NX + r) * 4;
        const int c = c0 + (lane >> 4);
        const int q = (lane & 15) ^ (c & 15);
        if constexpr (kH) {
            xbase[r] = (const char*)(X + (R0 + c0) * ldx);
            xoff[r] = (uint32_t)(((int64_t)(lane >> 4) * ldx + q) * 16);
        } else {
            // row R0 + c of the kind's stacked Mt; past its last row the last one again
            const int row = min(R0 + c, kd->count * kd->r4 - 1);
            const int a = row / kd->r4;
            xptr[r] = (const char*)(p.mt + p.mtoff[kd->first + a] + (int64_t)(row - a * kd->r4) * kd->ldm + q);
        }
    }
    const char* ybase[NY];
    uint32_t yoff[NY];
    int sel[NY];            // the lane's k-step within a stage
#pragma unroll
    for (int r = 0; r < NY; ++r) {
        const int c0 = (wave * NY + r) * 8;
        const int c = c0 + (lane >> 3);
        const int q = (lane & 7) ^ ((c >> 1) & 7);
        ybase[r] = (const char*)(p.y + (col0 + C0 + c0) * p.ldy);
        yoff[r] = (uint32_t)(((int64_t)(lane >> 3) * p.ldy + 2 * (q & 1)) * 8);
        if constexpr (!kH) yoff[r] += (uint32_t)(kd->yoff + 4 * (q >> 1)) * 8;
        sel[r] = q >> 1;
    }
    // constant address space: the table's entries come by scalar loads
    const ctab tab = (ctab)(const void*)p.stages;
    // stage s (for T: nothing)
    auto entry = [&](int s) -> i8 {
        if constexpr (kH) return tab[uni(s)];
        else return i8{0, 0, 0, 0, -1, 0, 0, 0};
    };
    typedef __attribute__((address_space(1))) const char gchar;
    typedef __attribute__((address_space(3))) char lchar;
    lchar* lbase = (lchar*)lds;
    // one stage: the phases of the first atom that ends in it, X, y (the wait
    // for a stage counts the X and y loads of the stages after it)
    auto issue = [&](int s, int buf, i8 e) {
        if constexpr (kH) {
            if (e[4] >= 0 && lane < 16 * CB) {
                gchar* g = (gchar*)(p.ph + (int64_t)e[4] * p.gtot + (col0 + C0 + wc * 16 * CB)) + lane * 16;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                                 (__attribute__((address_space(3))) void*)(lbase + buf * Tl::kStage +
                                                                                           Tl::kXBytes + Tl::kYBytes +
                                                                                           wave * Tl::kPhBytes),
                                                 16, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < NX; ++r) {
            gchar* g;
            if constexpr (kH) g = (gchar*)(xbase[r] + (int64_t)uni(s) * 256) + xoff[r];
            else g = (gchar*)(xptr[r] + (int64_t)s * 256);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                             (__attribute__((address_space(3))) void*)(lbase + buf * Tl::kStage +
                                                                                       (wave * NX + r) * 1024),
                                             16, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < NY; ++r) {
            gchar* g;
            if constexpr (kH) {
                const int lo = sel[r] & 1 ? e[1] : e[0], hi = sel[r] & 1 ? e[3] : e[2];
                const uint32_t row = (uint32_t)(sel[r] & 2 ? hi : lo) & ~3u;
                g = (gchar*)ybase[r] + (yoff[r] + row * 8);
            } else {
                g = (gchar*)(ybase[r] + (int64_t)s * 128) + yoff[r];
            }
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                             (__attribute__((address_space(3))) void*)(lbase + buf * Tl::kStage +
                                                                                       Tl::kXBytes +
                                                                                       (wave * NY + r) * 1024),
                                             16, 0, 0);
        }
    };

    d4 tr_[RB][CB], ti_[RB][CB];
    d4 cr[RB][CB], ci[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            tr_[i][j] = ti_[i][j] = d4{0.0, 0.0, 0.0, 0.0};
            if constexpr (kH) cr[i][j] = ci[i][j] = d4{0.0, 0.0, 0.0, 0.0};
        }

    // LDS offsets of the lane's fragments per k-step; further blocks of 16
    // and the second stage are constant distances away
    const int r0 = wr * 16 * RB + (lane & 15), c0 = wc * 16 * CB + (lane & 15);
    const int q0 = lane >> 4;
    int xat[4], yat[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        xat[ks] = r0 * 256 + 16 * ((q0 + 4 * ks) ^ (r0 & 15));
        yat[ks] = Tl::kXBytes + c0 * 128 + 16 * (((q0 >> 1) + 2 * ks) ^ ((c0 >> 1) & 7)) + 8 * (q0 & 1);
    }
    auto read_frags = [&](int buf, int ks, v2d* x, double* y) {
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            if constexpr (PARTS == 2) x[i].x = *(const double*)&lds[xat[ks] + 8 * part + (buf * Tl::kStage + i * 4096)];
            else x[i] = *(const v2d*)&lds[xat[ks] + (buf * Tl::kStage + i * 4096)];
        }
#pragma unroll
        for (int j = 0; j < CB; ++j) y[j] = *(const double*)&lds[yat[ks] + (buf * Tl::kStage + j * 2048)];
    };
    const int phat = Tl::kXBytes + Tl::kYBytes + wave * Tl::kPhBytes + (lane & 15) * 16;
    // Phases at this lane's H rows: of the first atom that ends in a stage,
    // from the stage; of further ones (atoms of few rows) from memory.
    auto stage_phases = [&](int buf, v2d* ph) {
#pragma unroll
        for (int j = 0; j < CB; ++j)
            ph[j] = *(const v2d*)&lds[phat + (buf * Tl::kStage + j * 256)];
    };
    auto far_phases = [&](int atom, v2d* ph) {
#pragma unroll
        for (int j = 0; j < CB; ++j) ph[j] = *(const v2d*)&p.ph[(int64_t)atom * p.gtot + (col0 + C0 + c0 + 16 * j)];
    };
    // C += conj(phase) T, T = 0
    int swap = 0;
    auto flush = [&](const v2d* ph) {
        if constexpr (PARTS == 2) {
            // the other part of T by way of LDS; two buffers, so that one barrier
            // per flush does
            char* mine = lds + NS * Tl::kStage + (swap * Tl::kWaves + wave) * (RB * CB * 2048) + lane * 16;
            const int other = part ? wave - Tl::kWR * Tl::kWC : wave + Tl::kWR * Tl::kWC;
            const char* its = lds + NS * Tl::kStage + (swap * Tl::kWaves + other) * (RB * CB * 2048) + lane * 16;
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    *(v2d*)&mine[(i * CB + j) * 2048] = v2d{tr_[i][j][0], tr_[i][j][1]};
                    *(v2d*)&mine[(i * CB + j) * 2048 + 1024] = v2d{tr_[i][j][2], tr_[i][j][3]};
                }
            __builtin_amdgcn_s_waitcnt(wait_vm(63, true));
            asm volatile("s_barrier" ::: "memory");
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const v2d o = *(const v2d*)&its[(i * CB + j) * 2048 + h * 1024];
#pragma unroll
                        for (int q = 2 * h; q < 2 * h + 2; ++q) {
                            // part 0: a mine, b the other; part 1 the other way round
                            const double m = tr_[i][j][q], v = h == 0 ? (q == 0 ? o.x : o.y) : (q == 2 ? o.x : o.y);
                            cr[i][j][q] = __builtin_fma(part ? -ph[j].y : ph[j].y, v, __builtin_fma(ph[j].x, m, cr[i][j][q]));
                            tr_[i][j][q] = 0.0;
                        }
                    }
            swap ^= 1;
            return;
        }
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double a = tr_[i][j][q], b = ti_[i][j][q];
                    cr[i][j][q] = __builtin_fma(ph[j].y, b, __builtin_fma(ph[j].x, a, cr[i][j][q]));
                    ci[i][j][q] = __builtin_fma(-ph[j].y, a, __builtin_fma(ph[j].x, b, ci[i][j][q]));
                    tr_[i][j][q] = 0.0;
                    ti_[i][j][q] = 0.0;
                }
    };

    // ---- main loop ----
    // (at the end the last stage is loaded again: in bounds, unused)
    const int last = nst - 1;
    // one k-step: T += X y; rows past the depth (in the last stage) are not
    // multiplied
    auto mfmas = [&](int s, int ks, const v2d* x, const double* y) {
        if (kH || 4 * s + ks < nsteps) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j)
                    tr_[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i].x, y[j], tr_[i][j], 0, 0, 0);
            if constexpr (PARTS == 1) {
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int j = 0; j < CB; ++j)
                        ti_[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i].y, y[j], ti_[i][j], 0, 0, 0);
            }
        }
    };
    i8 en[NS];              // stage s's entries in en[s % NS]
#pragma unroll
    for (int i = 0; i < NS; ++i) en[i] = entry(min(i, last));
#pragma unroll
    for (int i = 0; i + 1 < NS; ++i) issue(min(i, last), i, en[i]);
    __builtin_amdgcn_s_waitcnt(wait_vm((NS - 2) * (NX + NY), false));
    asm volatile("s_barrier" ::: "memory");
    issue(min(NS - 1, last), NS - 1, en[NS - 1]);
    if constexpr (NS > 2) {
        // Few waves per SIMD: the fragments (and phases) of a whole stage are
        // read while the one before is multiplied, three stages of loads in
        // flight behind it.
        v2d fx[2][4][RB];
        double fy[2][4][CB];
        v2d fp[2][CB];
        auto read_stage = [&](int buf, int set) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) read_frags(buf, ks, fx[set][ks], fy[set][ks]);
            if constexpr (kH) stage_phases(buf, fp[set]);
        };
        read_stage(0, 0);
        i8 next = entry(min(NS, last));     // the entry of the stage issued next
        auto stage = [&](auto at, int s) {
            constexpr int buf = decltype(at)::value % NS, set = decltype(at)::value & 1;
            const i8 e = en[buf];
            __builtin_amdgcn_s_waitcnt(wait_vm(63, true));
            if (s < last) {
                // this wave's loads of stage s+1 landed and its reads of stage
                // s are done; after the barrier that holds for every wave, and
                // stage s+NS may overwrite stage s
                __builtin_amdgcn_s_waitcnt(wait_vm((NS - 2) * (NX + NY), false));
                asm volatile("s_barrier" ::: "memory");
                issue(min(s + NS, last), buf, next);
                en[buf] = next;
                next = entry(min(s + NS + 1, last));
                read_stage((buf + 1) % NS, set ^ 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                mfmas(s, ks, fx[set][ks], fy[set][ks]);
                if constexpr (kH) {
                    if (e[ks] & 1) {
                        v2d ph[CB];
                        if (e[ks] & 2) {
                            far_phases(e[4] + ends_before(e, ks), ph);
                        } else {
#pragma unroll
                            for (int j = 0; j < CB; ++j) ph[j] = fp[set][j];
                        }
                        flush(ph);
                    }
                }
            }
        };
        constexpr int U = NS % 2 ? 2 * NS : NS;     // buffers and register sets in step
        auto round = [&](int s, auto... i) { (((int)i + s < nst ? stage(i, s + (int)i) : (void)0), ...); };
        for (int s = 0; s < nst; s += U) stages(round, s, std::make_integer_sequence<int, U>{});
    } else {
        v2d fx[RB];
        double fy[CB];
        read_frags(0, 0, fx, fy);
        // stage s from LDS buffer `buf`
        auto stage = [&](auto bufc, int s) {
            constexpr int buf = decltype(bufc)::value;
            const i8 e = en[buf];
            const i8 e2 = entry(min(s + 2, last));
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                v2d x[RB];
                double y[CB];
#pragma unroll
                for (int i = 0; i < RB; ++i) x[i] = fx[i];
#pragma unroll
                for (int j = 0; j < CB; ++j) y[j] = fy[j];
                v2d ph[CB];
                if (ks < 3) {
                    read_frags(buf, ks + 1, fx, fy);
                } else if (s < last) {
                    // an atom that ends with the stage still needs its phases
                    if (kH && (e[3] & 3) == 1) stage_phases(buf, ph);
                    // as above, with two stages
                    __builtin_amdgcn_s_waitcnt(wait_vm(0, true));
                    asm volatile("s_barrier" ::: "memory");
                    issue(min(s + 2, last), buf, e2);
                    read_frags(buf ^ 1, 0, fx, fy);
                }
                // reads ahead of the MFMAs, as written
                __builtin_amdgcn_sched_barrier(0);
                mfmas(s, ks, x, y);
                if constexpr (kH) {
                    if (e[ks] & 1) {
                        if (e[ks] & 2) far_phases(e[4] + ends_before(e, ks), ph);
                        else if (ks < 3 || s == last) stage_phases(buf, ph);
                        flush(ph);
                    }
                }
            }
            en[buf] = e2;
        };
        int s = 0;
        for (; s < last; s += 2) {
            stage(std::integral_constant<int, 0>{}, s);
            stage(std::integral_constant<int, 1>{}, s + 1);
        }
        if (s < nst) stage(std::integral_constant<int, 0>{}, s);
    }
    __builtin_amdgcn_s_waitcnt(0);

    // ---- store: lane holds rows (lane >> 4) + 4 q of column lane & 15 ----
    if constexpr (kMode == kSampleH) {
        const int ng = kp->ng, nb = min(ng, kSampleCols);
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                const int gi = i0 + c0 + 16 * j;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int gj = R0 + wr * 16 * RB + i * 16 + q0 + 4 * q;
                    if (gi < ng && gj < nb) kp->H[(int64_t)gj * kp->ldH + gi] = make_double2(cr[i][j][q], ci[i][j][q]);
                }
            }
    } else if constexpr (kH) {
        const int ng = kp->ng;
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                const int gi = C0 + c0 + 16 * j;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int gj = R0 + wr * 16 * RB + i * 16 + q0 + 4 * q;
                    if (gi >= ng || gi < gj) continue;
                    double2* h = kp->H + (int64_t)gj * kp->ldH + gi;
                    if constexpr (PARTS == 2) *((double*)h + part) = part && gi == gj ? 0.0 : cr[i][j][q];
                    else *h = make_double2(cr[i][j][q], gi == gj ? 0.0 : ci[i][j][q]);
                }
            }
    } else {
        const int nrow = kd->count * kd->r4;
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = R0 + wr * 16 * RB + i * 16 + q0 + 4 * q;
                int64_t dst = kd->woff + row;
                if (row < nrow && p.rowdst) dst = p.rowdst[dst];
                if (row < nrow && dst >= 0) {
                    const double2* phr = p.ph + (int64_t)(kd->first + row / kd->r4) * p.gtot;
#pragma unroll
                    for (int j = 0; j < CB; ++j) {
                        const int64_t col = C0 + c0 + 16 * j;
                        const double2 f = phr[col];
                        const double a = tr_[i][j][q], b = ti_[i][j][q];
                        p.W[col * p.ldw + dst] =
                            make_double2(__builtin_fma(f.x, a, -(f.y * b)), __builtin_fma(f.x, b, f.y * a));
                    }
                }
            }
    }
}

template <int BR, int BC, int RB, int CB, int NS, int kMode, int PARTS = 1>
__global__ __launch_bounds__((SphereTile<BR, BC, RB, CB, NS, PARTS>::kThreads), 4) void k_sphere_gemm(SphereArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    stamp(p, kMode == kTApp ? 1 : 2);
    sphere_gemm_tile<BR, BC, RB, CB, NS, kMode, PARTS>(p, (int)blockIdx.x, lds);
}

// H tiles of 32 x 32 and S tiles of 16 M x 16 M in one launch, for triangles
// whose H tiles leave CUs or the vector pipe idle: S costs no time of its own.
// PARTS 2: H tiles of 16 x 32.
template <int M, int PARTS>
__global__ __launch_bounds__(256, 4) void k_sphere_hs(SphereArgs p, int hblocks)
{
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    stamp(p, 2);
    if ((int)blockIdx.x < hblocks)
        sphere_gemm_tile<32 / PARTS, 32, 1, 1, kSphereSmall, kLowerH, PARTS>(p, (int)blockIdx.x, lds);
    else overlap_tile<M, M, false, false>(p, (int)blockIdx.x - hblocks, lds);
}

template <int BR, int BC, int RB, int CB, int NS, int kMode, int PARTS = 1>
static hipError_t launch_sphere_gemm(const SphereArgs& p, int64_t nblk, hipEvent_t stop, hipStream_t st)
{
    using Tl = SphereTile<BR, BC, RB, CB, NS, PARTS>;
    return launch(k_sphere_gemm<BR, BC, RB, CB, NS, kMode, PARTS>, dim3((unsigned)nblk), Tl::kThreads, Tl::kLds, stop, st, p);
}

// rtiles: row tiles of all kinds for the tile's rows (tile 64: 32 x 64)
hipError_t launch_sphere_tapp(const SphereArgs& p, int tile, int rtiles, hipEvent_t stop, hipStream_t st)
{
    SphereArgs q = p;
    q.rtiles = rtiles;
    const int64_t nblk = (int64_t)rtiles * (p.tcols / (tile == 32 ? 32 : 64));
    if (tile == 32) return launch_sphere_gemm<32, 32, 1, 1, 2, kTApp>(q, nblk, stop, st);
    return launch_sphere_gemm<32, 64, 1, 2, 2, kTApp>(q, nblk, stop, st);
}

static int64_t hblocks(const SphereArgs& p, int tile)
{
    return ((int64_t)p.nsquares * (tile == 48 || tile == 16 ? 2 : 1) + 7) / 8 * 8;
}

// tile: 64 (64 x 64), 48 (32 x 64), 32 (32 x 32) or 16 (16 x 32, by parts)
hipError_t launch_sphere_h(const SphereArgs& p, int tile, hipEvent_t stop, hipStream_t st)
{
    const int64_t n = hblocks(p, tile);
    if (tile == 16) return launch_sphere_gemm<16, 32, 1, 1, kSphereSmall, kLowerH, 2>(p, n, stop, st);
    if (tile == 32) return launch_sphere_gemm<32, 32, 1, 1, kSphereSmall, kLowerH>(p, n, stop, st);
    if (tile == 48) return launch_sphere_gemm<32, 64, 1, 2, 2, kLowerH>(p, n, stop, st);
    return launch_sphere_gemm<64, 64, 1, 2, 2, kLowerH>(p, n, stop, st);
}

// H of one k-point's columns hcol0 .. hcol1 - 1, multiples of 64
hipError_t launch_sphere_h_part(const SphereArgs& p, hipEvent_t stop, hipStream_t st)
{
    SphereArgs q = p;
    const int n = (p.one.ng + 31) / 32;
    q.nsquares = n * (n + 1) / 2;
    return launch_sphere_gemm<32, 32, 1, 1, kSphereSmall, kPartH>(q, (q.nsquares + 7) / 8 * 8, stop, st);
}

template <int M, int PARTS>
static hipError_t launch_hs(const SphereArgs& p, int64_t nstiles, hipEvent_t stop, hipStream_t st)
{
    const int64_t n = hblocks(p, 32 / PARTS);
    const size_t lds = std::max<size_t>(SphereTile<32 / PARTS, 32, 1, 1, kSphereSmall, PARTS>::kLds,
                                        OverlapTile<M, M>::lds((p.nl + 15) / 16));
    return launch(k_sphere_hs<M, PARTS>, dim3((unsigned)(n + nstiles)), 256, lds, stop, st, p, (int)n);
}

hipError_t launch_sphere_hs(const SphereArgs& p, int tile, int stile, int64_t nstiles, hipEvent_t stop, hipStream_t st)
{
    if (tile == 16) return launch_hs<1, 2>(p, nstiles, stop, st);
    return stile == 32 ? launch_hs<2, 1>(p, nstiles, stop, st) : launch_hs<1, 1>(p, nstiles, stop, st);
}

// G of the sampled columns: block ki, lane j.
__global__ __launch_bounds__(kSampleCols) void k_sample_g(SphereArgs p, const int32_t* __restrict__ cols, int32_t* __restrict__ out)
{
    const SphereK* kp = p.nk > 1 ? p.many + blockIdx.x : &p.one;
    const int at = blockIdx.x * kSampleCols + threadIdx.x;
    for (int q = 0; q < 3; ++q) out[3 * at + q] = kp->g[3 * cols[at] + q];
}

hipError_t launch_sample_g(const SphereArgs& p, const int32_t* cols, int32_t* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_sample_g, dim3(p.nk), dim3(kSampleCols), 0, st, p, cols, out);
    return hipGetLastError();
}

hipError_t launch_sample(const SphereArgs& p, bool do_h, bool do_s, hipStream_t st)
{
    hipError_t e = hipSuccess;
    if (do_h)
        e = launch_sphere_gemm<32, 32, 1, 1, kSphereSmall, kSampleH>(p, p.gtot / 32 * (kSampleCols / 32), nullptr, st);
    if (e == hipSuccess && do_s)
        e = launch(k_overlap_sample, dim3((unsigned)(p.gtot / 32 * (kSampleCols / 32))), 256,
                   (size_t)OverlapTile<2, 2>::lds((p.nl + 15) / 16), nullptr, st, p);
    return e;
}

}  // namespace hsgen
