// FP64 H and S from a system description: declarations of the kernels in
// sphere.hip and of the tables they share with the host.
//
// A matching coefficient of atom a at plane wave K factors into a phase and
// a real number: with real spherical harmonics y (cos / sin of m phi in place
// of e^{i m phi})
//   A_lm = ph_a(K) (D y_a(K))_lm, B_lm likewise,   ph_a = e^{i 2 pi K.tau_a},
// D the constant map from real to complex harmonics and y_a real, the same
// for all atoms of one "kind" (equal l cutoff, radius, radial data and
// rotation, bit for bit).  So
//   H_ij = sum_a conj(ph_a(i)) [ y_a(i)^T W_a(j) ],   W_a = ph_a (D^H M_a D) y_a
//   S_ij = sum_group F(i, j) sum_l (2l+1)/4pi (a_l a_l' + N_l b_l b_l') P_l(cos),
//          F(i, j) = sum_{a of the group} conj(ph_a(i)) ph_a(j)
// (the addition theorem): H takes one real-by-complex product per depth, half
// the operations of a complex one, and S next to none.
#pragma once

#include "hsgen_internal.h"

namespace hsgen {

// Column padding of the operand arrays, and the squares of H tiles along a
// patch that one XCD runs at a time (32 CUs, two 64 x 64 tiles each).
constexpr int kSphereCols = 64;
constexpr int kSpherePatch = 8;

// Atoms of one kind share the real vector y and the radial factors.
struct KindDev {
    int32_t lmax, nlm;
    int32_t r4;          // rows of y and of one W_a: 2 nlm rounded up to the MFMA depth of 4
    int32_t rep;         // first atom of the kind (system order): RadDev row
    int32_t yoff;        // first row of y
    int32_t rsoff;       // first row of its overlap group's radial factors, or -1 if another kind writes them
    int32_t woff;        // first row of W
    int32_t ldm;         // leading dimension of Mt: 2 nlm rounded up to the stage depth of 16
    int32_t rt32;        // T-application row tiles of 32 of the kinds before this one
    int32_t first, count;   // its atoms, in kind order
    double rmt;
    double rot[9];       // column-major R_atom * bmat
};

// Kinds that differ in their rotations only, all with the same cosines between
// plane waves (equal R^T R): one Legendre sum of S for all their atoms.
struct OverlapGroup {
    int32_t lmax;
    int32_t rep;         // an atom of it (system order): RadDev row
    int32_t rsoff;       // first row of the radial factors (a_l, b_l), then of the weighted ones
    int32_t first, count;   // its atoms, in kind order
    int32_t newdir;      // directions differ from the group before
    double rot[9];       // the rotation that stands for the cosines
};

// One k-point of a launch.
struct SphereK {
    double k[3];
    const int32_t* g;    // [ng][3], device or pinned host memory: read by the generator
    int32_t* gd;         // device copy of g that the generator makes, or g itself: read by S
    double2* H;
    double2* S;
    int64_t ldH, ldS;
    int64_t col0;        // first column in the operand arrays (a multiple of the tile side)
    int32_t ng;
    int32_t gcol0;       // plane waves of the k-points before this one
    int32_t stile0;      // S tiles before this one
    int32_t hsquare0;    // lower squares of H tiles before this one
};

// One T block to turn into real harmonics (device pointers).
struct MtJob {
    const double2* taa;
    const double2* tab;
    const double2* tbb;
    int64_t off;         // of its Mt (complex units)
    int32_t nlm, rows, ldm;
    int32_t pad;
};

// One M_a of the general T application: [T_aa T_ab; T_ab^H T_bb] with the B rows
// and columns divided by rsc (null: by 1), zero beyond 2 nlm.
struct MJob {
    const double2* taa;
    const double2* tab;
    const double2* tbb;
    const double* rsc;   // per l
    int64_t off;         // of its M (complex units)
    int32_t nlm, ld, cols;
    int32_t pad;
};

// One matrix of split precision's T application, from its Mt.
struct SplitMtJob {
    int64_t src, dst;    // offsets (complex units)
    int32_t nlm, rows, ldm;
    int32_t sq;          // first of the divisors of its B rows, per l
};

// One stage of 16 rows of H's depth, four k-steps of 4.
struct SphereStage {
    int32_t step[4];     // row of y of the k-step (a multiple of 4); bit 0: an atom ends with it; bit 1: and
                         // another one ended earlier in the stage
    int32_t atom;        // first atom (kind order) that ends in the stage, or -1
    int32_t pad[3];
};

// Everything the kernels read; one k-point travels in `one`, more in `many`.
struct SphereArgs {
    const KindDev* kinds;
    const OverlapGroup* groups;
    const AtomDev* atoms;      // system order
    const int32_t* order;      // [natoms] atoms in kind order
    const RadDev* rad;
    const double* ynorm;
    double bmat[9];
    double vol_prefac;
    int32_t natoms, nkinds, ngroups, max_lmax, nl, L;
    int32_t chunk;             // kinds per LDS chunk of the generator
    int32_t nk, ngcols;        // k-points; plane waves of all of them
    // split precision: the arrays hold columns cbase .. cbase + gtot - 1 of the
    // call, padding columns included (as zeros), and the T application stores
    // row r of W where rowdst[r] says (-1: nowhere)
    int64_t cbase;
    const int32_t* rowdst;     // null: FP64
    SphereK one;
    const SphereK* many;
    int64_t gtot;              // columns of the operand arrays
    int32_t tcols;             // columns of the T application
    // a call in parts (sphere_launch_parts): H columns of the launch, and whether
    // S adds to what an earlier launch left
    int32_t hcol0, hcol1, sadd;
    double2* ph;               // [natoms][gtot] phases, kind order
    double2* rs;               // [gtot][ldr] radial factors per overlap group: (a_l, b_l), then with S's weights
    int32_t ldr;
    double* y;                 // [gtot][ldy] real vectors of all kinds, or null (S alone)
    double2* W;                // [gtot][ldw]
    int64_t ldy, ldw;
    const double2* mt;
    const int64_t* mtoff;      // [natoms] Mt of each atom, kind order
    const SphereStage* stages;
    int32_t nksteps;
    int32_t rtiles;            // T application: tiles of rows of all kinds
    int32_t nsquares;          // lower squares of H tiles of all k-points
    // split precision's FP64 sample: kSampleCols columns per k-point of their own
    // operands, read beside the chunk's; H and S of a k-point are its samples
    const double2* smp_W;
    const double2* smp_ph;     // [natoms][smp_gtot]
    const double2* smp_rs;
    const int32_t* smp_g;      // [smp_gtot][3]
    int64_t smp_ldw, smp_gtot;
    uint64_t* stamp;           // starts of the generator, T application, H and S kernels (wall clock), or null
};

constexpr int kSampleCols = 64;
hipError_t launch_sample_g(const SphereArgs& p, const int32_t* cols, int32_t* out, hipStream_t st);
hipError_t launch_sample(const SphereArgs& p, bool do_h, bool do_s, hipStream_t st);
// Launchers; stop: null, or an event that takes the kernel's end.
int sphere_chunk(int nl, int L);
hipError_t launch_split_mt(const SplitMtJob* jobs, int njobs, int64_t max_elems, const double* sq, const double2* mt,
                           double2* out, hipStream_t st);
hipError_t launch_build_m(const MJob* jobs, int njobs, int64_t max_elems, double2* m, hipStream_t st);
hipError_t launch_build_mt(const MtJob* jobs, int njobs, int64_t max_elems, double2* mt, hipStream_t st);
hipError_t launch_sphere_gen(const SphereArgs& p, hipEvent_t stop, hipStream_t st);
hipError_t launch_sphere_tapp(const SphereArgs& p, int tile, int rtiles, hipEvent_t stop, hipStream_t st);
hipError_t launch_sphere_h(const SphereArgs& p, int tile, hipEvent_t stop, hipStream_t st);
// S tile side by the number of lower tiles; the bits do not depend on it
int overlap_tile_size(int64_t tiles64, int n_cu);
hipError_t launch_overlap(const SphereArgs& p, int tile, int64_t ntiles, hipEvent_t stop, hipStream_t st);
hipError_t launch_sphere_h_part(const SphereArgs& p, hipEvent_t stop, hipStream_t st);
// S of one k-point from the groups of p, added to S as it is where p.sadd
hipError_t launch_overlap_part(const SphereArgs& p, hipEvent_t stop, hipStream_t st);
// H tiles of 32 x 32 (or 16 x 32: tile 16, S tile 16) and S tiles of 16 or 32 in one launch
hipError_t launch_sphere_hs(const SphereArgs& p, int tile, int stile, int64_t nstiles, hipEvent_t stop, hipStream_t st);

}  // namespace hsgen
