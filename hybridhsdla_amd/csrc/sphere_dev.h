// Device functions shared by the generators (abgen.hip, sphere.hip): Bessel
// functions and the angles of a direction, by Fleur's schemes.
#pragma once

#include "hsgen_internal.h"

namespace hsgen {

// Fleur sphbes (sphbes.f:7-76) + dsphbs (dsphbs.f:11-47) for one x; writes
// fj[l], dfj[l] for l = 0..lmax into strided LDS slots.  lmax >= 1, x >= 0.
__device__ inline void bessel_lds(int lmax, double x, double* fj, double* dfj)
{
    const double small = 1.0e-3;
    double xx = x * x;
    if (x >= small) {
        double xinv = 1.0 / x;
        double s, c;
        sincos(x, &s, &c);
        double f0 = s * xinv;
        double f1 = (f0 - c) * xinv;
        fj[0] = f0;
        fj[1] = f1;
        if ((double)lmax < x) {
            double fm2 = f0, fm1 = f1;
            for (int l = 2; l <= lmax; ++l) {
                double f = (2 * l - 1) * xinv * fm1 - fm2;
                fj[l] = f;
                fm2 = fm1;
                fm1 = f;
            }
        } else if (lmax >= 2) {
            // Miller: aux(n) = 0, aux(n-1) = 1, aux(i-1) = (2i+1)/x aux(i) - aux(i+1).
            // n - 1 >= lmax + 9, so every aux(l), l <= lmax, comes out of the loop;
            // they are parked in fj[] and rescaled afterwards.
            int n = (int)(lmax + 10 + x);
            double anext = 0.0, acur = 1.0;
            for (int i = n - 1; i >= 1; --i) {
                double aprev = (2 * i + 1) * xinv * acur - anext;   // aux(i-1)
                if (i - 1 <= lmax) fj[i - 1] = aprev;
                anext = acur;
                acur = aprev;
            }
            // normalise with j0 or j1, whichever is larger in magnitude
            int mn = (fabs(f0) < fabs(f1)) ? 1 : 0;
            double quot = mn ? f1 / fj[1] : f0 / fj[0];
            fj[0] = f0;
            fj[1] = f1;
            for (int l = 2; l <= lmax; ++l) fj[l] = fj[l] * quot;
        }
        // x >= 1e-3 > 1e-4: dsphbs recurrence branch
        dfj[0] = -fj[1];
        for (int l = 1; l <= lmax; ++l) dfj[l] = fj[l - 1] - (l + 1) * fj[l] / x;
    } else {
        fj[0] = 1.0 - xx / 6.0 * (1.0 - xx / 20.0 * (1.0 - xx / 42.0));
        fj[1] = (x / 3.0) * (1.0 - xx / 10.0 * (1.0 - xx / 28.0));
        double fac = xx / 15.0;
        for (int l = 2; l <= lmax; ++l) {
            fj[l] = fac * (1.0 - xx / (4 * l + 6));
            fac = x * fac / (2 * l + 3);
        }
        dfj[0] = -fj[1];
        if (x < 1.0e-4) {
            double x2 = 0.5 * x * x;
            double f = 1.0 / 3.0;
            for (int l = 1; l <= lmax; ++l) {
                dfj[l] = f * (l - x2 * (l + 2) / (2 * l + 3));
                f = x * f / (2 * l + 3);
            }
        } else {
            for (int l = 1; l <= lmax; ++l) dfj[l] = fj[l - 1] - (l + 1) * fj[l] / x;
        }
    }
}

// l of lm = l(l+1)+m, |m| <= l
__device__ inline int l_of_lm(int lm)
{
    int l = (int)sqrtf((float)lm + 0.5f);
    if ((l + 1) * (l + 1) <= lm) ++l;
    if (l * l > lm) --l;
    return l;
}

// Angles of R^T K as ylm4 takes them (ylm4.f:170-191): cos and sin of theta
// and phi, with its conventions at the origin and on the z axis.
struct DirAngles {
    double cth, sth, cph, sph;
};

__device__ inline DirAngles dir_angles(const double* __restrict__ R, double K0, double K1, double K2)
{
    double kb0 = R[0] * K0 + R[1] * K1 + R[2] * K2;   // R^T K
    double kb1 = R[3] * K0 + R[4] * K1 + R[5] * K2;
    double kb2 = R[6] * K0 + R[7] * K1 + R[8] * K2;
    const double nrm = sqrt(kb0 * kb0 + kb1 * kb1 + kb2 * kb2);
    if (nrm != 0.0) {
        kb0 /= nrm;
        kb1 /= nrm;
        kb2 /= nrm;
    }
    const double small = 1.0e-12;
    const double xy = kb0 * kb0 + kb1 * kb1;
    const double r = sqrt(xy + kb2 * kb2);
    const double rxy = sqrt(xy);
    DirAngles d;
    if (r > small) {
        d.cth = kb2 / r;
        d.sth = rxy / r;
    } else {
        d.sth = 0.0;
        d.cth = 1.0;
    }
    if (rxy > small) {
        d.cph = kb0 / rxy;
        d.sph = kb1 / rxy;
    } else {
        d.cph = 1.0;
        d.sph = 0.0;
    }
    return d;
}

}  // namespace hsgen
