// bx_eos_dev.h -- the tabulated H2 equation of state on the device: the table
// layout that bx_eos.hip builds and the lookup of get_gamma2 (eos.f90:653-699),
// shared by the kernels that call state().
#pragma once

#include <climits>

#include "bx_internal.h"
#include "bx_math.h"

namespace bx {

// Fortran INT() of a real(8) as the reference's x86-64 build computes it
// (cvttsd2si): truncation, and INT_MIN for NaN and out-of-range values.
__host__ __device__ __forceinline__ int fort_int(double q)
{
    return (q > -2147483649.0 && q < 2147483648.0) ? (int)q : INT_MIN;
}

// One entry of table 2 at (itk, irho): the values and, for itk < NEOS, the
// slopes (v(itk+1)-v(itk))/(eng2(itk+1)-eng2(itk)) that get_gamma2 forms at
// run time -- the same IEEE divisions of the same table values, done once.
struct alignas(64) TabEntry {
    double eng, gam, muc, tk, sg, sm, st, pad;
};
// The entries (itk, irho) and (itk, irho+1) side by side in one 128-byte
// line: a lookup, which needs both rows at the same itk, reads one line.
struct alignas(128) TabPair {
    TabEntry lo, hi;
};
// Per density row: rho_table(irho), 1/(rho_table(irho+1)-rho_table(irho))
// (NaN where the reference does not interpolate in rho), log10 of the first
// energy, deng_eos_array, and the first and last energies of the row.
struct alignas(64) RhoRow {
    double r0, inv_dr, leng1, deng, e_first, e_last, pad0, pad1;
};

struct EosDev {
    int neos, nrho;
    double log_rho_low, drho, density, tk_bgrnd;
    const TabPair *tab;  // (irho, itk), itk fastest (code units); hi = row irho+1
    const RhoRow *rows;
};

// eos.f90:653-699
__device__ __forceinline__ void get_gamma2(const EosDev &e, double eps, double rho, double &tk, double &m,
                                           double &gam)
{
    int irho = fort_int((log10(rho * e.density) - e.log_rho_low) / e.drho) + 1;
    irho = irho < e.nrho ? irho : e.nrho;
    if (irho < 1) irho = 1;
    const RhoRow R = e.rows[irho - 1];
    double eng = eps / rho;
    int ientry = fort_int((log10(eng) - R.leng1) / R.deng) + 1;
    if (ientry > e.neos - 1) {
        ientry = e.neos - 1;
        eng = R.e_last;
    }
    if (ientry < 1 || eng < R.e_first) {
        ientry = 1;
        eng = R.e_first;
    }
    const TabPair *pr = e.tab + (int64_t)(irho - 1) * e.neos + (ientry - 1);
    const TabEntry a = pr->lo, ap = pr->hi;  // hi: row irho+1 (the row itself on the last row)
    gam = a.gam + a.sg * (eng - a.eng);
    m = a.muc + a.sm * (eng - a.eng);
    tk = a.tk + a.st * (eng - a.eng);
    // rho_table(irho) /= rho_table(irhop): interpolate in rho; written as
    // selects so that no branch waits on the table load
    const double gamp = ap.gam + ap.sg * (eng - ap.eng);
    const double mp = ap.muc + ap.sm * (eng - ap.eng);
    const double tkp = ap.tk + ap.st * (eng - ap.eng);
    const double slope = R.inv_dr * (rho - R.r0);
    const bool interp = R.inv_dr == R.inv_dr;
    gam = interp ? gam + (gamp - gam) * slope : gam;
    m = interp ? m + (mp - m) * slope : m;
    tk = interp ? tk + (tkp - tk) * slope : tk;
}

}  // namespace bx

struct bx_eos {
    bx::EosDev dev;
    bx::TabPair *tab;
    bx::RhoRow *rows;
    double *muc_plane;
};
