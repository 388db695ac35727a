// trk_tables.hip -- Ritchie-Howie CDF quadrature tables on the MI355X.
//
// Replaces the table builders of the reference:
//   TotIMFP                Cross_sections.f90:881-1050   (electron/hole inelastic + aidCS rows)
//   Tot_EMFP               Cross_sections.f90:2966-3139  (phonon-CDF elastic + rows)
//   Elastic_cross_section  Cross_sections.f90:2892-2963  (Mott branch)
//   Tot_Phot_IMFP          Cross_sections.f90:833-878
//   SHI_TotIMFP            Cross_sections.f90:2452-2597  (table and diff_SHI_MFP rows)
//   drivers                Analytical_IMFPs.f90:1830-2239, 2510-2751
//   How_many_electrons     Monte_Carlo.f90:1902-2057 (fused totals)
//
// Design.  The reference integrates row by row on host threads: for each
// incident energy E_i and shell it walks an adaptive omega grid and, at every
// omega node, a geometric q grid (Simpson with the left-node 1/q weight).
// Here the work is split into four launches so that the expensive part -- the
// q integral behind each omega node, ~10^7 of them per material -- runs one
// per lane of waves that each stay inside one row:
//   1. plan   (one wave per row)      walk the omega recurrence, count nodes
//   2. nodes  (one wave per row)      write left node E_k and step dE_k
//   3. eval   (one lane per point)    q-integral at the row start, E_k+dE_k/2, E_k+dE_k
//   4. scan   (one wave per row)      Simpson sums in the reference's order,
//                                      cumulative rows, MFP, dE/dx
// Steps 1, 2 and 4 perform exactly the reference's floating-point operations
// in the reference's order, and step 3 is a pure function of its inputs, so
// the tables are bit-identical to a sequential evaluation.  The q loop is
// VALU-bound FP64 work (a correctly rounded division per oscillator per
// node); it has no dense contraction, so MFMA is not used.
//
// Measured on the MI355X (ms per build: an Al2O3-like target of seven
// oscillators in three shells / an Al-like metal with masses from its density
// of states / the oxide with the FP32 quadrature): eval 42 -> 9.1, 71 -> 15.6
// and 76 -> 10 since a wave takes one row and its loop holds only what changes
// with q (1.75e10 -> 3.4e9 wave instructions, lanes in use 49 -> 98 %), plan and
// nodes 1.6 -> 0.9 and 2.8 -> 1.7, scan 4.6 -> 0.42 and 6.9 -> 0.76.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>
#include "trk_ctx.h"
#include "trk_delta.h"
#include "trk_beb.h"

namespace trk {

#define HIP_OK(x)                                                                 \
    do {                                                                          \
        hipError_t e_ = (x);                                                      \
        if (e_ != hipSuccess) {                                                   \
            err = std::string(#x) + ": " + hipGetErrorString(e_);                 \
            return TRK_ERR_DEVICE;                                                \
        }                                                                         \
    } while (0)

// ---------------------------------------------------------------- physics
// Loss_func (Cross_sections.f90:446-486) with Extend_E0_to_finite_q (346-393).
// mode 0: electron/hole in the target, 1: photon (q = 0), 2: phonon (atoms).
TRK_DEV double loss(const MatDev &m, int mode, double A, double E, double G, double dE, double dq)
{
    double E0, G1;
    if (mode == 1) {
        G1 = G;
        E0 = E;
    } else {
        double hq2 = ((kH * kH) * dq) * dq;
        if (mode == 2) {
            E0 = E + hq2 / (2.0 * m.Mtarget);
            G1 = G;
        } else {
            double Mass;
            if (m.use_k) {
                double qlim = trk_fabs(dq) * trk_sqrt(kE);
                if (qlim <= m.k[m.nk - 1]) {
                    int j = find_mono_1d(m.k, m.nk, qlim);
                    Mass = m.Effm[j - 1];
                } else {
                    Mass = 1.0;
                }
            } else if (m.El_eff_mass > 0.0) {
                Mass = m.El_eff_mass;
            } else {
                Mass = 1.0;
            }
            double sqq = hq2 / ((2.0 * Mass) * kMe);
            if (m.kind_of_DR == 2) {
                E0 = trk_sqrt(((E * E) + (((m.v_f * m.v_f) * hq2) * 0.3333333333333)) + (sqq * sqq));
                G1 = G;
            } else if (m.kind_of_DR == 3) {
                E0 = trk_pow(trk_pow(E, 0.666666666666) + trk_pow(sqq, 0.666666666666), 1.5);
                G1 = trk_sqrt((G * G) + (sqq * sqq));
            } else {
                E0 = E + sqq;
                G1 = G;
            }
        }
    }
    double dE2 = dE * dE;
    double E02 = E0 * E0;
    return ((A * G1) * dE) / (((dE2 - E02) * (dE2 - E02)) + ((G1 * G1) * dE2));
}

// Imewq, Cross_sections.f90:397-442
TRK_DEV double imewq(const MatDev &m, double hw, double hq, int shell, int photon)
{
    double ImE = 0.0;
    const int o1 = m.osc_off[shell + 1];
    for (int i = m.osc_off[shell]; i < o1; ++i)
        ImE = ImE + loss(m, photon ? 1 : 0, m.oA[i], m.oE0[i], m.oG[i], hw, hq);
    return ImE;
}

// The q quadratures advance by 1% per step, a few thousand steps over any
// physical range; the step limit only ends a loop whose start is 0 or NaN.
constexpr int kMaxQSteps = 1 << 20;
// Nodes of one transfer-energy row (the reference's rows hold up to ~1400).
constexpr int kMaxRowSteps = 1 << 20;

// ---- the q quadrature of one point
// Quotients of the quadrature's inner loop.  recip and quot are the steps of
// the hardware's full division without its operand scaling and special cases:
// the same rounded result wherever a full division would not scale, which
// q_in_range states for a whole point before its loop starts.
TRK_DEV double recip(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}
TRK_DEV double quot(double n, double d, double y)
{
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
}
// n / c for a constant c, y the rounded 1/c.  One correction of n y is the
// rounded quotient (Markstein's theorem) if n y lies within 1 ulp of it,
// which |c y - 1| <= 2^-54 ensures (100 and 6); with any other c a second
// correction follows.
TRK_DEV double quot_const(double n, double c, double y) { return quot(n, c, y); }
TRK_HD double quot_any(double n, double c, double y)
{
    double q = n * y;
    q = __builtin_fma(__builtin_fma(-c, q, n), y, q);
    return __builtin_fma(__builtin_fma(-c, q, n), y, q);
}

// The oscillators of a point's sum: a shell's, or the phonons.
struct OscSpan {
    const double *A, *E, *G;
    int n;
};

// The effective masses of a density of states in LDS: the momenta k, and of
// every interval the denominator (2 m*) m_e with its reciprocal.
struct DosMass {
    const double *k, *c, *y;
    int nk;
};
constexpr int kMaxDosMass = 2048;    // 48 KB of LDS
constexpr double kOneCv = (2.0 * 1.0) * kMe;

// Every quotient of the loop stays far from the ends of the exponent range,
// and every numerator is non-zero.
// The bounds leave numerators in 1e-60..1e60 over denominators in
// 1e-60..1e100, their Simpson terms in 1e-210..1e180 over momenta in
// 1e-30..1e60, so no quotient nor reciprocal comes near 2^+-768.
TRK_DEV bool q_in_range(const OscSpan &o, double w, double cmin, double cmax, double qmin, double qmax)
{
    bool ok = qmin >= 1.0e-30 && qmax <= 1.0e60 && w >= 1.0e-24 && w <= 1.0e24 && cmin >= 1.0e-60 && cmax <= 1.0e60;
    const double top = qmax * 1.02;
    const double smax = ((kH * kH) * top) * top;
    ok = ok && smax <= 1.0e23 * cmin;
    for (int i = 0; i < o.n; ++i) {
        const double num = trk_fabs((o.A[i] * o.G[i]) * w), g2 = (o.G[i] * o.G[i]) * (w * w);
        ok = ok && num >= 1.0e-60 && num <= 1.0e60 && g2 >= 1.0e-60 && g2 <= 1.0e60 && trk_fabs(o.E[i]) <= 1.0e23;
    }
    return ok;
}

// Simpson over the geometric q grid (left-node 1/q weight) of the loss
// function with E0(q) = E + hbar^2 q^2 / c.  Bound by FP64 issue: per step
// and oscillator two terms of 18 operations, 11 of them the quotient.  What
// does not change along the loop (A G w, G^2 w^2, 1/c) is computed before it,
// the step's own quotients (by 100, 6 and c) are multiplications by a rounded
// reciprocal with correction, and both nodes of a step share one pass over
// the oscillators.  kN oscillators (0: any number, read in the loop);
// kDos: c follows q through the density of states; kPh: weight 1/q as a factor.
template <int kN, bool kDos, bool kPh>
TRK_DEV double q_simpson(const OscSpan &o, const DosMass &dm, double w, double c, double qmin, double qmax)
{
    constexpr int kA = kN ? kN : 1;
    const int n = kN ? kN : o.n;
    const double w2 = w * w;
    double num[kA], g2[kA], E[kA];
    if (kN) {
#pragma unroll
        for (int i = 0; i < kA; ++i) {
            num[i] = (o.A[i] * o.G[i]) * w;
            g2[i] = (o.G[i] * o.G[i]) * w2;
            E[i] = o.E[i];
        }
    }
    constexpr double y100 = 1.0 / 100.0, y6 = 1.0 / 6.0;
    const double rootE = kDos ? trk_sqrt(kE) : 0.0;
    double y = kDos ? 0.0 : 1.0 / c;
    // kDos: the interval of q is the number of k entries not above it; q only
    // grows, so it is looked for once and then followed.  One past the last
    // entry the mass is that entry's; beyond, the free electron's.
    int at = 0;
    double knext = 0.0;
    auto interval = [&](double v) {
        while (v >= knext) {
            ++at;
            if (at < dm.nk) {
                knext = dm.k[at];
                c = dm.c[at];
                y = dm.y[at];
            } else if (at == dm.nk) {
                knext = __longlong_as_double(__double_as_longlong(dm.k[dm.nk - 1]) + 1);
                c = dm.c[dm.nk - 1];
                y = dm.y[dm.nk - 1];
            } else {
                knext = __builtin_inf();
                c = kOneCv;
                y = recip(kOneCv);
            }
        }
    };
    // An empty range (qmin not below qmax) may come with limits that are not
    // finite, as an infinite hole mass gives: no look then, interval would
    // never pass an infinite momentum.
    if (kDos && qmin < qmax) {
        const double v = qmin * rootE;
        int lo = -1, hi = dm.nk;      // k[lo] <= v < k[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (dm.k[mid] <= v) lo = mid;
            else hi = mid;
        }
        at = hi - 1;
        knext = -__builtin_inf();     // the first look sets c and y
        interval(v);
    }
    double dLs = 0.0, hq = qmin, dLs0 = 0.0;
    for (int g = 0; hq < qmax && g < kMaxQSteps; ++g) {
        const double dq = quot_const(hq, 100.0, y100);
        const double a = hq + dq * 0.5;
        const double b = hq + dq;
        const double ha = ((kH * kH) * a) * a, hb = ((kH * kH) * b) * b;
        double sa, sb;
        if (kDos) {
            interval(a * rootE);
            sa = quot(ha, c, y);
            interval(b * rootE);
            sb = quot(hb, c, y);
        } else {
            sa = quot_any(ha, c, y);
            sb = quot_any(hb, c, y);
        }
        double Fa = 0.0, Fb = 0.0;
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const double nu = kN ? num[kN ? i : 0] : (o.A[i] * o.G[i]) * w;
            const double gg = kN ? g2[kN ? i : 0] : (o.G[i] * o.G[i]) * w2;
            const double Ei = kN ? E[kN ? i : 0] : o.E[i];
            const double Ea = Ei + sa, Eb = Ei + sb;
            const double xa = w2 - Ea * Ea, xb = w2 - Eb * Eb;
            const double da = xa * xa + gg, db = xb * xb + gg;
            Fa = Fa + quot(nu, da, recip(da));
            Fb = Fb + quot(nu, db, recip(db));
        }
        const double t = quot_const(dq, 6.0, y6) * ((dLs0 + 4.0 * Fa) + Fb);
        const double yq = recip(hq);
        dLs = dLs + (kPh ? t * quot(1.0, hq, yq) : quot(t, hq, yq));
        dLs0 = Fb;
        hq = b;
    }
    return dLs;
}

template <bool kDos, bool kPh>
TRK_DEV double q_simpson_n(const OscSpan &o, const DosMass &dm, double w, double c, double qmin, double qmax)
{
    switch (o.n) {
    case 1: return q_simpson<1, kDos, kPh>(o, dm, w, c, qmin, qmax);
    case 2: return q_simpson<2, kDos, kPh>(o, dm, w, c, qmin, qmax);
    case 3: return q_simpson<3, kDos, kPh>(o, dm, w, c, qmin, qmax);
    case 4: return q_simpson<4, kDos, kPh>(o, dm, w, c, qmin, qmax);
    case 5: return q_simpson<5, kDos, kPh>(o, dm, w, c, qmin, qmax);
    default: return q_simpson<0, kDos, kPh>(o, dm, w, c, qmin, qmax);
    }
}

// The q integral of one point: the form above for the free-electron
// dispersion, else (plasmon-pole and Ritchie dispersions, densities of states
// whose k do not increase, values outside q_in_range in any lane) the loss
// function as it is written.  shell < 0: the phonons.  All lanes of a wave
// come here with the same shell.
TRK_DEV double q_integral(const MatDev &m, const DosMass &dm, int shell, double w, double qmin, double qmax)
{
    const bool ph = shell < 0;
    OscSpan o;
    if (ph) o = OscSpan{m.phA, m.phE0, m.phG, m.n_ph};
    else {
        const int o0 = m.osc_off[shell];
        o = OscSpan{m.oA + o0, m.oE0 + o0, m.oG + o0, m.osc_off[shell + 1] - o0};
    }
    const bool dos = !ph && m.use_k;
    if ((ph || (m.kind_of_DR != 2 && m.kind_of_DR != 3)) && (!dos || dm.nk > 0)) {
        double c;
        if (ph) c = 2.0 * m.Mtarget;
        else c = (2.0 * ((m.El_eff_mass > 0.0) ? m.El_eff_mass : 1.0)) * kMe;
        // the masses of a usable density of states lie in 1e-6..1e6
        const bool ok = dos ? q_in_range(o, w, 1.0e-6 * kOneCv, 1.0e6 * kOneCv, qmin, qmax) : q_in_range(o, w, c, c, qmin, qmax);
        if (!__any(!ok && qmin < qmax)) {
            if (ph) return q_simpson_n<false, true>(o, dm, w, c, qmin, qmax);
            if (dos) return q_simpson_n<true, false>(o, dm, w, c, qmin, qmax);
            return q_simpson_n<false, false>(o, dm, w, c, qmin, qmax);
        }
    }
    double dLs = 0.0, hq = qmin, dLs0 = 0.0;
    for (int g = 0; (ph ? trk_fabs(hq) < trk_fabs(qmax) : hq < qmax) && g < kMaxQSteps; ++g) {
        double dq = hq / 100.0;
        double a = hq + dq / 2.0;
        double b = hq + dq;
        double temp1 = 0.0, dL = 0.0;
        for (int i = 0; i < o.n; ++i) temp1 = temp1 + loss(m, ph ? 2 : 0, o.A[i], o.E[i], o.G[i], w, a);
        for (int i = 0; i < o.n; ++i) dL = dL + loss(m, ph ? 2 : 0, o.A[i], o.E[i], o.G[i], w, b);
        const double t = (dq / 6.0) * ((dLs0 + 4.0 * temp1) + dL);
        if (ph) dLs = dLs + t * (1.0 / hq);
        else dLs = dLs + t / hq;
        dLs0 = dL;
        hq = hq + dq;
    }
    return dLs;
}

// Diff_cross_section, Cross_sections.f90:2217-2282
TRK_DEV double diff_cs(const MatDev &m, const DosMass &dm, int shell, double Ee, double dE, double Mass)
{
    double qmin, qmax;
    double pre = trk_sqrt((2.0 * Mass) * kMe) / kH;
    if (dE > Ee) {
        qmin = pre * trk_sqrt(Ee);
        qmax = pre * trk_sqrt(Ee);
    } else {
        qmin = pre * (trk_sqrt(Ee) - trk_sqrt(Ee - dE));
        qmax = pre * (trk_sqrt(Ee) + trk_sqrt(Ee - dE));
    }
    const double dLs = q_integral(m, dm, shell, dE, qmin, qmax);
    double T_fact = (m.temp > 0.0) ? 1.0 / (1.0 - trk_exp(-((dE / m.temp) * kKb))) : 1.0;
    return ((1.0 / ((kPi * kA0) * Ee)) * dLs) * T_fact;
}

// Diff_cross_section_phonon, Cross_sections.f90:3142-3300 (screening 1)
TRK_DEV double diff_cs_phonon(const MatDev &m, const DosMass &dm, double Ee, double dE, double Mass)
{
    const double eps = 1.0e-12;
    double qmin, qmax;
    double pre = trk_sqrt((2.0 * Mass) * kMe) / kH;
    if (trk_fabs(dE) < eps) return 1.31e30;
    else if (dE > (Ee - eps)) qmin = pre * trk_sqrt(Ee);
    else qmin = pre * (trk_sqrt(Ee) - trk_sqrt(trk_fabs(Ee - dE)));
    qmax = ((1.0 * trk_sqrt((2.0 * Mass) * kMe)) / kH) * (trk_sqrt(Ee) + trk_sqrt(trk_fabs(Ee - dE)));
    const double dLs = q_integral(m, dm, -1, dE, qmin, qmax);
    if (m.temp > 1.0e-6)
        return ((1.0 / ((kPi * kA0) * Ee)) * dLs) / (1.0 - trk_exp(-((dE / m.temp) * kKb)));
    return (1.0 / ((kPi * kA0) * Ee)) * dLs;
}

// SHI_Diff_cross_section, Cross_sections.f90:2683-2744
TRK_DEV double shi_diff_cs(const MatDev &m, const DosMass &dm, int shell, double Ee, double MSHI, double Emax, double hw)
{
    double qmin, qmax;
    if (Ee > 0.0) qmin = (hw / kH) / trk_sqrt((2.0 * Ee) / MSHI);
    else qmin = 0.0;
    if (Emax > 0.0) qmax = (trk_sqrt(2.0 * kMe) / kH) * trk_sqrt(Emax);
    else return 0.0;
    const double dLs = q_integral(m, dm, shell, hw, qmin, qmax);
    double T_fact = (m.temp > 0.0) ? 1.0 / (1.0 - trk_exp(-((hw / m.temp) * kKb))) : 1.0;
    return dLs * T_fact;
}

// Brand_Kitagawa, Cross_sections.f90:2878-2889: the effective charge of an
// ion of nuclear charge Zp and equilibrium charge Zeff seen at momentum
// transfer hq (reference units: [sqrt(eV/J)/m], times a0 sqrt(e) in metres)
TRK_DEV double bk_charge(double hq, double Zp, double Zeff)
{
    const double a = 0.2400519147;
    const double Z = (Zp - Zeff) / Zp;
    const double Z23 = (Z == 0.0) ? 0.0 : trk_pow(Z, 2.0 / 3.0);   // 0**(2/3) = 0
    const double kl = ((((hq * ((kA0 * 1.0e-10) * trk_sqrt(kE))) * 2.0) * a) * Z23) /
                      (trk_pow(Zp, 2.0 / 3.0) * (1.0 - Z / 7.0));
    const double kl2 = kl * kl;
    return (Zp * ((1.0 - Z) + kl2)) / (1.0 + kl2);
}

// SHI_Diff_cross_section_BK, Cross_sections.f90:2826-2875: the point-charge
// integrand weighted by the squared Brandt-Kitagawa charge at each q
TRK_DEV double shi_diff_cs_bk(const MatDev &m, int shell, double Ee, double MSHI, double Emax, double hw, double Zp,
                              double Zeff)
{
    const double qmin = (hw / kH) / trk_sqrt((2.0 * Ee) / MSHI);
    const double qmax = (trk_sqrt(2.0 * kMe) / kH) * trk_sqrt(Emax);
    double dLs = 0.0, hq = qmin, dLs0 = 0.0;
    for (int g = 0; hq < qmax && g < kMaxQSteps; ++g) {
        double dq = hq / 100.0;
        double a = hq + dq / 2.0;
        double rho = bk_charge(a, Zp, Zeff);
        double temp1 = (imewq(m, hw, a, shell, 0) * rho) * rho;
        double b = hq + dq;
        rho = bk_charge(b, Zp, Zeff);
        double dL = (imewq(m, hw, b, shell, 0) * rho) * rho;
        dLs = dLs + ((dq / 6.0) * ((dLs0 + 4.0 * temp1) + dL)) / hq;
        dLs0 = dL;
        hq = hq + dq;
    }
    // dLs / (1 - exp(-hw/T kB)); at T = 0 the exponential is 0
    if (m.temp > 0.0) return dLs / (1.0 - trk_exp(-((hw / m.temp) * kKb)));
    return dLs;
}

// ---------------------------------------------------------------- row jobs
enum RowType { ROW_INEL = 0, ROW_PHONON = 1, ROW_SHI = 2, ROW_SHI_DIFF = 3 };

struct RowJob {
    double Ele, Estart, Emax, E_low, E_high, dE_min, Mass, Zeff, MSHI;
    double Zp;   // the ion's nuclear charge (ROW_SHI with bk)
    int n, shell, type, with_row;
    int kind, ie;
    int q32;     // FP32 compensated quadrature (ROW_INEL, ROW_SHI, ROW_SHI_DIFF)
    int bk;      // ROW_SHI of a Brandt-Kitagawa ion (SHI_TotIMFP_BK, CS:2748-2823)
};

// ---------------------------------------------------------------- FP32 quadrature
// The same cross sections with the quadrature of the precision form: kQ32W
// transfer-energy intervals, geometric from Estart to Emax, each with its
// midpoint (4001 points), and at each point kQ32Q Simpson intervals in ln q
// (2001 points), evaluated and summed in FP32 with compensated (Kahan) sums.
// Momenta are carried as q/q1 with q1 = sqrt(2 m_e * 1 eV)/hbar, so that
// hbar^2 q^2 / (2 m* m_e) is (q/q1)^2 / m* eV and every FP32 value stays in
// range; int dq/q is int d(ln q), unchanged by the scale.
constexpr int kQ32W = 2000;
constexpr int kQ32Q = 1000;

struct Kahan32 {
    float s = 0.0f, c = 0.0f;
    TRK_DEV void add(float x)
    {
        const float y = x - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
    TRK_DEV double value() const { return (double)s - (double)c; }
};

// Imewq with Loss_func and the dispersion of Extend_E0_to_finite_q (CS:346-486)
// for a constant effective mass, in FP32; q2 = (q/q1)^2.
TRK_DEV float imewq32(const MatDev &m, int shell, float w, float q2, float inv_mstar, float c_vf)
{
    const float sqq = q2 * inv_mstar;
    const float w2 = w * w;
    float ImE = 0.0f;
    const int o1 = m.osc_off[shell + 1];
    for (int i = m.osc_off[shell]; i < o1; ++i) {
        const float E = (float)m.oE0[i], G = (float)m.oG[i], A = (float)m.oA[i];
        float E0, G1;
        if (m.kind_of_DR == 2) {
            E0 = sqrtf(E * E + c_vf * q2 + sqq * sqq);
            G1 = G;
        } else if (m.kind_of_DR == 3) {
            E0 = powf(powf(E, 0.666666666666f) + powf(sqq, 0.666666666666f), 1.5f);
            G1 = sqrtf(G * G + sqq * sqq);
        } else {
            E0 = E + sqq;
            G1 = G;
        }
        const float d = w2 - E0 * E0;
        ImE = ImE + (A * G1 * w) / (d * d + G1 * G1 * w2);
    }
    return ImE;
}

// n / d in FP32: the steps of the hardware's full division without its
// scaling and special cases, the same rounded result inside in_range32.
TRK_DEV float quot32(float n, float d)
{
    float y = __builtin_amdgcn_rcpf(d);
    y = __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
    float q = n * y;
    q = __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), y, q);
}

// Numerators in 1e-6..1e10 over denominators in 1e-12..1e30: quotients of
// 1e-36..1e22, where no operand is scaled.
TRK_DEV bool in_range32(const OscSpan &o, float w, double qhi, float inv_mstar)
{
    const float smax = ((float)qhi * (float)qhi) * 1.01f * inv_mstar;
    bool ok = w >= 1.0e-7f && w <= 1.0e7f && smax >= 0.0f && smax <= 1.0e7f;
    for (int i = 0; i < o.n; ++i) {
        const float E = (float)o.E[i], G = (float)o.G[i], A = (float)o.A[i];
        const float num = fabsf(A * G * w), g2 = G * G * (w * w);
        ok = ok && num >= 1.0e-6f && num <= 1.0e10f && g2 >= 1.0e-12f && g2 <= 1.0e28f && E >= 0.0f && E <= 1.0e7f;
    }
    return ok;
}

// The Simpson sum over ln q with the free-electron dispersion and kN
// oscillators (0: any number).  Bound by FP32 issue, one quotient per
// oscillator and node; the numerators and widths are converted and
// multiplied once per point.
template <int kN>
TRK_DEV double q32_simpson(const OscSpan &o, float w, float u0, float h, float inv_mstar)
{
    constexpr int kA = kN ? kN : 1;
    const int n = kN ? kN : o.n;
    const float w2 = w * w;
    float num[kA], g2[kA], E[kA];
    if (kN) {
#pragma unroll
        for (int i = 0; i < kA; ++i) {
            const float G = (float)o.G[i], A = (float)o.A[i];
            num[i] = A * G * w;
            g2[i] = G * G * w2;
            E[i] = (float)o.E[i];
        }
    }
    auto term = [&](int k) {
        const float q = __expf(u0 + h * (float)k);
        const float sqq = (q * q) * inv_mstar;
        float f = 0.0f;
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const float G = kN ? 0.0f : (float)o.G[i];
            const float nu = kN ? num[kN ? i : 0] : (float)o.A[i] * G * w;
            const float gg = kN ? g2[kN ? i : 0] : G * G * w2;
            const float E0 = (kN ? E[kN ? i : 0] : (float)o.E[i]) + sqq;
            const float d = w2 - E0 * E0;
            f = f + quot32(nu, d * d + gg);
        }
        return f;
    };
    Kahan32 S;
    S.add(1.0f * term(0));
    for (int k = 1; k + 1 < kQ32Q; k += 2) {
        const float f1 = term(k), f2 = term(k + 1);
        S.add(4.0f * f1);
        S.add(2.0f * f2);
    }
    S.add(4.0f * term(kQ32Q - 1));
    S.add(1.0f * term(kQ32Q));
    return S.value();
}

// One point of a row: the q integral of Diff_cross_section (CS:2217-2282) or
// SHI_Diff_cross_section (CS:2683-2744) at transfer energy x, in FP32.
TRK_DEV double eval32(const MatDev &m, const RowJob &j, double x)
{
    // limits in units of q1 (FP64), then the integral in FP32
    double qlo, qhi, pref;
    if (j.type == ROW_INEL) {
        if (!(x < j.Ele)) return 0.0;
        const double sm = trk_sqrt(j.Mass), se = trk_sqrt(j.Ele), sr = trk_sqrt(j.Ele - x);
        qlo = sm * (se - sr);
        qhi = sm * (se + sr);
        pref = 1.0 / ((kPi * kA0) * j.Ele);
    } else {
        if (!(j.Ele > 0.0) || !(j.Emax > 0.0)) return 0.0;
        const double q1 = trk_sqrt(2.0 * kMe) / kH;
        qlo = ((x / kH) / trk_sqrt((2.0 * j.Ele) / j.MSHI)) / q1;
        qhi = trk_sqrt(j.Emax);
        pref = 1.0;
    }
    if (m.temp > 0.0) pref = pref / (1.0 - trk_exp(-((x / m.temp) * kKb)));
    if (!(qlo > 0.0) || !(qhi > qlo)) return 0.0;
    const float inv_mstar = (float)(1.0 / m.El_eff_mass);
    const float c_vf = (float)(((m.v_f * m.v_f) * (2.0 * kMe)) / 3.0);
    const float u0 = (float)trk_log(qlo), h = (float)((trk_log(qhi) - trk_log(qlo)) / (double)kQ32Q);
    const float w = (float)x;
    const int s0 = m.osc_off[j.shell];
    const OscSpan o{m.oA + s0, m.oE0 + s0, m.oG + s0, m.osc_off[j.shell + 1] - s0};
    double S;
    if (m.kind_of_DR != 2 && m.kind_of_DR != 3 && !__any(!in_range32(o, w, qhi, inv_mstar))) {
        switch (o.n) {
        case 1: S = q32_simpson<1>(o, w, u0, h, inv_mstar); break;
        case 2: S = q32_simpson<2>(o, w, u0, h, inv_mstar); break;
        case 3: S = q32_simpson<3>(o, w, u0, h, inv_mstar); break;
        case 4: S = q32_simpson<4>(o, w, u0, h, inv_mstar); break;
        case 5: S = q32_simpson<5>(o, w, u0, h, inv_mstar); break;
        default: S = q32_simpson<0>(o, w, u0, h, inv_mstar); break;
        }
    } else {
        Kahan32 K;
        for (int k = 0; k <= kQ32Q; ++k) {
            const float q = __expf(u0 + h * (float)k);
            const float f = imewq32(m, j.shell, w, q * q, inv_mstar, c_vf);
            const float wk = (k == 0 || k == kQ32Q) ? 1.0f : ((k & 1) ? 4.0f : 2.0f);
            K.add(wk * f);
        }
        S = K.value();
    }
    return (double)((float)pref * ((h / 3.0f) * (float)S));
}

// define_dE (CS:1374-1412) along a row, the nodes E_k+1 = E_k + dE(E_k).  One
// chain of dependent operations per row, so a wave walks it for all its
// lanes, 64 steps without a branch (lane t keeps node t), and the quotient by
// n is a multiplication by its rounded reciprocal with one correction
// (quot_const; a full division where n or the range do not allow it).
struct RowWalk {
    double n, y, lo, hi, inner, dE_min;
    bool quick;
    TRK_DEV explicit RowWalk(const RowJob &j)
        : n((double)j.n), y(1.0 / (double)j.n), lo(j.E_low), hi(j.E_high), inner((j.E_high - j.E_low) / (double)j.n),
          dE_min(j.dE_min)
    {
        quick = j.Estart >= 1.0e-200 && j.E_low >= 1.0e-200 && j.Emax <= 1.0e200 &&
                trk_fabs(__builtin_fma(n, y, -1.0)) <= 0x1.0p-54;
    }
    template <bool kQuick>
    TRK_DEV double step(double E) const
    {
        const double q = kQuick ? quot_const(E, n, y) : E / n;
        const double dE = ((E > lo) & (E < hi)) ? inner : q;
        return (dE > dE_min) ? dE : dE_min;
    }
    template <bool kQuick>
    TRK_DEV void walk(double &E, double &node, double &width) const
    {
        const int lane = threadIdx.x & 63;
#pragma unroll 8
        for (int t = 0; t < 64; ++t) {
            const double dE = step<kQuick>(E);
            if (lane == t) {
                node = E;
                width = dE;
            }
            E = E + dE;
        }
    }
    // the next 64 nodes from E on, and their steps; E moves behind them
    TRK_DEV void next(double &E, double &node, double &width) const
    {
        if (quick) walk<true>(E, node, width);
        else walk<false>(E, node, width);
    }
    // nodes from E on up to Emax
    TRK_DEV int count(double E, double Emax) const
    {
        for (int c = 0; c < kMaxRowSteps; c += 64) {
            double node = 0.0, width = 0.0;
            next(E, node, width);
            const unsigned long long in = __ballot(node <= Emax);
            if (~in) return c + __builtin_ctzll(~in);
        }
        return kMaxRowSteps;
    }
};

// One wave per row.
__global__ void k_row_plan(const RowJob *__restrict__ jobs, int nrows, int *__restrict__ cnt, int *__restrict__ len)
{
    const int r = blockIdx.x * (blockDim.x / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
    if (r >= nrows) return;
    const RowJob j = jobs[r];
    int c = 0, L = 0;
    if (j.q32) {
        // the fixed geometric intervals of the FP32 quadrature (none when
        // the range is empty); rows hold at least 10 entries, as the
        // reference's allocation does
        c = (j.Emax > j.Estart && j.Estart > 0.0) ? kQ32W : 0;
        if (j.with_row) L = (j.type == ROW_SHI_DIFF) ? c : (c > 10 ? c : 10);
    } else {
        const RowWalk w(j);
        // phonon rows compare the magnitudes; they start at a positive energy
        c = (j.type == ROW_PHONON) ? w.count(j.Estart, trk_fabs(j.Emax)) : w.count(j.Estart, j.Emax);
        if (c >= kMaxRowSteps) {
            c = -1;
        } else if (j.with_row) {
            if (j.type == ROW_SHI_DIFF) {
                L = c;
            } else {
                // allocation count of get_diff_CS_grid_size (CS:1278-1343): from E_low
                const int nref = w.count(j.E_low, j.Emax);
                L = c;
                if (nref > L) L = nref;
                if (L < 10) L = 10;
            }
        }
    }
    if ((threadIdx.x & 63) == 0) {
        cnt[r] = c;
        len[r] = L;
    }
}

// Points of a row: its start, then the midpoint and the right node of every
// step.  A wave of k_eval takes kPointsWave points of one row.
constexpr int kPointsWave = 64;
constexpr int kEvalBlock = 256;
TRK_HD int64_t row_chunks(int64_t steps) { return (2 * steps + 1 + kPointsWave - 1) / kPointsWave; }

__global__ void k_row_nodes(const RowJob *__restrict__ jobs, int nrows, const int64_t *__restrict__ step_off,
                            const int64_t *__restrict__ chunk_off, double *__restrict__ Ek, double *__restrict__ dEk,
                            int *__restrict__ chunk_row)
{
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * (blockDim.x / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
    if (r >= nrows) return;
    const RowJob j = jobs[r];
    const int64_t o = step_off[r], n = step_off[r + 1] - o;
    for (int64_t c = chunk_off[r] + lane; c < chunk_off[r + 1]; c += 64) chunk_row[c] = r;
    if (j.q32) {
        const double lr = trk_log(j.Emax / j.Estart) / (double)kQ32W;
        for (int64_t i = lane; i < n; i += 64) {
            const double a = j.Estart * trk_exp(lr * (double)i);
            const double b = (i + 1 == n) ? j.Emax : j.Estart * trk_exp(lr * (double)(i + 1));
            Ek[o + i] = a;
            dEk[o + i] = b - a;
        }
        return;
    }
    const RowWalk w(j);
    double E = j.Estart;
    for (int64_t i = 0; i < n; i += 64) {
        double node = 0.0, width = 0.0;
        w.next(E, node, width);
        if (i + lane < n) {
            Ek[o + i + lane] = node;
            dEk[o + i + lane] = width;
        }
    }
}

TRK_DEV double eval_point(const MatDev &m, const DosMass &dm, const RowJob &j, double x)
{
    if (j.q32) return eval32(m, j, x);
    switch (j.type) {
    case ROW_INEL: return diff_cs(m, dm, j.shell, j.Ele, x, j.Mass);
    case ROW_PHONON: return diff_cs_phonon(m, dm, j.Ele, x, j.Mass);
    default:
        if (j.bk) return shi_diff_cs_bk(m, j.shell, j.Ele, j.MSHI, j.Emax, x, j.Zp, j.Zeff);
        return shi_diff_cs(m, dm, j.shell, j.Ele, j.MSHI, j.Emax, x);
    }
}

// One q integral per lane, a wave's points all of one row: the row's job, its
// shell's oscillators and the number of them are then scalars, and
// neighbouring lanes take nearly the same number of q steps.  A row ends
// its last wave short (half a wave of some hundred points).  dos_n: entries of
// the density of states to stage for the masses (0: none).
__global__ void __launch_bounds__(kEvalBlock, 6)
k_eval(MatDev m, const RowJob *__restrict__ jobs, const int *__restrict__ chunk_row,
       const int64_t *__restrict__ chunk_off, const int64_t *__restrict__ step_off, int64_t nchunks,
       const double *__restrict__ Ek, const double *__restrict__ dEk, double *__restrict__ f0,
       double *__restrict__ fa, double *__restrict__ fb, int dos_n)
{
    extern __shared__ double lds[];
    for (int i = threadIdx.x; i < dos_n; i += kEvalBlock) {
        const double c = (2.0 * m.Effm[i]) * kMe;
        lds[i] = m.k[i];
        lds[dos_n + i] = c;
        lds[2 * dos_n + i] = recip(c);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t c0 = (int64_t)blockIdx.x * (kEvalBlock / kPointsWave) +
                       __builtin_amdgcn_readfirstlane((int)threadIdx.x / kPointsWave);
    if (c0 >= nchunks) return;
    const int r = __builtin_amdgcn_readfirstlane(chunk_row[c0]);
    const RowJob j = jobs[r];
    const int64_t o = step_off[r];
    const int64_t p = (c0 - chunk_off[r]) * kPointsWave + lane;
    if (p > 2 * (step_off[r + 1] - o)) return;
    const DosMass dm{lds, lds + dos_n, lds + 2 * dos_n, dos_n};
    const int64_t k = o + ((p - 1) >> 1);
    double x = j.Estart;
    if (p > 0) x = Ek[k] + ((p & 1) ? dEk[k] / 2.0 : dEk[k]);
    const double f = eval_point(m, dm, j, x);
    if (p == 0) f0[r] = f;
    else if (p & 1) fa[k] = f;
    else fb[k] = f;
}

// inv[k] = 1/L[k] for one row of the ion's transfer table; *nonmono is set
// if the inverse ever decreases (or is NaN) along the row.
__global__ void k_inv_row(const double *__restrict__ L, int n, double *__restrict__ inv, int *nonmono)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    double a = 1.0 / L[k];
    inv[k] = a;
    if (k + 1 < n) {
        double b = 1.0 / L[k + 1];
        if (!(a <= b)) atomicOr(nonmono, 1);
    }
}

__global__ void k_log(const double *__restrict__ x, int64_t n, double *__restrict__ out)
{
    int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = trk_log(x[k]);
}

// mono[slot] = 1 if lam of the row never increases (and holds no NaN): the
// row search can then count entries instead of bisecting
// One wave per row, 64 entries at a time.
__global__ void k_row_mono(const int64_t *__restrict__ off, int64_t nslots, const double *__restrict__ lam,
                           unsigned char *__restrict__ mono)
{
    const int64_t k = (int64_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
    if (k >= nslots) return;
    const int64_t a = off[k], b = off[k + 1];
    bool bad = false;
    for (int64_t i = a + (threadIdx.x & 63); i < b; i += 64) {
        const double v = lam[i];
        if (!(v == v)) bad = true;
        if (i + 1 < b && !(v >= lam[i + 1])) bad = true;
    }
    const bool any = __any(bad);
    if ((threadIdx.x & 63) == 0) mono[k] = any ? 0 : 1;
}

struct RowOut {
    double *L, *dEdx;        // table arrays for the row's kind (shell-major)
    int n;                   // table grid size
    double *hw, *lam;        // concatenated rows of the kind
    const int64_t *row_off;  // [nsh*n+1]
};

TRK_DEV double lane_value(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// One wave per row, 64 steps at a time: the lanes load the steps' values
// coalesced, compute their Simpson terms, and the wave adds them one after the
// other in the row's order (each sum is a chain of rounded additions, so
// its order is the result); every lane keeps its own partial sum and
// writes its entry of the row.  A thread per row waited for memory at every
// step instead.
__global__ void k_row_scan(const RowJob *__restrict__ jobs, int nrows, const int64_t *__restrict__ step_off,
                           const double *__restrict__ Ek, const double *__restrict__ dEk,
                           const double *__restrict__ f0, const double *__restrict__ fa,
                           const double *__restrict__ fb, const RowOut *__restrict__ outs,
                           double *__restrict__ dE_rows, double *__restrict__ dL_rows,
                           const int64_t *__restrict__ drow_off)
{
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * (blockDim.x / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
    if (r >= nrows) return;
    const RowJob j = jobs[r];
    const int64_t o = step_off[r], o1 = step_off[r + 1];
    const RowOut &out = outs[j.kind];
    double *hw = nullptr, *cum = nullptr;
    int64_t rlen = 0;
    if (j.with_row && j.type != ROW_SHI_DIFF) {
        int64_t ro = out.row_off[(int64_t)j.shell * out.n + j.ie];
        rlen = out.row_off[(int64_t)j.shell * out.n + j.ie + 1] - ro;
        hw = out.hw + ro;
        cum = out.lam + ro;
    }
    double *dEr = nullptr, *dLr = nullptr;
    if (j.type == ROW_SHI_DIFF) {
        dEr = dE_rows + drow_off[j.shell];
        dLr = dL_rows + drow_off[j.shell];
    }
    const double Z2M = (j.Zeff * j.Zeff) * j.Mass;
    // an entry of the row: the transfer energy at the step's end and the mean
    // free path of the sum up to it
    auto entry = [&](int64_t i, double e, double sum) {
        hw[i] = e;
        if (j.type == ROW_INEL) sum = (sum < 1.0e-15) ? 1.0e15 : 1.0 / (j.Mass * sum);
        else if (j.type == ROW_PHONON) sum = (sum < 1.0e-15) ? 1.0e20 : 1.0 / (Z2M * sum);
        cum[i] = sum;
    };
    const bool weighted = (j.type == ROW_SHI && !j.bk) || j.type == ROW_SHI_DIFF;
    double Ltot1 = 0.0, ddEdx = 0.0, prev = f0[r];
    Kahan32 S, D;
    for (int64_t base = o; base < o1; base += 64) {
        const int m = (int)((o1 - base < 64) ? o1 - base : 64);
        const int64_t k = base + ((lane < m) ? lane : m - 1);
        const double E = Ek[k], dE = dEk[k];
        const double temp1 = fa[k], dL = fb[k];
        const double left = __shfl_up(dL, 1);
        const double Ltot0 = lane ? left : prev;
        prev = lane_value(dL, m - 1);
        double part;
        if (j.q32) {
            // FP32 Simpson over the transfer-energy intervals with compensated
            // sums; the cumulative values leave in FP64 for the normalisation
            const float L0 = (float)Ltot0, La = (float)temp1, Lb = (float)dL;
            const float t2 = (float)(dE / 6.0) * ((L0 + 4.0f * La) + Lb);
            // stopping power: Simpson on w * dsigma/dw over the interval
            const float a = (float)(E + dE / 2.0), b = (float)(E + dE);
            const float td = (float)(dE / 6.0) * (((float)E * L0 + (a * 4.0f) * La) + b * Lb);
            Kahan32 mine;
            for (int t = 0; t < m; ++t) {
                S.add(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(t2), t)));
                D.add(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(td), t)));
                if (lane == t) mine = S;
            }
            part = mine.value();
        } else {
            double temp2, dd;
            if (j.type == ROW_PHONON) temp2 = (trk_fabs(dE) / 6.0) * ((Ltot0 + 4.0 * temp1) + dL);
            else temp2 = (dE / 6.0) * ((Ltot0 + 4.0 * temp1) + dL);
            if (weighted) {
                double a = E + dE / 2.0;
                double b = E + dE;
                dd = (dE / 6.0) * (((E * Ltot0) + ((a * 4.0) * temp1)) + (b * dL));
            } else {
                dd = E * temp2;
            }
            part = 0.0;
            for (int t = 0; t < m; ++t) {
                Ltot1 = Ltot1 + lane_value(temp2, t);
                ddEdx = ddEdx + lane_value(dd, t);
                if (lane == t) part = Ltot1;
            }
        }
        if (lane < m) {
            const int64_t i = base - o + lane;
            if (hw) entry(i, E + dE, part);
            if (dEr) {
                dEr[i] = E;
                dLr[i] = (((kPi * kA0) * j.Ele) * kMe) / (((j.MSHI * j.Zeff) * j.Zeff) * part);
            }
        }
    }
    if (j.q32) {
        Ltot1 = S.value();
        ddEdx = D.value();
    }
    if (hw)
        for (int64_t t = o1 - o + lane; t < rlen; t += 64) entry(t, 0.0, 0.0);
    if (lane) return;
    int64_t tix = (int64_t)j.shell * out.n + j.ie;
    if (j.type == ROW_INEL) {
        double Sigma, D;
        if (Ltot1 < 1.0e-15) { Sigma = 1.0e20; D = 0.0; }
        else { Sigma = 1.0 / (j.Mass * Ltot1); D = j.Mass * ddEdx; }
        out.L[tix] = Sigma;
        out.dEdx[tix] = D;
    } else if (j.type == ROW_PHONON) {
        double Sigma;
        if ((j.Mass < 1.0e-20) || (Ltot1 < 1.0e-15)) Sigma = 1.0e29;
        else Sigma = 1.0 / (Z2M * Ltot1);
        if (Sigma > 1.0e30) Sigma = 1.0e30;
        out.L[j.ie] = Sigma;
        out.dEdx[j.ie] = Z2M * ddEdx;
    } else if (j.type == ROW_SHI) {
        double pre = (1.0 / ((kPi * kA0) * j.Ele)) * j.MSHI;
        // a Brandt-Kitagawa ion carries its charge inside the integrand
        double Sigma = j.bk ? (pre / kMe) * Ltot1 : (((pre / kMe) * j.Zeff) * j.Zeff) * Ltot1;
        if (Sigma > 1.0e30) Sigma = 1.0e30;
        out.L[tix] = (Sigma > 1.0e-10) ? 1.0 / Sigma : 1.0e28;
        out.dEdx[tix] = j.bk ? (pre / kMe) * ddEdx : (((pre / kMe) * j.Zeff) * j.Zeff) * ddEdx;
    }
}

// Mott elastic MFP (Elastic_cross_section Mott branch, CS:2939-2962 with
// Atomic_elastic_sigma CS:3495-3514); kind_of_EMFP = -1 gives 1e30 (AI:1125).
__global__ void k_mott(MatDev m, const double *__restrict__ E, int n, int hole, double *__restrict__ L,
                       double *__restrict__ dEdx)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double Ee = E[i];
    dEdx[i] = 0.0;
    if (m.kind_of_EMFP != 0) { L[i] = 1.0e30; return; }
    double Mass = 1.0;
    if (hole) {
        if (m.hole_mass >= 0.0) Mass = m.hole_mass;
        else Mass = m.dosM[find_mono_1d(m.dosE, m.n_dos, Ee) - 1];
    }
    double S = 0.0;
    for (int a = 0; a < m.n_atoms; ++a) {
        double Zat = (double)m.Zat[a];
        double mec2e = ((kMe * kC) * kC) / kE;
        double Zat137 = Zat / 137.0;
        double RyEe = kRy / Ee;
        double beta2 = (2.0 * Ee) / mec2e;
        double pc = ((1.7e-5 * trk_pow(Zat, 2.0 / 3.0)) * (1.0 - beta2)) / beta2;
        double nc = pc * (1.13 + (((3.76 * (Zat137 * Zat137)) / beta2) * trk_sqrt(Ee / (Ee + mec2e))));
        double sig = (((((((kPi * kA0) * kA0) * Zat) * (Zat + 1.0)) / (nc * (nc + 1.0))) * RyEe) * RyEe) * 1.0e-16;
        S = S + sig * m.Pers[a];
    }
    S = (S / m.sumPers) * Mass;
    L[i] = 1.0e8 / (S * m.At_Dens);
}

// Tot_Phot_IMFP, CS:833-878 (CDF branch)
__global__ void k_phot(MatDev m, const double *__restrict__ E, int n, double *__restrict__ L, double *__restrict__ dEdx)
{
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * m.nsh) return;
    int s = t / n, i = t % n;
    double Ele = E[i];
    double Sigma;
    if (Ele < m.Ip[s]) {
        Sigma = 1.0e30;
    } else {
        double ImE = imewq(m, Ele, 0.0, s, 1);
        Sigma = ((kC * kH) / ((ImE * Ele) * kE)) * 1.0e10;
    }
    L[t] = Sigma;
    dEdx[t] = Ele / Sigma;
}

// How_many_electrons, MC:1990-2055: total MFP = 1/sum(1/lambda_shell)
// TotIMFP's Delta-CDF branch, CS:952-956: per (energy, shell) of an electron
// or hole inelastic table, the mean free path and stopping power of the
// delta peaks (with the electron's mass for holes too, as the reference),
// over the quadrature's values
__global__ void k_delta_tables(MatDev m, const double *__restrict__ alpha, const double *__restrict__ E, int n,
                               int nsh, double *__restrict__ L, double *__restrict__ dEdx)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n * nsh) return;
    const int s = (int)(t / n), i = (int)(t % n);
    double Emin = m.Ip[s];
    if (Emin <= 1.0e-3) Emin = 1.0e-3;
    const int o0 = m.osc_off[s], o1 = m.osc_off[s + 1];
    const double Sigma = delta_cs(m.oE0, alpha, o0, o1, E[i], Emin, m.At_Dens, 0.0);
    L[(size_t)s * n + i] = delta_mfp(Sigma, m.At_Dens);
    dEdx[(size_t)s * n + i] = delta_eloss(m.oE0, alpha, o0, o1, E[i], Emin, m.At_Dens);
}

__global__ void k_fuse(const double *__restrict__ L, int n, int nsh, int skip_small, double *__restrict__ out)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int k = 0; k < nsh; ++k) {
        double l = L[(int64_t)k * n + i];
        if (!skip_small || l > 1.0e-10) s = s + 1.0 / l;
    }
    out[i] = (s < 1.0e-10) ? 1.0e30 : 1.0 / s;
}

// ---------------------------------------------------------------- host
static double dmax(double a, double b) { return a > b ? a : b; }
static double dmin(double a, double b) { return a < b ? a : b; }

static void osc_window(const HostMat &h, int s, double &lo, double &hi)
{
    for (int i = h.osc_off[s]; i < h.osc_off[s + 1]; ++i) {
        double l = h.m.osc_E0[i] - 5.0 * h.m.osc_Gamma[i];
        double u = h.m.osc_E0[i] + 5.0 * h.m.osc_Gamma[i];
        if (i == h.osc_off[s] || l < lo) lo = l;
        if (i == h.osc_off[s] || u > hi) hi = u;
    }
}

static double hole_mass_at(const HostMat &h, double Ele)
{
    if (h.m.hole_mass >= 0.0) return h.m.hole_mass;
    int j = find_mono_1d(h.dosE.data(), h.m.n_dos, Ele);
    return h.dosM[j - 1];
}

// get_E_low, CS:1251-1274
static void get_E_low(double lo_b, double hi_b, double Emin, double Emax, double &lo, double &hi)
{
    if ((Emin > hi_b) || (Emax < lo_b)) {
        lo = Emin;
        hi = Emax;
    } else {
        lo = dmax(lo_b, Emin);
        hi = dmin(hi_b, Emax);
        if (trk_fabs(lo - hi) < 1.0e-3) {
            lo = Emin;
            hi = Emax;
        } else {
            double dE = hi_b - lo_b;
            lo = dmin(lo, hi - dE);
            lo = dmax(lo, Emin);
        }
    }
}

// TotIMFP limits, CS:903-948
static RowJob inel_job(const HostMat &h, double Ele, int s, int hole, int with_row, int kind, int ie)
{
    RowJob j{};
    double Emin = h.m.Ip[s];
    if (Emin <= 1.0e-3) Emin = 1.0e-3;
    double Emax, Mass;
    if (hole) {
        Mass = hole_mass_at(h, Ele);
        Emax = ((4.0 * Ele) * Mass) / ((Mass + 1.0) * (Mass + 1.0));
    } else {
        Emax = (Ele + Emin) / 2.0;
        Mass = 1.0;
    }
    if (h.o.plasmon_Emax && Emin == h.Egap) {
        double Ep = trk_sqrt((((((h.m.N_VB_el * h.m.At_Dens) * 1.0e6) * kH) * kH) / (kMe * kE0)) + (h.Egap * h.Egap));
        if (Ep >= Emax) Emax = Ep;
        if (Ele < Emax) Emax = Ele;
    }
    double lo = 0, hi = 0;
    osc_window(h, s, lo, hi);
    j.Ele = Ele;
    j.Estart = Emin;
    j.Emax = Emax;
    j.E_low = dmax(lo, Emin);
    j.E_high = dmin(hi, Emax);
    j.dE_min = 1.0e-3;
    j.Mass = Mass;
    j.n = 100;
    j.shell = s;
    j.type = ROW_INEL;
    j.with_row = with_row;
    j.kind = kind;
    j.ie = ie;
    return j;
}

// Tot_EMFP limits, CS:2992-3041
static RowJob phonon_job(const HostMat &h, double Ele, int hole, int kind, int ie)
{
    RowJob j{};
    double qd = trk_pow(((6.0 * kPi) * kPi) * (h.m.At_Dens * 1.0e6), 0.33333333);
    double Edebay = ((kH * h.m.Vsound) * qd) / kE;
    Edebay = Edebay * 3.0;
    double Emin = 1.0 * 0.1e-8;
    double Mass = hole ? hole_mass_at(h, Ele) : 1.0;
    double Emax = ((((4.0 * Ele) * Mass) * kMe) * h.Mtarget) / ((h.Mtarget + Mass * kMe) * (h.Mtarget + Mass * kMe));
    if (Edebay >= Emax) Emax = Edebay;
    if (Ele < Emax) Emax = Ele;
    Emax = 1.0 * Emax;
    double lo = 0, hi = 0;
    for (int i = 0; i < h.m.n_phonon; ++i) {
        double l = h.m.ph_E0[i] - 5.0 * h.m.ph_Gamma[i];
        double u = h.m.ph_E0[i] + 5.0 * h.m.ph_Gamma[i];
        if (i == 0 || l < lo) lo = l;
        if (i == 0 || u > hi) hi = u;
    }
    double El, Eh;
    get_E_low(lo, hi, Emin, Emax, El, Eh);
    j.Ele = Ele;
    j.Estart = El;
    j.Emax = Emax;
    j.E_low = El;
    j.E_high = Eh;
    j.dE_min = 1.0e-5;
    j.Mass = Mass;
    j.Zeff = zeff_target(h, Ele);
    j.n = 20;
    j.shell = 0;
    j.type = ROW_PHONON;
    j.with_row = 1;
    j.kind = kind;
    j.ie = ie;
    return j;
}

// SHI_TotIMFP limits, CS:2470-2508
static RowJob shi_job(const HostMat &h, double Ele, int s, int diff, int ie)
{
    RowJob j{};
    double MSHI = kMp * h.ion.Mass;
    double Emin = h.m.Ip[s];
    if (Emin <= 1.0e-3) Emin = 1.0e-3;
    double Emax = (((4.0 * Ele) * kMe) * MSHI) / ((MSHI + kMe) * (MSHI + kMe));
    if (h.o.plasmon_Emax && Emin == h.Egap) {
        double Ep = trk_sqrt((((((h.m.N_VB_el * h.m.At_Dens) * 1.0e6) * kH) * kH) / (kMe * kE0)) + (h.Egap * h.Egap));
        if (Ep >= Emax) Emax = Ep;
    }
    double lo = 0, hi = 0;
    osc_window(h, s, lo, hi);
    j.Ele = Ele;
    j.Estart = Emin;
    j.Emax = Emax;
    j.E_low = dmax(lo, Emin);
    j.E_high = dmin(hi, Emax);
    j.dE_min = 1.0e-3;
    j.MSHI = MSHI;
    j.Zeff = shi_zeff(h, Ele);
    j.n = 1000;
    j.shell = s;
    j.type = diff ? ROW_SHI_DIFF : ROW_SHI;
    j.with_row = diff;
    // the ion's mean free paths of a Brandt-Kitagawa ion (SHI_Total_IMFP,
    // CS:2431-2446); its transfer rows stay those of a point charge
    j.bk = (!diff && h.ion.Kind_ion == 1) ? 1 : 0;
    j.Zp = (double)h.ion.Zat;
    j.kind = diff ? TRK_TAB_SHI_DIFF : TRK_TAB_SHI;
    j.ie = ie;
    return j;
}

template <class T>
static int dalloc(T **p, size_t n, std::string &err)
{
    if (n == 0) n = 1;
    HIP_OK(hipMalloc((void **)p, n * sizeof(T)));
    return 0;
}

// Entries of the density of states that k_eval follows by their momentum: all
// of them if the material takes its masses from there, the momenta increase,
// and the masses are ordinary numbers; else 0 (a search of every momentum).
static int dos_masses(const HostMat &h, const MatDev &md)
{
    if (!md.use_k || md.nk < 1 || md.nk > kMaxDosMass) return 0;
    const bool metal = h.Egap < 0.2;       // the choice of the uploaded pair
    const std::vector<double> &k = metal ? h.doskI : h.dosk, &M = metal ? h.dosMI : h.dosM;
    if ((int)k.size() < md.nk || (int)M.size() < md.nk) return 0;
    for (int i = 0; i < md.nk; ++i) {
        if (!(k[i] >= 0.0) || !(M[i] >= 1.0e-6 && M[i] <= 1.0e6)) return 0;
        if (i && !(k[i] >= k[i - 1])) return 0;
    }
    return (k[md.nk - 1] > 0.0 && k[md.nk - 1] < 1.0e300) ? md.nk : 0;
}

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

void free_tables(TableSet &ts)
{
    if (ts.shared_material) {
        // forget the borrowed material arrays; free only the ion's own
        for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_E_EL, TRK_TAB_H_EL, TRK_TAB_PHOT}) {
            ts.tab[k] = TableDev();
            ts.ln_E[k] = ts.ln_L[k] = ts.ln_hw[k] = ts.ln_lam[k] = nullptr;
        }
        ts.el_imfp = ts.hole_imfp = ts.phot_imfp = nullptr;
        ts.ln_el_imfp = ts.ln_hole_imfp = ts.ln_Lel = ts.ln_LHel = nullptr;
        ts.dsf[0] = ts.dsf[1] = DsfDev{};
        ts.shared_material = false;
    }
    for (int p = 0; p < 2; ++p) {
        if (ts.dsf_buf[p]) (void)hipFree(ts.dsf_buf[p]);
        ts.dsf_buf[p] = nullptr;
        ts.dsf[p] = DsfDev{};
    }
    for (auto &t : ts.tab) {
        if (t.E) (void)hipFree(t.E);
        if (t.L) (void)hipFree(t.L);
        if (t.dEdx) (void)hipFree(t.dEdx);
        if (t.row_off) (void)hipFree(t.row_off);
        if (t.hw) (void)hipFree(t.hw);
        if (t.lam) (void)hipFree(t.lam);
        if (t.row_mono) (void)hipFree(t.row_mono);
        if (t.dE) (void)hipFree(t.dE);
        if (t.dL) (void)hipFree(t.dL);
        if (t.dInv) (void)hipFree(t.dInv);
        if (t.dNonMono) (void)hipFree(t.dNonMono);
        t = TableDev();
    }
    if (ts.el_imfp) (void)hipFree(ts.el_imfp);
    if (ts.hole_imfp) (void)hipFree(ts.hole_imfp);
    if (ts.phot_imfp) (void)hipFree(ts.phot_imfp);
    if (ts.shi_path) (void)hipFree(ts.shi_path);
    ts.el_imfp = ts.hole_imfp = ts.phot_imfp = ts.shi_path = nullptr;
    for (double *&p : ts.ln_E) { if (p) (void)hipFree(p); p = nullptr; }
    for (int k = 0; k < 7; ++k)
        for (double **p : {&ts.ln_L[k], &ts.ln_hw[k], &ts.ln_lam[k]}) { if (*p) (void)hipFree(*p); *p = nullptr; }
    double **lp[] = {&ts.ln_el_imfp, &ts.ln_hole_imfp, &ts.ln_Lel, &ts.ln_LHel, &ts.ln_shi_path};
    for (double **p : lp) { if (*p) (void)hipFree(*p); *p = nullptr; }
    void *sp[] = {ts.sd_n, ts.sd_off, ts.sd_M, ts.sd_c, ts.sd_bk};
    for (void *p : sp) if (p) (void)hipFree(p);
    ts.sd_n = nullptr; ts.sd_off = nullptr; ts.sd_M = nullptr; ts.sd_c = nullptr; ts.sd_bk = nullptr;
    ts.sd_consts = false;
    ts.grids_increasing = false;
}

static int upload_grid(TableDev &t, const std::vector<double> &g, int nsh, std::string &err)
{
    t.n = (int)g.size();
    t.nsh = nsh;
    if (dalloc(&t.E, g.size(), err)) return TRK_ERR_DEVICE;
    HIP_OK(hipMemcpy(t.E, g.data(), g.size() * sizeof(double), hipMemcpyHostToDevice));
    if (dalloc(&t.L, (size_t)nsh * g.size(), err)) return TRK_ERR_DEVICE;
    if (dalloc(&t.dEdx, (size_t)nsh * g.size(), err)) return TRK_ERR_DEVICE;
    t.has_rows.assign(nsh, 0);
    return 0;
}

// The material kinds of a built table set, borrowed by an ion's table set.
static void borrow_material(TableSet &ts, const TableSet &mat)
{
    for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_E_EL, TRK_TAB_H_EL, TRK_TAB_PHOT}) {
        ts.tab[k] = mat.tab[k];
        ts.ln_E[k] = mat.ln_E[k]; ts.ln_L[k] = mat.ln_L[k]; ts.ln_hw[k] = mat.ln_hw[k]; ts.ln_lam[k] = mat.ln_lam[k];
    }
    ts.el_imfp = mat.el_imfp; ts.hole_imfp = mat.hole_imfp; ts.phot_imfp = mat.phot_imfp;
    ts.ln_el_imfp = mat.ln_el_imfp; ts.ln_hole_imfp = mat.ln_hole_imfp; ts.ln_Lel = mat.ln_Lel; ts.ln_LHel = mat.ln_LHel;
    ts.dsf[0] = mat.dsf[0];
    ts.dsf[1] = mat.dsf[1];
    ts.shared_material = true;
}

int build_tables(const HostMat &h, const MatDev &md, TableSet &ts, hipStream_t st, std::string &err,
                 const TableSet *mat, const double *delta_alpha)
{
    auto t_start = std::chrono::steady_clock::now();
    free_tables(ts);
    const bool own = (mat == nullptr);     // build the material kinds too
    const int nsh = h.nsh;
    double dosmax = h.dosE.empty() ? 0.0 : h.dosE[0];
    for (double v : h.dosE) dosmax = (v > dosmax) ? v : dosmax;

    // grids (get_grid_4CS, AI:158, 210, 2270-2273)
    std::vector<double> gE, gH, gEel, gHel, gP, gS;
    grid_4cs(h.m, 0.1, h.e_emax, gE);
    grid_4cs(h.m, 0.1, dosmax + 1.0, gH);
    grid_4cs(h.m, 0.01, h.e_emax, gEel);
    grid_4cs(h.m, 0.01, dosmax + 1.0, gHel);
    if (h.o.kind_of_EMFP == 2) {
        // the elastic tables of DSF scattering live on the DSF's own energies
        // (Elastic_MFP%Total%E = DSF_DEMFP%E, Analytical_IMFPs.f90:905-911)
        if (h.dsfE[0].size() < 2 || h.dsfE[1].size() < 2) {
            err = "DSF elastic scattering (kind_of_EMFP = 2) needs the electron and hole DSF tables (trk_dsf_set)";
            return TRK_ERR_STATE;
        }
        gEel = h.dsfE[0];
        gHel = h.dsfE[1];
    }
    if (h.o.include_photons) grid_4cs(h.m, 0.1, h.e_emax, gP);
    {
        double M = h.ion.Mass * kMp;
        double Emin = std::ceil(((((M + kMe) * (M + kMe)) / (M * kMe)) * h.Egap) / 4.0);
        double Emax = (h.o.shi_grid_Emax > 0.0) ? h.o.shi_grid_Emax : (175.6e6 / 2.0) * h.ion.Mass;
        grid_4cs(h.m, Emin, Emax, gS);
    }
    TableDev *T = ts.tab;
    int rc;
    if (own) {
        if ((rc = upload_grid(T[TRK_TAB_E_INEL], gE, nsh, err))) return rc;
        if ((rc = upload_grid(T[TRK_TAB_H_INEL], gH, nsh, err))) return rc;
        if ((rc = upload_grid(T[TRK_TAB_E_EL], gEel, 1, err))) return rc;
        if ((rc = upload_grid(T[TRK_TAB_H_EL], gHel, 1, err))) return rc;
        if (!gP.empty() && (rc = upload_grid(T[TRK_TAB_PHOT], gP, nsh, err))) return rc;
    } else {
        borrow_material(ts, *mat);
    }
    if ((rc = upload_grid(T[TRK_TAB_SHI], gS, nsh, err))) return rc;
    T[TRK_TAB_SHI_DIFF].nsh = nsh;

    // row jobs
    std::vector<RowJob> jobs;
    if (own) {
        for (int i = 0; i < (int)gE.size(); ++i)
            for (int s = 0; s < nsh; ++s) jobs.push_back(inel_job(h, gE[i], s, 0, 1, TRK_TAB_E_INEL, i));
        for (int i = 0; i < (int)gH.size(); ++i)
            for (int s = 0; s < nsh; ++s) jobs.push_back(inel_job(h, gH[i], s, 1, s == h.vb, TRK_TAB_H_INEL, i));
        if (h.o.kind_of_EMFP == 1) {
            for (int i = 0; i < (int)gEel.size(); ++i) jobs.push_back(phonon_job(h, gEel[i], 0, TRK_TAB_E_EL, i));
            for (int i = 0; i < (int)gHel.size(); ++i) jobs.push_back(phonon_job(h, gHel[i], 1, TRK_TAB_H_EL, i));
        }
    }
    for (int i = 0; i < (int)gS.size(); ++i)
        for (int s = 0; s < nsh; ++s) jobs.push_back(shi_job(h, gS[i], s, 0, i));
    for (int s = 0; s < nsh; ++s) jobs.push_back(shi_job(h, h.ion.E, s, 1, 0));
    // the precision form's quadrature for the inelastic and ion rows (the
    // phonon rows keep the reference's)
    if (h.o.quadrature == 1)
        for (RowJob &j : jobs)
            if (j.type != ROW_PHONON && !j.bk) j.q32 = 1;
    if (own) {
        T[TRK_TAB_E_INEL].has_rows.assign(nsh, 1);
        T[TRK_TAB_H_INEL].has_rows[h.vb] = 1;
        if (h.o.kind_of_EMFP == 1) {
            T[TRK_TAB_E_EL].has_rows[0] = 1;
            T[TRK_TAB_H_EL].has_rows[0] = 1;
        }
    }
    const int nrows = (int)jobs.size();

    RowJob *d_jobs = nullptr;
    int *d_cnt = nullptr, *d_len = nullptr;
    if (dalloc(&d_jobs, nrows, err) || dalloc(&d_cnt, nrows, err) || dalloc(&d_len, nrows, err)) return TRK_ERR_DEVICE;
    HIP_OK(hipMemcpyAsync(d_jobs, jobs.data(), sizeof(RowJob) * nrows, hipMemcpyHostToDevice, st));
    k_row_plan<<<nblk(nrows, 4), 256, 0, st>>>(d_jobs, nrows, d_cnt, d_len);
    HIP_OK(hipGetLastError());
    std::vector<int> cnt(nrows), len(nrows);
    HIP_OK(hipMemcpyAsync(cnt.data(), d_cnt, sizeof(int) * nrows, hipMemcpyDeviceToHost, st));
    HIP_OK(hipMemcpyAsync(len.data(), d_len, sizeof(int) * nrows, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    for (int r = 0; r < nrows; ++r)
        if (cnt[r] < 0) {
            err = "transfer-energy grid of row " + std::to_string(r) + " (kind " + std::to_string(jobs[r].kind) +
                  ", shell " + std::to_string(jobs[r].shell) + ", E " + std::to_string(jobs[r].Ele) + " eV) does not close";
            return TRK_ERR_NUMERIC;
        }

    // step offsets
    std::vector<int64_t> step_off(nrows + 1, 0), chunk_off(nrows + 1, 0);
    for (int r = 0; r < nrows; ++r) {
        step_off[r + 1] = step_off[r] + cnt[r];
        chunk_off[r + 1] = chunk_off[r] + row_chunks(cnt[r]);
    }
    const int64_t nsteps = step_off[nrows], nchunks = chunk_off[nrows];

    // row storage per kind: row_off over (shell, ie)
    if (own)
        for (int kind : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_E_EL, TRK_TAB_H_EL}) {
            TableDev &t = T[kind];
            t.row_off_h.assign((size_t)t.nsh * t.n + 1, 0);
        }
    std::vector<int64_t> rowlen_by_slot[4];
    if (own)
        for (int kind = 0; kind < 4; ++kind) rowlen_by_slot[kind].assign((size_t)T[kind].nsh * T[kind].n, 0);
    std::vector<int> dn(nsh, 0);
    for (int r = 0; r < nrows; ++r) {
        const RowJob &j = jobs[r];
        if (j.type == ROW_SHI_DIFF) { dn[j.shell] = len[r]; continue; }
        if (!j.with_row) continue;
        rowlen_by_slot[j.kind][(size_t)j.shell * T[j.kind].n + j.ie] = len[r];
    }
    for (int kind = 0; kind < 4 && own; ++kind) {
        TableDev &t = T[kind];
        for (size_t i = 0; i < rowlen_by_slot[kind].size(); ++i) t.row_off_h[i + 1] = t.row_off_h[i] + rowlen_by_slot[kind][i];
        int64_t tot = t.row_off_h.back();
        if (dalloc(&t.row_off, t.row_off_h.size(), err)) return TRK_ERR_DEVICE;
        HIP_OK(hipMemcpyAsync(t.row_off, t.row_off_h.data(), sizeof(int64_t) * t.row_off_h.size(), hipMemcpyHostToDevice, st));
        if (dalloc(&t.hw, tot, err) || dalloc(&t.lam, tot, err)) return TRK_ERR_DEVICE;
    }
    TableDev &td = T[TRK_TAB_SHI_DIFF];
    td.dn = dn;
    td.doff.assign(nsh + 1, 0);
    for (int s = 0; s < nsh; ++s) td.doff[s + 1] = td.doff[s] + dn[s];
    int64_t *d_doff = nullptr;
    if (dalloc(&td.dE, td.doff[nsh], err) || dalloc(&td.dL, td.doff[nsh], err) || dalloc(&d_doff, nsh + 1, err))
        return TRK_ERR_DEVICE;
    HIP_OK(hipMemcpyAsync(d_doff, td.doff.data(), sizeof(int64_t) * (nsh + 1), hipMemcpyHostToDevice, st));

    // nodes and evaluations
    int64_t *d_step_off = nullptr, *d_chunk_off = nullptr;
    double *d_Ek = nullptr, *d_dEk = nullptr, *d_f0 = nullptr, *d_fa = nullptr, *d_fb = nullptr;
    int *d_chunk_row = nullptr;
    if (dalloc(&d_step_off, nrows + 1, err) || dalloc(&d_chunk_off, nrows + 1, err) || dalloc(&d_Ek, nsteps, err) ||
        dalloc(&d_dEk, nsteps, err) || dalloc(&d_f0, nrows, err) || dalloc(&d_fa, nsteps, err) ||
        dalloc(&d_fb, nsteps, err) || dalloc(&d_chunk_row, nchunks, err))
        return TRK_ERR_DEVICE;
    HIP_OK(hipMemcpyAsync(d_step_off, step_off.data(), sizeof(int64_t) * (nrows + 1), hipMemcpyHostToDevice, st));
    HIP_OK(hipMemcpyAsync(d_chunk_off, chunk_off.data(), sizeof(int64_t) * (nrows + 1), hipMemcpyHostToDevice, st));
    k_row_nodes<<<nblk(nrows, 4), 256, 0, st>>>(d_jobs, nrows, d_step_off, d_chunk_off, d_Ek, d_dEk, d_chunk_row);
    HIP_OK(hipGetLastError());
    int64_t npts = nrows + 2 * nsteps;
    const int dos_n = dos_masses(h, md);
    k_eval<<<nblk(nchunks, kEvalBlock / kPointsWave), kEvalBlock, sizeof(double) * 3 * dos_n, st>>>(
        md, d_jobs, d_chunk_row, d_chunk_off, d_step_off, nchunks, d_Ek, d_dEk, d_f0, d_fa, d_fb, dos_n);
    HIP_OK(hipGetLastError());
    ts.dcs_evals = npts;

    RowOut outs[7];
    for (int k = 0; k < 7; ++k) {
        outs[k].L = T[k].L;
        outs[k].dEdx = T[k].dEdx;
        outs[k].n = T[k].n;
        outs[k].hw = T[k].hw;
        outs[k].lam = T[k].lam;
        outs[k].row_off = T[k].row_off;
    }
    RowOut *d_outs = nullptr;
    if (dalloc(&d_outs, 7, err)) return TRK_ERR_DEVICE;
    HIP_OK(hipMemcpyAsync(d_outs, outs, sizeof(outs), hipMemcpyHostToDevice, st));
    k_row_scan<<<nblk(nrows, 4), 256, 0, st>>>(d_jobs, nrows, d_step_off, d_Ek, d_dEk, d_f0, d_fa, d_fb, d_outs,
                                                td.dE, td.dL, d_doff);
    HIP_OK(hipGetLastError());

    // inverse rows of the ion's transfer table and their monotonicity
    if (dalloc(&td.dInv, td.doff[nsh] > 0 ? td.doff[nsh] : 1, err) || dalloc(&td.dNonMono, nsh, err))
        return TRK_ERR_DEVICE;
    HIP_OK(hipMemsetAsync(td.dNonMono, 0, sizeof(int) * nsh, st));
    for (int s = 0; s < nsh; ++s)
        if (dn[s] > 0)
            k_inv_row<<<nblk(dn[s], 256), 256, 0, st>>>(td.dL + td.doff[s], dn[s], td.dInv + td.doff[s], td.dNonMono + s);
    HIP_OK(hipGetLastError());

    // the Delta-CDF model's mean free paths and stopping powers
    if (own && h.o.kind_of_DR == 4) {
        if (!delta_alpha) { err = "the Delta-CDF model needs the oscillators' weights"; return TRK_ERR_STATE; }
        for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL})
            k_delta_tables<<<nblk((int64_t)T[k].n * nsh, 128), 128, 0, st>>>(md, delta_alpha, T[k].E, T[k].n, nsh,
                                                                             T[k].L, T[k].dEdx);
        HIP_OK(hipGetLastError());
    }
    // BEB shells (TotIMFP's BEB branch, CS:1035-1041): the closed forms of
    // the mean free path and stopping power, on the host (a few values per
    // shell), over the quadrature's values; the rows are not used
    std::vector<std::vector<double>> beb_vals;
    if (own) {
        for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL}) {
            const std::vector<double> &g = (k == TRK_TAB_E_INEL) ? gE : gH;
            for (int s = 0; s < nsh; ++s) {
                if (h.m.kocs[s] != 2) continue;
                const double B = h.m.Ip[s], U = h.m.Ek[s], N = h.m.Nel[s];
                const double temp1 = ((h.m.At_Dens * 1.0e-24) * h.m.Pers[h.atom_of[s]]) / h.sumPers;
                std::vector<double> L(g.size()), D(g.size());
                for (size_t i = 0; i < g.size(); ++i) {
                    const double Ele = g[i];
                    const double Mass = (k == TRK_TAB_H_INEL) ? hole_mass_at(h, Ele) : 1.0;
                    L[i] = 1.0 / ((Mass * temp1) * beb_sigma(Ele, B, U, N));
                    D[i] = (Mass * temp1) * beb_dsigma_w_int(Ele, (Ele - 1.0) / 2.0, B, U, N);
                }
                beb_vals.push_back(std::move(L));
                HIP_OK(hipMemcpyAsync(T[k].L + (size_t)s * T[k].n, beb_vals.back().data(), sizeof(double) * g.size(),
                                      hipMemcpyHostToDevice, st));
                beb_vals.push_back(std::move(D));
                HIP_OK(hipMemcpyAsync(T[k].dEdx + (size_t)s * T[k].n, beb_vals.back().data(), sizeof(double) * g.size(),
                                      hipMemcpyHostToDevice, st));
            }
        }
        if (!beb_vals.empty()) HIP_OK(hipStreamSynchronize(st));   // the host values are then free to go
    }
    // DSF elastic tables: the total mean free path is each row's last entry
    // (its emission and absorption parts likewise), no stopping power; the
    // rows go to the device for the transfer sampling
    if (own && h.o.kind_of_EMFP == 2) {
        for (int p = 0; p < 2; ++p) {
            const int k = p ? TRK_TAB_H_EL : TRK_TAB_E_EL;
            const int nE = (int)h.dsfE[p].size(), nW = h.dsf_nW[p];
            const size_t cells = (size_t)nE * nW;
            std::vector<double> host(3 * cells + 3 * (size_t)nE);
            double *Lt = host.data() + 3 * cells, *Le = Lt + nE, *La = Le + nE;
            for (int i = 0; i < nE; ++i) {
                const size_t last = (size_t)i * nW + (nW - 1);
                Lt[i] = h.dsfL[p][last];
                Le[i] = h.dsfLe[p][last];
                La[i] = h.dsfLa[p][last];
            }
            std::copy(h.dsfdE[p].begin(), h.dsfdE[p].end(), host.begin());
            std::copy(h.dsfLe[p].begin(), h.dsfLe[p].end(), host.begin() + cells);
            std::copy(h.dsfLa[p].begin(), h.dsfLa[p].end(), host.begin() + 2 * cells);
            if (dalloc(&ts.dsf_buf[p], host.size(), err)) return TRK_ERR_DEVICE;
            HIP_OK(hipMemcpy(ts.dsf_buf[p], host.data(), sizeof(double) * host.size(), hipMemcpyHostToDevice));
            HIP_OK(hipMemcpy(T[k].L, Lt, sizeof(double) * nE, hipMemcpyHostToDevice));
            HIP_OK(hipMemset(T[k].dEdx, 0, sizeof(double) * nE));
            DsfDev &dv = ts.dsf[p];
            dv.nE = nE; dv.nW = nW;
            dv.E = T[k].E; dv.Lt = T[k].L;
            dv.dE = ts.dsf_buf[p]; dv.dLe = ts.dsf_buf[p] + cells; dv.dLa = ts.dsf_buf[p] + 2 * cells;
            dv.Le = ts.dsf_buf[p] + 3 * cells + nE; dv.La = dv.Le + nE;
        }
    }
    // Mott / disabled elastic tables
    if (own && h.o.kind_of_EMFP != 1 && h.o.kind_of_EMFP != 2) {
        k_mott<<<nblk(T[TRK_TAB_E_EL].n, 128), 128, 0, st>>>(md, T[TRK_TAB_E_EL].E, T[TRK_TAB_E_EL].n, 0,
                                                              T[TRK_TAB_E_EL].L, T[TRK_TAB_E_EL].dEdx);
        k_mott<<<nblk(T[TRK_TAB_H_EL].n, 128), 128, 0, st>>>(md, T[TRK_TAB_H_EL].E, T[TRK_TAB_H_EL].n, 1,
                                                              T[TRK_TAB_H_EL].L, T[TRK_TAB_H_EL].dEdx);
        HIP_OK(hipGetLastError());
    }
    if (own && !gP.empty()) {
        k_phot<<<nblk((int64_t)T[TRK_TAB_PHOT].n * nsh, 128), 128, 0, st>>>(md, T[TRK_TAB_PHOT].E, T[TRK_TAB_PHOT].n,
                                                                             T[TRK_TAB_PHOT].L, T[TRK_TAB_PHOT].dEdx);
        HIP_OK(hipGetLastError());
    }
    // fused totals
    if (dalloc(&ts.shi_path, T[TRK_TAB_SHI].n, err)) return TRK_ERR_DEVICE;
    k_fuse<<<nblk(T[TRK_TAB_SHI].n, 128), 128, 0, st>>>(T[TRK_TAB_SHI].L, T[TRK_TAB_SHI].n, nsh, 0, ts.shi_path);
    if (own) {
        if (dalloc(&ts.el_imfp, T[TRK_TAB_E_INEL].n, err) || dalloc(&ts.hole_imfp, T[TRK_TAB_H_INEL].n, err))
            return TRK_ERR_DEVICE;
        k_fuse<<<nblk(T[TRK_TAB_E_INEL].n, 128), 128, 0, st>>>(T[TRK_TAB_E_INEL].L, T[TRK_TAB_E_INEL].n, nsh, 1, ts.el_imfp);
        k_fuse<<<nblk(T[TRK_TAB_H_INEL].n, 128), 128, 0, st>>>(T[TRK_TAB_H_INEL].L, T[TRK_TAB_H_INEL].n, nsh, 0, ts.hole_imfp);
    }
    if (own && !gP.empty()) {
        if (dalloc(&ts.phot_imfp, T[TRK_TAB_PHOT].n, err)) return TRK_ERR_DEVICE;
        k_fuse<<<nblk(T[TRK_TAB_PHOT].n, 128), 128, 0, st>>>(T[TRK_TAB_PHOT].L, T[TRK_TAB_PHOT].n, nsh, 0, ts.phot_imfp);
    }
    HIP_OK(hipGetLastError());
    // logs of the grids and of the tables the transport interpolates most
    for (int k = 0; k < 6; ++k) {
        if (!own && k != TRK_TAB_SHI) continue;
        if (T[k].n <= 0 || !T[k].E) continue;
        if (dalloc(&ts.ln_E[k], T[k].n, err)) return TRK_ERR_DEVICE;
        k_log<<<nblk(T[k].n, 128), 128, 0, st>>>(T[k].E, T[k].n, ts.ln_E[k]);
    }
    struct { const double *src; int n; double **dst; bool mat; } lg[] = {
        {ts.el_imfp, T[TRK_TAB_E_INEL].n, &ts.ln_el_imfp, true}, {ts.hole_imfp, T[TRK_TAB_H_INEL].n, &ts.ln_hole_imfp, true},
        {T[TRK_TAB_E_EL].L, T[TRK_TAB_E_EL].n, &ts.ln_Lel, true}, {T[TRK_TAB_H_EL].L, T[TRK_TAB_H_EL].n, &ts.ln_LHel, true},
        {ts.shi_path, T[TRK_TAB_SHI].n, &ts.ln_shi_path, false}};
    for (auto &g : lg) {
        if (!g.src || g.n <= 0 || (g.mat && !own)) continue;
        if (dalloc(g.dst, g.n, err)) return TRK_ERR_DEVICE;
        k_log<<<nblk(g.n, 128), 128, 0, st>>>(g.src, g.n, *g.dst);
    }
    // per-shell mean free paths (shell choice) and cumulative rows (transfer
    // sampling): interpolation then takes one log of the argument
    for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_SHI}) {
        const int64_t m = (int64_t)T[k].nsh * T[k].n;
        if (!T[k].L || m <= 0 || (!own && k != TRK_TAB_SHI)) continue;
        if (dalloc(&ts.ln_L[k], m, err)) return TRK_ERR_DEVICE;
        k_log<<<(unsigned)((m + 127) / 128), 128, 0, st>>>(T[k].L, m, ts.ln_L[k]);
    }
    for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_E_EL, TRK_TAB_H_EL}) {
        const int64_t m = T[k].row_off_h.empty() ? 0 : T[k].row_off_h.back();
        if (!own || !T[k].hw || m <= 0) continue;
        if (dalloc(&ts.ln_hw[k], m, err) || dalloc(&ts.ln_lam[k], m, err)) return TRK_ERR_DEVICE;
        k_log<<<(unsigned)((m + 127) / 128), 128, 0, st>>>(T[k].hw, m, ts.ln_hw[k]);
        k_log<<<(unsigned)((m + 127) / 128), 128, 0, st>>>(T[k].lam, m, ts.ln_lam[k]);
        const int64_t nslots = (int64_t)T[k].nsh * T[k].n;
        if (dalloc(&T[k].row_mono, nslots, err)) return TRK_ERR_DEVICE;
        k_row_mono<<<nblk(nslots, 4), 256, 0, st>>>(T[k].row_off, nslots, T[k].lam, T[k].row_mono);
    }
    HIP_OK(hipGetLastError());
    HIP_OK(hipStreamSynchronize(st));
    // run constants: a particle's last bracket may stand in for a search only
    // on strictly increasing grids; the ion's first free path sizes batches
    {
        bool inc = own || mat->grids_increasing;
        for (const std::vector<double> *g : {&gE, &gEel, &gH, &gHel, &gS})
            for (size_t i = 1; i < g->size(); ++i)
                if (!((*g)[i - 1] < (*g)[i])) inc = false;
        ts.grids_increasing = inc;
        std::vector<double> sp(gS.size());
        HIP_OK(hipMemcpy(sp.data(), ts.shi_path, sizeof(double) * sp.size(), hipMemcpyDeviceToHost));
        ts.shi_path0 = nfp_2d_host(gS.data(), sp.data(), (int)gS.size(), h.ion.E);
        const TableDev &td = T[TRK_TAB_SHI_DIFF];
        if (dalloc(&ts.sd_n, (size_t)nsh, err) || dalloc(&ts.sd_off, (size_t)nsh + 1, err) ||
            dalloc(&ts.sd_M, (size_t)2 * nsh, err) || dalloc(&ts.sd_c, (size_t)2 * nsh, err) ||
            dalloc(&ts.sd_bk, (size_t)nsh * (kShiBuckets + 1), err))
            return TRK_ERR_DEVICE;
        HIP_OK(hipMemcpy(ts.sd_n, td.dn.data(), sizeof(int) * nsh, hipMemcpyHostToDevice));
        HIP_OK(hipMemcpy(ts.sd_off, td.doff.data(), sizeof(int64_t) * (nsh + 1), hipMemcpyHostToDevice));
        ts.sd_consts = false;
    }
    (void)hipFree(d_jobs); (void)hipFree(d_cnt); (void)hipFree(d_len); (void)hipFree(d_doff);
    (void)hipFree(d_step_off); (void)hipFree(d_Ek); (void)hipFree(d_dEk); (void)hipFree(d_f0);
    (void)hipFree(d_fa); (void)hipFree(d_fb); (void)hipFree(d_chunk_off); (void)hipFree(d_chunk_row); (void)hipFree(d_outs);
    ts.launches = 12;
    ts.build_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t_start).count();
    return 0;
}

// After tables were replaced from host arrays (trk_table_set / trk_row_set):
// the fused paths, the logs, the row flags, the ion's inverse transfer rows
// and the run constants derived from them, recomputed in place.
int refresh_derived(const HostMat &h, TableSet &ts, hipStream_t st, std::string &err)
{
    const int nsh = h.nsh;
    TableDev *T = ts.tab;
    const bool own = !ts.shared_material;
    if (own) {
        k_fuse<<<nblk(T[TRK_TAB_E_INEL].n, 128), 128, 0, st>>>(T[TRK_TAB_E_INEL].L, T[TRK_TAB_E_INEL].n, nsh, 1, ts.el_imfp);
        k_fuse<<<nblk(T[TRK_TAB_H_INEL].n, 128), 128, 0, st>>>(T[TRK_TAB_H_INEL].L, T[TRK_TAB_H_INEL].n, nsh, 0, ts.hole_imfp);
        if (ts.phot_imfp)
            k_fuse<<<nblk(T[TRK_TAB_PHOT].n, 128), 128, 0, st>>>(T[TRK_TAB_PHOT].L, T[TRK_TAB_PHOT].n, nsh, 0, ts.phot_imfp);
    }
    k_fuse<<<nblk(T[TRK_TAB_SHI].n, 128), 128, 0, st>>>(T[TRK_TAB_SHI].L, T[TRK_TAB_SHI].n, nsh, 0, ts.shi_path);
    for (int k = 0; k < 6; ++k) {
        if (!own && k != TRK_TAB_SHI) continue;
        if (T[k].n > 0 && T[k].E && ts.ln_E[k]) k_log<<<nblk(T[k].n, 128), 128, 0, st>>>(T[k].E, T[k].n, ts.ln_E[k]);
    }
    struct { const double *src; int n; double *dst; bool mat; } lg[] = {
        {ts.el_imfp, T[TRK_TAB_E_INEL].n, ts.ln_el_imfp, true}, {ts.hole_imfp, T[TRK_TAB_H_INEL].n, ts.ln_hole_imfp, true},
        {T[TRK_TAB_E_EL].L, T[TRK_TAB_E_EL].n, ts.ln_Lel, true}, {T[TRK_TAB_H_EL].L, T[TRK_TAB_H_EL].n, ts.ln_LHel, true},
        {ts.shi_path, T[TRK_TAB_SHI].n, ts.ln_shi_path, false}};
    for (auto &g : lg)
        if (g.src && g.dst && g.n > 0 && (own || !g.mat)) k_log<<<nblk(g.n, 128), 128, 0, st>>>(g.src, g.n, g.dst);
    for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_SHI}) {
        const int64_t m = (int64_t)T[k].nsh * T[k].n;
        if (!T[k].L || !ts.ln_L[k] || m <= 0 || (!own && k != TRK_TAB_SHI)) continue;
        k_log<<<(unsigned)((m + 127) / 128), 128, 0, st>>>(T[k].L, m, ts.ln_L[k]);
    }
    for (int k : {TRK_TAB_E_INEL, TRK_TAB_H_INEL, TRK_TAB_E_EL, TRK_TAB_H_EL}) {
        const int64_t m = T[k].row_off_h.empty() ? 0 : T[k].row_off_h.back();
        if (!own || !T[k].hw || !ts.ln_hw[k] || m <= 0) continue;
        k_log<<<(unsigned)((m + 127) / 128), 128, 0, st>>>(T[k].hw, m, ts.ln_hw[k]);
        k_log<<<(unsigned)((m + 127) / 128), 128, 0, st>>>(T[k].lam, m, ts.ln_lam[k]);
        const int64_t nslots = (int64_t)T[k].nsh * T[k].n;
        k_row_mono<<<nblk(nslots, 4), 256, 0, st>>>(T[k].row_off, nslots, T[k].lam, T[k].row_mono);
    }
    TableDev &td = T[TRK_TAB_SHI_DIFF];
    HIP_OK(hipMemsetAsync(td.dNonMono, 0, sizeof(int) * nsh, st));
    for (int sh = 0; sh < nsh; ++sh)
        if (td.dn[sh] > 0)
            k_inv_row<<<nblk(td.dn[sh], 256), 256, 0, st>>>(td.dL + td.doff[sh], td.dn[sh], td.dInv + td.doff[sh],
                                                            td.dNonMono + sh);
    HIP_OK(hipGetLastError());
    std::vector<double> sE(T[TRK_TAB_SHI].n), sp(T[TRK_TAB_SHI].n);
    HIP_OK(hipMemcpyAsync(sE.data(), T[TRK_TAB_SHI].E, sizeof(double) * sE.size(), hipMemcpyDeviceToHost, st));
    HIP_OK(hipMemcpyAsync(sp.data(), ts.shi_path, sizeof(double) * sp.size(), hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    ts.shi_path0 = nfp_2d_host(sE.data(), sp.data(), (int)sE.size(), h.ion.E);
    ts.sd_consts = false;
    return 0;
}

}  // namespace trk
