// chem_device.hpp -- device-side thermally perfect gas and finite-rate chemistry (gfx950).
//
// One lane advances one cell.  The gas and mechanism tables (ChemDev) live in a read-only
// device buffer; every lane of a wave reads the same entries, so those loads are uniform
// (scalar).  Per-cell state is held in registers: arrays are sized by the template
// parameters NSP (species, exact) and NRM (an upper bound on the reactions, the actual
// count cd->nr is uniform at run time).  FP64 throughout, built without FMA contraction (an
// fma is one that is written).  The formulas are those of the reference functions cited beside
// them.  The curves of a species and the controller's decisions keep the reference's operation
// order; the summed curves (TpgMix), the rate constants (arrhenius), the alpha-QSS step and every
// quick_div are rearranged, as their comments say, and agree with it to rounding.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

#include "quick_math.hpp"

namespace gdtk {

constexpr int CH_MAX_SP = 8;
constexpr int CH_MAX_R = 32;

// src/gas/thermo/cea_thermo_curves.d:24-176; T_low..s_high are the constructor's
// end-point values (:45-54).
struct CEADev {
    int nseg;
    double T_breaks[4], T_blends[2], coeffs[3][9];
    double R, T_low, T_high, Cp_low, Cp_high, h_low, h_high, s_low, s_high;
};

// src/kinetics/reaction.d:58-457.  The reactant, product and efficiency lists keep the
// reference's order (reaction.d:213, 338, 483-491); nu[s] is the net stoichiometric
// coefficient of species s and part[s] marks the participants (reaction.d:100-143).
// Device code never indexes a register array with a run-time species index (that would
// put the per-cell arrays in scratch memory): it walks the species in compile-time order,
// or picks an entry through a select chain for lists that are not in ascending order.
struct ReacDev {
    int collider;
    int nreac, reac_sp[3], reac_nu[3];
    int nprod, prod_sp[3], prod_nu[3];
    int neff, eff_sp[CH_MAX_SP];
    double eff[CH_MAX_SP];
    // Dense form, used when every list is in ascending species order (then a walk over the
    // species in index order visits the entries in list order): coefficient per species
    // (0 = absent) and efficiency per species with a presence mask.
    int sorted;
    int reac_d[CH_MAX_SP], prod_d[CH_MAX_SP];
    unsigned eff_set;
    double eff_d[CH_MAX_SP];
    int f_from_eq, b_from_eq;
    double fA, fn, fC, bA, bn, bC;
    int f_park, b_park;  // Park2TRateConstant: the rate at T^s Tv^(1-s) (two-temperature reactor)
    double f_s, b_s;
    int nu[CH_MAX_SP];
    int part[CH_MAX_SP];
};

// One reaction of the branch-free rate evaluation, for a mechanism whose lists are all in
// ascending species order: per species the third-body efficiency (0 where the species is
// not in the list, or the reaction has no third body) and a code word holding the reactant
// exponent (bits 0-1, 0 = absent), the product exponent (bits 2-3), the net coefficient
// as a 4-bit two's complement number (bits 4-7) and the third-body list membership (bit
// 8).  flags bit 0: third-body reaction.  Rows
// past the reaction count are all zero: every species' net coefficient is 0 there, so they
// add nothing.
struct RateRow {
    double eff[CH_MAX_SP];
    int code[CH_MAX_SP];
    int flags;
    int pad_[3];
};

// How the rate code walks a mechanism (chosen on the host, mechanism_walk): its species lists,
// the rows above, or code in which the structure of the mechanism is known at compile time.
enum ChemWalk : int { WALK_LIST = 0, WALK_ROWS = 1, WALK_AIR5_PARK = 2, WALK_AIR5_GUPTA = 3, WALK_N2_PAIR = 4 };

// A species' code word in a row: its exponent as reactant and product, and whether it is in the
// third-body list.
constexpr int row_code(int reac, int prod, int third) {
    return reac | (prod << 2) | (((prod - reac) & 15) << 4) | (third << 8);
}

// Mechanism structures with rate code of their own: which species react in what order and
// which act as third bodies, no rates and no efficiencies.  They are the structures of the
// mechanisms that the package ships: dissociation of 5-species air (N2, O2, NO, N, O) with the
// two Zeldovich exchanges, the same with N2 + N <=> 3 N apart, and dissociating nitrogen (N2, N).
// A row walk spends most of its instructions on the selects that the code words steer (of 750
// a rate evaluation of air, 60 are arithmetic) and waits for each row's scalar loads; with the
// structure known both go: 1048576 cells of air over 1e-7 s (63e6 step attempts) integrate in
// 2.6 ms instead of 8.4, 3001 cells with at most 49 attempts each in 0.16 ms instead of 0.77 (with the
// step algebra of alpha_qss_step).
template <int WALK>
struct MechShape {  // the walks without a structure
    static constexpr int nsp = 0, nr = 0;
    static __host__ __device__ constexpr int code(int, int) { return 0; }
    static __host__ __device__ constexpr int flags(int) { return 0; }
};
template <>
struct MechShape<WALK_AIR5_PARK> {
    static constexpr int nsp = 5, nr = 5;
    static __host__ __device__ constexpr int code(int ir, int s) {
        constexpr int none = row_code(0, 0, 0), m = row_code(0, 0, 1), a = row_code(1, 0, 0), b = row_code(0, 1, 0);
        constexpr int am = row_code(1, 0, 1), bm = row_code(0, 1, 1), b2m = row_code(0, 2, 1);
        constexpr int t[5][5] = {{am, m, m, b2m, m},       // N2 + M <=> 2 N + M
                                 {m, am, m, m, b2m},       // O2 + M <=> 2 O + M
                                 {m, m, am, bm, bm},       // NO + M <=> N + O + M
                                 {none, b, a, b, a},       // NO + O <=> O2 + N
                                 {a, none, b, b, a}};      // N2 + O <=> NO + N
        return t[ir][s];
    }
    static __host__ __device__ constexpr int flags(int ir) { return ir < 3 ? 1 : 0; }
};
template <>
struct MechShape<WALK_AIR5_GUPTA> {
    static constexpr int nsp = 5, nr = 6;
    static __host__ __device__ constexpr int code(int ir, int s) {
        constexpr int none = row_code(0, 0, 0), m = row_code(0, 0, 1), a = row_code(1, 0, 0), b = row_code(0, 1, 0);
        constexpr int am = row_code(1, 0, 1), bm = row_code(0, 1, 1), b2 = row_code(0, 2, 0), b2m = row_code(0, 2, 1);
        constexpr int t[6][5] = {{m, am, m, m, b2m},                       // O2 + M <=> 2 O + M
                                 {am, m, m, b2, m},                        // N2 + M <=> 2 N + M, M not N
                                 {a, none, none, row_code(1, 3, 0), none}, // N2 + N <=> 3 N
                                 {m, m, am, bm, bm},                       // NO + M <=> N + O + M
                                 {none, b, a, b, a},                       // NO + O <=> O2 + N
                                 {a, none, b, b, a}};                      // N2 + O <=> NO + N
        return t[ir][s];
    }
    static __host__ __device__ constexpr int flags(int ir) { return (ir < 2 || ir == 3) ? 1 : 0; }
};
template <>
struct MechShape<WALK_N2_PAIR> {
    static constexpr int nsp = 2, nr = 2;
    static __host__ __device__ constexpr int code(int ir, int s) {
        constexpr int t[2][2] = {{row_code(2, 1, 0), row_code(0, 2, 0)},   // 2 N2 <=> N2 + 2 N
                                 {row_code(1, 0, 0), row_code(1, 3, 0)}};  // N2 + N <=> 3 N
        return t[ir][s];
    }
    static __host__ __device__ constexpr int flags(int) { return 0; }
};

// The species' curves as the mixture sums them (TpgMix).  The temperature line is cut where any
// species changes its range (its end points and the edges of its blends, cea_thermo_curves.d:
// 137-176); region r lies between lo[r] and hi[r] and has an expansion point T0, its lower edge.  There every
// species' coefficients {a0, a1, q0..q4, H0} are c[0] + z c[1], z = T - T0 (linear in T in a
// blend of two segments; flat[r] = 1 where no species blends and c[1] is 0), with
//   h / R  = H0 + a1 log(T / T0) + z (a0 / (T T0) + q0 + z (q1/2 + z (q2/3 + z (q3/4 + z q4/5)))),
//   Cp / R = (a0 / T + a1) / T + q0 + z (q1 + z (q2 + z (q3 + z q4))):
// the NASA-9 forms of cea_thermo_curves.d:56-102 expanded about T0 (in extended precision on
// the host), where every term but H0 vanishes, so that sums do not cancel as the terms of the
// plain form do (by a factor 60 above 6000 K: u to 8e-16 of Cv T there, rms, against 1e-14 in
// the plain form).
constexpr int MIX_REGIONS = 6 * CH_MAX_SP + 1;  // up to 6 cuts a species
struct MixTable {
    int nreg;
    int flat[MIX_REGIONS];
    double lo[MIX_REGIONS], hi[MIX_REGIONS], T0[MIX_REGIONS], iT0[MIX_REGIONS];
    double c[MIX_REGIONS][2][CH_MAX_SP][8];
};

struct ChemDev {
    int nsp, nr;
    double M[CH_MAX_SP], R[CH_MAX_SP];
    CEADev cea[CH_MAX_SP];
    ReacDev r[CH_MAX_R];
    int all_sorted;  // every reaction in dense form: rr[] holds the mechanism
    int walk;        // ChemWalk of the mechanism
    MixTable mix;
    RateRow rr[CH_MAX_R];
    double T_lower, T_upper;
    int method;  // 0 alpha-QSS, 1 RKF
    double eps1, eps2, delta;
    int maxIters;
    double errTol;
    int maxSubcycles, maxAttempts;
    double T_frozen;
    int tight;  // tightTempCoupling: T(u) and the rate constants after every subcycle
};

// The walk of a filled table: a structure of its own code where the rows match it word for
// word, the rows where every list is in ascending species order, otherwise the lists.
template <int WALK>
inline bool shape_matches(const ChemDev& cd) {
    using S = MechShape<WALK>;
    if (cd.nsp != S::nsp || cd.nr != S::nr) return false;
    for (int ir = 0; ir < S::nr; ++ir) {
        if (cd.rr[ir].flags != S::flags(ir)) return false;
        for (int s = 0; s < S::nsp; ++s)
            if (cd.rr[ir].code[s] != S::code(ir, s)) return false;
    }
    return true;
}
inline int mechanism_walk(const ChemDev& cd) {
    if (!cd.all_sorted) return WALK_LIST;
    if (shape_matches<WALK_AIR5_PARK>(cd)) return WALK_AIR5_PARK;
    if (shape_matches<WALK_AIR5_GUPTA>(cd)) return WALK_AIR5_GUPTA;
    if (shape_matches<WALK_N2_PAIR>(cd)) return WALK_N2_PAIR;
    return WALK_ROWS;
}

constexpr double CH_R_UNIVERSAL = 8.31451;               // gas/physical_constants.d
constexpr double CH_P_ATM = 101.325e3;
constexpr double CH_T_MIN = 10.0, CH_T_MAX = 100000.0;   // gas/gas_model.d:45-46
constexpr double CH_MIN_MOLES = 1.0e-30;                 // gas/gas_model.d:44
constexpr double CH_MIN_MASSF = 1.0e-30;                 // gas/gas_model.d:43

// Element k of a register array for a wave-uniform index k: a select chain over
// compile-time indices, so the array stays in registers.
template <int N>
__device__ __forceinline__ double pick(const double* a, int k) {
    double r = a[0];
#pragma unroll
    for (int s = 1; s < N; ++s) r = (k == s) ? a[s] : r;
    return r;
}

// cea_thermo_curves.d:137-176.  The reference throws where no segment matches (only a NaN
// temperature gets there with contiguous breaks); NaN coefficients stand in for that here.
__host__ __device__ inline void cea_coeffs(const CEADev& c, double T, double a[9]) {
    const int nb = c.nseg + 1;
    if (T < (c.T_breaks[1] - 0.5 * c.T_blends[0])) {
        for (int j = 0; j < 9; ++j) a[j] = c.coeffs[0][j];
        return;
    }
    if (T > (c.T_breaks[nb - 2] + 0.5 * c.T_blends[c.nseg - 2])) {
        for (int j = 0; j < 9; ++j) a[j] = c.coeffs[c.nseg - 1][j];
        return;
    }
    for (int i = 1; i < nb - 1; ++i) {
        double T_blend_low = c.T_breaks[i] - 0.5 * c.T_blends[i - 1];
        double T_blend_high = c.T_breaks[i] + 0.5 * c.T_blends[i - 1];
        if (T >= T_blend_low && T <= T_blend_high) {
            double wB = (1. / c.T_blends[i - 1]) * (T - T_blend_low);
            double wA = 1.0 - wB;
            for (int j = 0; j < 9; ++j) a[j] = wA * c.coeffs[i - 1][j] + wB * c.coeffs[i][j];
            return;
        }
        if (i < c.nseg - 1 && T > T_blend_high && T < (c.T_breaks[i + 1] - 0.5 * c.T_blends[i])) {
            for (int j = 0; j < 9; ++j) a[j] = c.coeffs[i][j];
            return;
        }
    }
    for (int j = 0; j < 9; ++j) a[j] = __builtin_nan("");
}

// cea_thermo_curves.d:56-70
__host__ __device__ inline double cea_Cp(const CEADev& c, double T) {
    if (T < c.T_low) return c.Cp_low;
    if (T > c.T_high) return c.Cp_high;
    double a[9];
    cea_coeffs(c, T, a);
    double Cp_on_R = a[0] / (T * T) + a[1] / T + a[2] + a[3] * T;
    Cp_on_R += a[4] * T * T + a[5] * T * T * T + a[6] * T * T * T * T;
    return c.R * Cp_on_R;
}

// cea_thermo_curves.d:71-102
__host__ __device__ inline double cea_h(const CEADev& c, double T) {
    if (T < c.T_low) return c.h_low - c.Cp_low * (c.T_low - T);
    if (T > c.T_high) return c.h_high + c.Cp_high * (T - c.T_high);
    double a[9];
    cea_coeffs(c, T, a);
    double h_on_RT = -a[0] / T + a[1] * log(T) + a[2] * T + a[3] * T * T / 2.0;
    h_on_RT += a[4] * T * T * T / 3.0 + a[5] * T * T * T * T / 4.0 + a[6] * T * T * T * T * T / 5.0 + a[7];
    return c.R * h_on_RT;
}

// The powers of T that every species' curve divides by, with their reciprocals, once per
// temperature.
struct CeaT {
    double T, TT, rT, rTT, logT;
    __host__ __device__ explicit CeaT(double t, double lg) : T(t), TT(t * t), rT(1.0 / t), rTT(1.0 / (t * t)), logT(lg) {}
};

// cea_h and cea_s (cea_thermo_curves.d:71-130) at one temperature from one coefficient
// selection, log(T) and the reciprocals of CeaT: the same values bit for bit.  The
// divisor 2 T T of the entropy is exactly 2 TT, whose reciprocal is exactly rTT / 2.
__host__ __device__ inline void cea_h_s(const CEADev& c, const CeaT& p, double& h, double& sv) {
    const double T = p.T;
    if (T < c.T_low) {
        h = c.h_low - c.Cp_low * (c.T_low - T);
        sv = c.s_low - c.Cp_low * log(c.T_low / T);
        return;
    }
    if (T > c.T_high) {
        h = c.h_high + c.Cp_high * (T - c.T_high);
        sv = c.s_high + c.Cp_high * log(T / c.T_high);
        return;
    }
    double a[9];
    cea_coeffs(c, T, a);
    double h_on_RT = div_by(-a[0], T, p.rT) + a[1] * p.logT + a[2] * T + a[3] * T * T / 2.0;
    h_on_RT += div_by(a[4] * T * T * T, 3.0, 1.0 / 3.0) + a[5] * T * T * T * T / 4.0 +
               div_by(a[6] * T * T * T * T * T, 5.0, 1.0 / 5.0) + a[7];
    h = c.R * h_on_RT;
    double s_on_R = div_by(-a[0], 2.0 * p.TT, 0.5 * p.rTT) - div_by(a[1], T, p.rT) + a[2] * p.logT + a[3] * T;
    s_on_R += a[4] * T * T / 2.0 + div_by(a[5] * T * T * T, 3.0, 1.0 / 3.0) + a[6] * T * T * T * T / 4.0 + a[8];
    sv = c.R * s_on_R;
}

// cea_thermo_curves.d:103-130
__host__ __device__ inline double cea_s(const CEADev& c, double T) {
    if (T < c.T_low) return c.s_low - c.Cp_low * log(c.T_low / T);
    if (T > c.T_high) return c.s_high + c.Cp_high * log(T / c.T_high);
    double a[9];
    cea_coeffs(c, T, a);
    double logT = log(T);
    double s_on_R = -a[0] / (2.0 * T * T) - a[1] / T + a[2] * logT + a[3] * T;
    s_on_R += a[4] * T * T / 2.0 + a[5] * T * T * T / 3.0 + a[6] * T * T * T * T / 4.0 + a[8];
    return c.R * s_on_R;
}

// perf_gas_mix_eos.d:43-76
template <int NSP>
__device__ __forceinline__ double tpg_Rmix(const ChemDev& cd, const double* massf) {
    double R = 0.0;
#pragma unroll
    for (int i = 0; i < NSP; ++i) R += massf[i] * cd.R[i];
    return R;
}

// The curves of one composition near one temperature as a single curve: the sums over the
// species of weight times coefficient (therm_perf_gas_mix_eos.d:61-67 and gas_model.d:410-419
// take the sum over the species' curves at each temperature; the curves are linear in their
// coefficients).  An evaluation then costs one logarithm, one reciprocal and 17 fused
// operations whatever the number of species, where the per-species form takes some 45
// instructions and a range search for each; a Newton solve evaluates three times on one build.
// Valid on [lo, hi]; in a blend of two segments the coefficients depend on T and the interval
// is empty.
struct TpgMix {
    double a0, a1, q0, q1, q2, q3, q4, H0, T0, iT0, lo, hi;
    __device__ __forceinline__ void clear() {  // no curve yet
        lo = __builtin_huge_val();
        hi = -__builtin_huge_val();
    }
    __device__ __forceinline__ bool covers(double T) const { return T >= lo && T <= hi; }
};

// The weighted curves at T: sum of y_s (h_s / R_s) - lin T + cst, y_s usually massf_s R_s.  A
// temperature that is not a number leaves a curve whose value is none either.
template <int NSP>
__device__ __forceinline__ void tpg_mix_build(const ChemDev& cd, const double* y, double lin, double cst, double T,
                                              TpgMix& m) {
    double c[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) c[j] = 0.0;
    m.T0 = 0.0;
    m.iT0 = 1.0;
    m.clear();
    bool found = false;
    const int nreg = cd.mix.nreg;
#pragma clang loop unroll(disable)
    for (int r = 0; r < nreg; ++r) {
        const double lo = cd.mix.lo[r], hi = cd.mix.hi[r];
        if (!found && T >= lo && T <= hi) {
            found = true;
            const bool flat = cd.mix.flat[r] != 0;
            m.T0 = cd.mix.T0[r];
            m.iT0 = cd.mix.iT0[r];
            if (flat) {
                m.lo = lo;
                m.hi = hi;
            }
            double w = 1.0;
#pragma clang loop unroll(disable)
            for (int k = 0; k < (flat ? 1 : 2); ++k) {
                const double(*t)[8] = cd.mix.c[r][k];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    double acc = y[0] * t[0][j];
#pragma unroll
                    for (int s = 1; s < NSP; ++s) acc = fma(y[s], t[s][j], acc);
                    c[j] = fma(w, acc, c[j]);
                }
                w = T - m.T0;
            }
        }
    }
    m.a0 = c[0];
    m.a1 = c[1];
    m.q0 = c[2] - lin;
    m.q1 = c[3];
    m.q2 = c[4];
    m.q3 = c[5];
    m.q4 = c[6];
    m.H0 = fma(-lin, m.T0, c[7]) + cst;
}

__device__ __forceinline__ double tpg_mix_slope(const TpgMix& m, double z, double rT) {
    const double q = fma(fma(fma(fma(m.q4, z, m.q3), z, m.q2), z, m.q1), z, m.q0);
    return fma(fma(m.a0, rT, m.a1), rT, q);
}

// Value and slope of the summed curve at T.  Below 1e-3 K (only a state without physical
// meaning gets there; the curves' constant-Cp extension has a0 = a1 = 0) the logarithm and the
// reciprocal are those of 1e-3 K.
__device__ __forceinline__ void tpg_mix_eval(const TpgMix& m, double T, double& val, double& slope) {
    const double Tp = fmax(T, 1.0e-3), rT = quick_rcp(Tp), z = T - m.T0;
    double p = fma(0.2 * m.q4, z, 0.25 * m.q3);
    p = fma(fma(fma(p, z, (1.0 / 3.0) * m.q2), z, 0.5 * m.q1), z, m.q0);
    p = fma(m.a0, rT * m.iT0, p);
    val = fma(p, z, fma(m.a1, log(Tp * m.iT0), m.H0));
    slope = tpg_mix_slope(m, z, rT);
}

// The specific energy of a composition at T.
template <int NSP>
__device__ __forceinline__ double tpg_energy(const ChemDev& cd, const double* massf, double T) {
    double y[NSP], Rm = 0.0, u, Cv;
#pragma unroll
    for (int i = 0; i < NSP; ++i) {
        y[i] = massf[i] * cd.R[i];
        Rm += y[i];
    }
    TpgMix m;
    tpg_mix_build<NSP>(cd, y, Rm, 0.0, T, m);
    tpg_mix_eval(m, T, u, Cv);
    return u;
}

// Cv at T from the curve of a temperature solve (rebuilt if T lies outside its range).
template <int NSP>
__device__ __forceinline__ double tpg_Cv(const ChemDev& cd, const double* massf, double T, TpgMix& m) {
    if (!m.covers(T)) {
        double y[NSP], Rm = 0.0;
#pragma unroll
        for (int i = 0; i < NSP; ++i) {
            y[i] = massf[i] * cd.R[i];
            Rm += y[i];
        }
        tpg_mix_build<NSP>(cd, y, Rm, 0.0, T, m);
    }
    return tpg_mix_slope(m, T - m.T0, quick_rcp(fmax(T, 1.0e-3)));
}

// therm_perf_gas_mix_eos.d:68-151 with the safeguarded Newton of nm/newton.d:71-140.
// T and u are in/out as in the reference: every evaluation of the zero function writes T
// and u, and a converged root then overwrites T, so u ends as the energy of the last
// evaluated temperature.  Returns false where the reference throws; T is then restored
// and u = energy(T), which is the state the reference leaves behind.  m: the summed curve of
// the last evaluation, for the callers that go on to Cv.
//
// The reference evaluates u at both ends of the bracket [T1, T2] = [T - 500, T + 500] only
// for the signs of f = e_tgt - u there (and exact zeros), then starts the Newton iteration
// with an evaluation at T.  Here the evaluation at T comes first, and with it the signs are
// often fixed without the two end evaluations: u(T) rises at Cv >= 1.5 R_mix for any gas
// (translational energy alone; the CEA curves, their blends and their constant-Cp
// extensions all keep Cp >= 2.5 R per species), so with g = e_tgt - u(T),
//   f(T1) >= g + 1.4 R_mix (T - T1)   and   f(T2) <= g - 1.4 R_mix (T2 - T).
// When the first bound is above and the second below a rounding margin (1e-6 of the
// energies + 1 J/kg, against ~1e5 J/kg of slope over 500 K), f(T1) > 0 > f(T2) as the
// reference would compute them: its pass 0 takes the bracket (xH, xL) = (T1, T2) and the
// same iteration from T.  Otherwise (a root far from T, a temperature near the 10 K floor, a
// negative mass fraction) the ends are evaluated and the reference's passes run as written.
// One loop serves every evaluation (at T, at the ends, at the iterates), so the curve's code
// stands once: a kernel that calls this is 6 to 10 times smaller than with an inlined
// evaluation at each place, which lone waves of small grids feel as instruction fetches.
template <int NSP>
__device__ __forceinline__ bool tpg_update_temperature(const ChemDev& cd, const double* massf, double& T, double& u,
                                                       TpgMix& m) {
    enum { AT_T, AT_MIN, AT_MAX, ITERATE };
    const double Tsave = T;
    const double TOL = 1.0e-6;
    const double e_tgt = u;
    const double delT = 1000.0;
    const double T1 = fmax(T - 0.5 * delT, CH_T_MIN);
    const double T2 = T1 + delT;
    double y[NSP], Rm = 0.0;
    bool nonneg = true;
#pragma unroll
    for (int i = 0; i < NSP; ++i) {
        y[i] = massf[i] * cd.R[i];
        Rm += y[i];
        nonneg = nonneg && (massf[i] >= 0.0);
    }
    m.clear();
    int at = AT_T, pass = 0, j = 0;
    double u0 = 0.0, Cv0 = 0.0, fL = 0.0, xL = 0.0, xH = 0.0, rts = Tsave, dx = 0.0, dxold = 0.0;
    while (true) {
        double Cv;
        if (!m.covers(T)) tpg_mix_build<NSP>(cd, y, Rm, 0.0, T, m);
        tpg_mix_eval(m, T, u, Cv);
        double f0 = e_tgt - u;
        bool next_pass = false;
        if (at == ITERATE) {
            if (f0 < 0.0) xL = rts;
            else xH = rts;
            next_pass = (++j == 30);
        } else if (at == AT_T) {
            u0 = u;
            Cv0 = Cv;
            const double slope = 1.4 * Rm;
            const double margin = 1.0e-6 * (fabs(e_tgt) + fabs(u0)) + 1.0;
            const bool signs_known = nonneg && (Tsave - T1 >= 1.0) && (T2 - Tsave >= 1.0) &&
                                     (f0 + slope * (Tsave - T1) > margin) && (f0 - slope * (T2 - Tsave) < -margin);
            if (!signs_known) {
                T = T1;
                at = AT_MIN;
                continue;
            }
            xH = T1;
            xL = T2;
            dx = dxold = T2 - T1;
            at = ITERATE;
        } else if (at == AT_MIN) {
            fL = f0;
            T = (pass == 0) ? T2 : CH_T_MAX;
            at = AT_MAX;
            continue;
        } else {
            const double xMin = (pass == 0) ? T1 : CH_T_MIN, xMax = (pass == 0) ? T2 : CH_T_MAX, fH = f0;
            if ((fL > 0.0 && fH > 0.0) || (fL < 0.0 && fH < 0.0)) {
                next_pass = true;
            } else {
                if (fL == 0.0) { T = xMin; return true; }
                if (fH == 0.0) { T = xMax; return true; }
                if (fL < 0.0) { xL = xMin; xH = xMax; }
                else { xH = xMin; xL = xMax; }
                rts = Tsave;
                dx = dxold = xMax - xMin;
                u = u0;
                Cv = Cv0;
                f0 = e_tgt - u0;
                j = 0;
                at = ITERATE;
            }
        }
        if (next_pass) {
            if (++pass == 2) break;
            T = CH_T_MIN;
            at = AT_MIN;
            continue;
        }
        const double df0 = -1.0 * Cv;
        if ((((rts - xH) * df0 - f0) * ((rts - xL) * df0 - f0) > 0.0) || (fabs(2.0 * f0) > fabs(dxold * df0))) {
            dxold = dx;
            dx = 0.5 * (xH - xL);
            rts = xL + dx;
            T = rts;
            if (xL == rts) return true;
        } else {
            dxold = dx;
            dx = quick_div(f0, df0);
            const double tmp = rts;
            rts -= dx;
            T = rts;
            if (tmp == rts) return true;
        }
        if (fabs(dx) < TOL) return true;
    }
    T = Tsave;
    u = u0;
    return false;
}

// therm_perf_gas.d:394-404: frozen sound speed sqrt(gamma * (R T)), gamma = Cp/Cv, from the
// curve of a temperature solve.
template <int NSP>
__device__ __forceinline__ double tpg_sound_speed(const ChemDev& cd, const double* massf, double T, TpgMix& m) {
    const double R = tpg_Rmix<NSP>(cd, massf);
    const double Cv = tpg_Cv<NSP>(cd, massf, T, m);
    const double gamma = quick_div(Cv + R, Cv);
    return sqrt(gamma * (R * T));
}

// c^n for the stoichiometric coefficients 1..3 of reaction.d's rate products (the host
// rejects other coefficients).
__device__ __forceinline__ double ch_ipow(double c, int n) {
    return (n == 1) ? c : (n == 2) ? c * c : c * (c * c);
}
// pow(P_atm/(R_u T), nuSum) of reaction.d:43-44 for whole nuSum.
__device__ __forceinline__ double ch_pow_nusum(double x, double nuSum) {
    return (nuSum == 0.0) ? 1.0 : (nuSum == 1.0) ? x : (nuSum == -1.0) ? 1.0 / x : (nuSum == 2.0) ? x * x : pow(x, nuSum);
}

// ln t to about twice the working precision's last bit: the rounding of log (up to 9e-16 for a
// temperature) is what t exp(-log t) differs from 1 by.
struct LnPair {
    double hi, lo;
};
__device__ __forceinline__ LnPair ln_pair(double t) {
    LnPair l;
    l.hi = log(t);
    l.lo = fma(t, exp(-l.hi), -1.0);
    return l;
}

// A T^n exp(-C / T) of rate_constant.d as A exp(n ln T - C / T), rT = 1 / T: one exponential
// instead of a power and an exponential (a power is four times the exponential's code and
// time).  The rounding errors of the exponent, some 1e-15 and so of the rate constant where they
// stay, are summed apart and applied to first order.
__device__ __forceinline__ double arrhenius(double A, double n, double C, double T, double rT, const LnPair& l) {
    const double a = n * l.hi, b = C * rT;
    const double x = a - b, bb = x - a;
    double e = (a - (x - bb)) - (b + bb);                           // x + e = a - b
    e += fma(n, l.hi, -a) - fma(C, rT, -b);                         // the products' errors
    e += fma(n, l.lo, -(b * fma(-T, rT, 1.0)));                     // those of ln T and of 1 / T
    const double v = A * exp(x);
    return fma(v, e, v);
}

// reaction_mechanism.d:50-63 with reaction.d:27-52 (equilibrium constant), 94-143 and
// rate_constant.d (Arrhenius A T^n exp(-C/T)); T clamped to the mechanism's tempLimits.
// Participants are summed in ascending species order, the order of the reference's
// sorted participant list.  The reactions pass through one copy of the code: unrolled, with
// its powers, the setup kernel of 5 reactions was 64 KB of code, and the 12 workgroups of a
// small grid spent 30 us on fetching it.
template <int NSP, int NRM>
__device__ __forceinline__ void eval_rate_constants(const ChemDev& cd, double Tin, double* kf, double* kb) {
    double T = Tin;
    if (T < cd.T_lower) T = cd.T_lower;
    if (T > cd.T_upper) T = cd.T_upper;
    const LnPair lnT = ln_pair(T);
    const CeaT pw(T, lnT.hi);
    double g[NSP];
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        double h, sv;
        cea_h_s(cd.cea[s], pw, h, sv);
        g[s] = (h - T * sv) * cd.M[s];
    }
#pragma unroll
    for (int ir = 0; ir < NRM; ++ir) {
        kf[ir] = 0.0;
        kb[ir] = 0.0;
    }
    const double RT = CH_R_UNIVERSAL * T, c_atm = CH_P_ATM / RT;
    const int nr = cd.nr;
#pragma clang loop unroll(disable)
    for (int ir = 0; ir < nr; ++ir) {
        const ReacDev& r = cd.r[ir];
        double Keq = 1.0;
        if (r.f_from_eq || r.b_from_eq) {
            double dG = 0.0, nuSum = 0.0;
#pragma unroll
            for (int s = 0; s < NSP; ++s) {
                if (!r.part[s]) continue;
                dG += r.nu[s] * g[s];
                nuSum += r.nu[s];
            }
            Keq = exp(-dG / RT) * ch_pow_nusum(c_atm, nuSum);
        }
        double kfv = 0.0, kbv = 0.0;
        if (!r.f_from_eq) kfv = arrhenius(r.fA, r.fn, r.fC, T, pw.rT, lnT);
        if (!r.b_from_eq) kbv = arrhenius(r.bA, r.bn, r.bC, T, pw.rT, lnT);
        if (r.f_from_eq) kfv = kbv * Keq;
        if (r.b_from_eq) kbv = kfv / Keq;
        if constexpr (NRM > 8) {  // arrays of this size live in memory
            kf[ir] = kfv;
            kb[ir] = kbv;
        } else {
#pragma unroll
            for (int j = 0; j < NRM; ++j) {
                kf[j] = (j == ir) ? kfv : kf[j];
                kb[j] = (j == ir) ? kbv : kb[j];
            }
        }
    }
}

// The forward and backward rates of one reaction row (dense form) at conc, with c2 = conc^2:
// reaction.d:289-330 (eval_forward_rate / eval_backward_rate) for lists in ascending order.
// With the structure in WALK every select below is decided at compile time; the products and
// sums and their order are the same.
template <int NSP, int WALK>
__device__ __forceinline__ void dense_row_rates(const RateRow& rr, int ir, double kf, double kb, const double* conc,
                                                const double* c2, double& wf_out, double& wb_out) {
    constexpr bool SHAPED = WALK > WALK_ROWS;
    int code[NSP];
#pragma unroll
    for (int s = 0; s < NSP; ++s) code[s] = SHAPED ? MechShape<WALK>::code(ir, s) : rr.code[s];
    const int flags = SHAPED ? MechShape<WALK>::flags(ir) : rr.flags;
    double collider = 0.0;
    if (!SHAPED || (flags & 1)) {
#pragma unroll
        for (int s = 0; s < NSP; ++s) collider += (code[s] & 256) ? rr.eff[s] * conc[s] : 0.0;
    }
    double wf = (flags & 1) ? kf * collider : kf;
    double wb = (flags & 1) ? kb * collider : kb;
    // c^e for e in 0..3 as (c or 1) * (c^2 or 1): c * (c * c) for e = 3, as ch_ipow
#pragma unroll
    for (int s = 0; s < NSP; ++s) wf *= ((code[s] & 1) ? conc[s] : 1.0) * ((code[s] & 2) ? c2[s] : 1.0);
#pragma unroll
    for (int s = 0; s < NSP; ++s) wb *= ((code[s] & 4) ? conc[s] : 1.0) * ((code[s] & 8) ? c2[s] : 1.0);
    wf_out = wf;
    wb_out = wb;
}

// Net coefficient of species s in a dense row (4-bit two's complement in bits 4-7).
template <int WALK>
__device__ __forceinline__ int dense_row_nu(const RateRow& rr, int ir, int s) {
    const int code = (WALK > WALK_ROWS) ? MechShape<WALK>::code(ir, s) : rr.code[s];
    return (int)((unsigned)code << 24) >> 28;
}

// reaction_mechanism.d:83-96 (eval_split_rates) with reaction.d's forward/backward rates
// (collider sum over the efficiency list, then the concentration products in list order)
// and production/loss per participant in reaction order.
//
// WALK_ROWS and the shapes (every list of the mechanism in ascending species order, rr[] filled;
// the host picks the instantiation) take a branch-free walk over the rows: an absent reactant or
// product multiplies by exactly 1, a species outside the third-body list or the reaction
// adds exactly 0 (a selected zero, not a product with zero), and a reaction without third
// body takes kf as it is, so every result equals the list walk bit for bit while the table
// words load in bulk instead of one load and branch per entry.
template <int NSP, int NRM, int WALK>
__device__ __forceinline__ void eval_split_rates(const ChemDev& cd, const double* kf, const double* kb,
                                                 const double* conc, double* q, double* L) {
#pragma unroll
    for (int s = 0; s < NSP; ++s) { q[s] = 0.0; L[s] = 0.0; }
    if constexpr (WALK != WALK_LIST) {
        double c2[NSP];
#pragma unroll
        for (int s = 0; s < NSP; ++s) c2[s] = conc[s] * conc[s];
        const int nr = cd.nr;
#pragma unroll
        for (int ir = 0; ir < NRM; ++ir) {
            if (WALK == WALK_ROWS && ir >= nr) break;  // a shape has NRM reactions
            const RateRow& rr = cd.rr[ir];
            double wf, wb;
            dense_row_rates<NSP, WALK>(rr, ir, kf[ir], kb[ir], conc, c2, wf, wb);
#pragma unroll
            for (int s = 0; s < NSP; ++s) {
                const int nu = dense_row_nu<WALK>(rr, ir, s);
                const double m = (double)(nu < 0 ? -nu : nu);
                const bool pos = nu > 0;
                q[s] += (nu != 0) ? m * (pos ? wf : wb) : 0.0;
                L[s] += (nu != 0) ? m * (pos ? wb : wf) : 0.0;
            }
        }
    } else {
#pragma unroll
        for (int ir = 0; ir < NRM; ++ir) {
            if (ir >= cd.nr) continue;
            const ReacDev& r = cd.r[ir];
            double collider = 0.0, wf, wb;
            if (r.sorted) {
                if (r.collider) {
#pragma unroll
                    for (int s = 0; s < NSP; ++s)
                        if ((r.eff_set >> s) & 1u) collider += r.eff_d[s] * conc[s];
                }
                wf = r.collider ? kf[ir] * collider : kf[ir];
#pragma unroll
                for (int s = 0; s < NSP; ++s)
                    if (r.reac_d[s]) wf *= ch_ipow(conc[s], r.reac_d[s]);
                wb = r.collider ? kb[ir] * collider : kb[ir];
#pragma unroll
                for (int s = 0; s < NSP; ++s)
                    if (r.prod_d[s]) wb *= ch_ipow(conc[s], r.prod_d[s]);
            } else {
                if (r.collider) {
#pragma unroll
                    for (int e = 0; e < NSP; ++e)
                        if (e < r.neff) collider += r.eff[e] * pick<NSP>(conc, r.eff_sp[e]);
                }
                wf = r.collider ? kf[ir] * collider : kf[ir];
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (k < r.nreac) wf *= ch_ipow(pick<NSP>(conc, r.reac_sp[k]), r.reac_nu[k]);
                wb = r.collider ? kb[ir] * collider : kb[ir];
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (k < r.nprod) wb *= ch_ipow(pick<NSP>(conc, r.prod_sp[k]), r.prod_nu[k]);
            }
#pragma unroll
            for (int s = 0; s < NSP; ++s) {
                const int nu = r.nu[s];
                if (nu > 0) {
                    q[s] += nu * wf;
                    L[s] += nu * wb;
                } else if (nu < 0) {
                    q[s] += -nu * wb;
                    L[s] += -nu * wf;
                }
            }
        }
    }
}

// reaction_mechanism.d:162-203
template <int NSP, int NRM, int WALK>
__device__ __forceinline__ double estimate_step_size(const ChemDev& cd, const double* kf, const double* kb, const double* conc) {
    const double MUCH_LARGER_FACTOR = 10000.0, ZERO_EPS = 1.0e-50, ZERO_TOL = 1.0e-30, EPS1 = 1.0e-3;
    double q[NSP], L[NSP];
    eval_split_rates<NSP, NRM, WALK>(cd, kf, kb, conc, q, L);
    double min_dt = 1.0e6, dt;
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        double c = conc[s];
        if (c > 0.0 && (fabs(q[s] - L[s]) > ZERO_TOL)) {
            if (q[s] > MUCH_LARGER_FACTOR * L[s]) dt = c / (L[s] + ZERO_EPS);
            else dt = fabs(c / (q[s] - L[s]));
            min_dt = (dt < min_dt) ? dt : min_dt;
        }
    }
    double dt_chem = EPS1 * min_dt;
    dt_chem = (1.0e-10 < dt_chem) ? 1.0e-10 : dt_chem;
    dt_chem = (dt_chem < 1.0e-15) ? 1.0e-15 : dt_chem;
    return dt_chem;
}

// AlphaQssStep.opCall, chemistry_update.d:533-655: predictor, up to maxIters correctors
// with alpha-bar from p_p, convergence against the first predictor, and the step
// suggestion from three Newton iterations for sqrt(sigma).  yOut is written on success.
// Trip 0 of the loop is the predictor (rates at y0), trips 1..maxIters the correctors
// (rates at yp), so the rate code is inlined once:
//   predictor  yp = y0 + h (q0 - p0 y0) / (1 + alpha(p0) h p0)
//   corrector  yc = y0 + h (q~ - p- y0) / (1 + alpha(pp) h p-),
//              q~ = alpha(pp) qp + (1 - alpha(pp)) q0,  p- = (p0 + pp) / 2
// The reference's alpha(r), r = 1 / (p h + 1e-50) (:599-604), is N(x) / D(x) in x = p h with
//   N = x^3 + 11 x^2 + 60 x + 180,  D = x^3 + 12 x^2 + 60 x + 360,  D - N = x^2 + 180,
// so both forms are taken over the common denominator D,
//   y = y0 + (h (N q + (D - N) q0) - x- y0 D) / (D + N x-),  x- = h p-,
// with 2 divisions a species and trip (p, and y) instead of 4, and neither a reciprocal of p h
// nor alpha itself.  x is bounded at 1e60, where alpha is 1, so that x^3 stays finite.
// sigma = max n / d over the species is kept as its n and d (compared by cross products), and
// the three Newton iterations from x = sigma for its root, x <- (x + sigma / x) / 2, give
// with S = n + d, P = S^2 + 4 n d
//   1 / x3 = 8 d P S / (P^2 + 16 n d S^2):
// one division for the step suggestion instead of 8.
template <int NSP, int NRM, int WALK>
__device__ __forceinline__ bool alpha_qss_step(const ChemDev& cd, const double* kf, const double* kb, const double* y0,
                                               double h, double* yOut, double& hSuggest, int& iters) {
    const double ZERO_EPS = 1.0e-50;
    double q0[NSP], x0[NSP], yp[NSP], yp0[NSP], yc[NSP];
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        q0[s] = 0.0;
        x0[s] = 0.0;
        yp[s] = y0[s];
    }
    bool converged = false;
    for (int trip = 0; trip <= cd.maxIters; ++trip) {
        const bool pred = (trip == 0);
        double q[NSP], L[NSP];
        eval_split_rates<NSP, NRM, WALK>(cd, kf, kb, yp, q, L);  // yp = y0 on the predictor trip
        bool passes = true;
#pragma unroll
        for (int s = 0; s < NSP; ++s) {
            const double xp = h * quick_div(L[s], yp[s] + ZERO_EPS);
            if (pred) {
                q0[s] = q[s];
                x0[s] = xp;
            }
            const double xm = 0.5 * (x0[s] + xp);  // xp itself on the predictor trip
            const double x = fmin(xp, 1.0e60);
            const double N = fma(fma(x + 11.0, x, 60.0), x, 180.0);
            const double W = fma(x, x, 180.0);  // D - N
            const double D = N + W;
            // on the predictor trip q = q0, and N q + W q0 is D q0
            const double num = fma(-(xm * y0[s]), D, h * fma(N, q[s], W * q0[s]));
            const double ynew = y0[s] + quick_div(num, fma(N, xm, D));
            if (pred) {
                yp0[s] = ynew;
            } else if (ynew >= ZERO_EPS) {
                if (fabs(ynew - yp0[s]) >= (cd.eps1 * (ynew + cd.delta))) passes = false;
            }
            yc[s] = ynew;
        }
        if (!pred) {
            ++iters;
            if (passes) {
                converged = true;
                break;
            }
        }
#pragma unroll
        for (int s = 0; s < NSP; ++s) yp[s] = yc[s];
    }
    double n = 0.0, d = 1.0;
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        if (yc[s] < ZERO_EPS) continue;
        const double ns = fabs(yc[s] - yp0[s]), ds = cd.eps2 * (yc[s] + cd.delta);
        if (ns * d > n * ds) {
            n = ns;
            d = ds;
        }
    }
    if (n <= 0.0) {
        hSuggest = 10.0 * h;
    } else {
        const double S = n + d, nd4 = 4.0 * n * d;
        const double P = fma(S, S, nd4);
        hSuggest = h * (quick_div(8.0 * d * P * S, fma(P, P, 4.0 * nd4 * S * S)) + 0.005);
    }
    if (converged) {
#pragma unroll
        for (int s = 0; s < NSP; ++s) yOut[s] = yc[s];
    }
    return converged;
}

// RKFStep.opCall, chemistry_update.d:385-484 (Cash-Karp tableau); yOut is always written.
template <int NSP, int NRM, int WALK>
__device__ __forceinline__ bool rkf_step(const ChemDev& cd, const double* kf, const double* kb, const double* y0, double h,
                         double* yOut, double& hSuggest, double* yLast = nullptr) {
    const double a21 = 1. / 5., a31 = 3. / 40., a32 = 9. / 40., a41 = 3. / 10., a42 = -9. / 10., a43 = 6. / 5.,
                 a51 = -11. / 54., a52 = 5. / 2., a53 = -70. / 27., a54 = 35. / 27., a61 = 1631. / 55296.,
                 a62 = 175. / 512., a63 = 575. / 13824., a64 = 44275. / 110592., a65 = 253. / 4096.;
    const double b51 = 37. / 378., b53 = 250. / 621., b54 = 125. / 594., b56 = 512. / 1771., b41 = 2825. / 27648.,
                 b43 = 18575. / 48384., b44 = 13525. / 55296., b45 = 277. / 14336., b46 = 1.0 / 4.0;
    double k1[NSP], k2[NSP], k3[NSP], k4[NSP], k5[NSP], k6[NSP], yT[NSP], q[NSP], L[NSP];
    auto rates = [&](const double* y, double* k) {
        eval_split_rates<NSP, NRM, WALK>(cd, kf, kb, y, q, L);
#pragma unroll
        for (int s = 0; s < NSP; ++s) k[s] = q[s] - L[s];
    };
    rates(y0, k1);
#pragma unroll
    for (int s = 0; s < NSP; ++s) yT[s] = y0[s] + h * (a21 * k1[s]);
    rates(yT, k2);
#pragma unroll
    for (int s = 0; s < NSP; ++s) yT[s] = y0[s] + h * (a31 * k1[s] + a32 * k2[s]);
    rates(yT, k3);
#pragma unroll
    for (int s = 0; s < NSP; ++s) yT[s] = y0[s] + h * (a41 * k1[s] + a42 * k2[s] + a43 * k3[s]);
    rates(yT, k4);
#pragma unroll
    for (int s = 0; s < NSP; ++s) yT[s] = y0[s] + h * (a51 * k1[s] + a52 * k2[s] + a53 * k3[s] + a54 * k4[s]);
    rates(yT, k5);
#pragma unroll
    for (int s = 0; s < NSP; ++s)
        yT[s] = y0[s] + h * (a61 * k1[s] + a62 * k2[s] + a63 * k3[s] + a64 * k4[s] + a65 * k5[s]);
    rates(yT, k6);
    // the concentrations of the last rate evaluation (whose reaction rates the
    // two-temperature reactor's energy source reads)
    if (yLast) {
#pragma unroll
        for (int s = 0; s < NSP; ++s) yLast[s] = yT[s];
    }
    double err = 0.0;
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        yOut[s] = y0[s] + h * (b51 * k1[s] + b53 * k3[s] + b54 * k4[s] + b56 * k6[s]);
        double yE = yOut[s] - (y0[s] + h * (b41 * k1[s] + b43 * k3[s] + b44 * k4[s] + b45 * k5[s] + b46 * k6[s]));
        double ay0 = fabs(y0[s]), ay1 = fabs(yOut[s]);
        double sk = cd.errTol + cd.errTol * ((ay0 < ay1) ? ay1 : ay0);
        err += (yE / sk) * (yE / sk);
    }
    err = sqrt(err / NSP);
    const double maxscale = 10.0, minscale = 0.2, safe = 0.9, alpha = 0.2;
    double scale;
    if (err <= 1.0) {
        if (err == 0.0) {
            scale = maxscale;
        } else {
            scale = safe * pow(err, -alpha);
            if (scale < minscale) scale = minscale;
            if (scale > maxscale) scale = maxscale;
        }
        hSuggest = scale * h;
        return true;
    }
    scale = safe * pow(err, -alpha);
    scale = (scale < minscale) ? minscale : scale;
    hSuggest = scale * h;
    return false;
}

// Phobos std.algorithm.sum over NSP doubles: 0.0 + the pairwise sum of the D runtime
// (pairs summed into a store collapsed at powers of two, the store then summed from its
// last entry down).
template <int NSP>
__device__ __forceinline__ double phobos_sum(const double* x) {
    double store[NSP];
    int idx = 0;
#pragma unroll
    for (int k = 0; k < NSP / 2; ++k) {
        store[idx] = x[2 * k] + x[2 * k + 1];
        int lastToKeep = idx - __builtin_ctz((unsigned)(k + 1));
        while (idx > lastToKeep) {
            store[idx - 1] += store[idx];
            --idx;
        }
        ++idx;
    }
    if (NSP % 2 == 1) {
        store[idx] = x[NSP - 1];
        ++idx;
    }
    double s = store[idx - 1];
    for (int j = idx - 2; j >= 0; --j) s += store[j];
    return 0.0 + s;
}

// gas_model.d:255-271 (conc2massf) followed by the mass-fraction sum of
// chemistry_update.d:180-185 and 292-294.
template <int NSP>
__device__ __forceinline__ double conc_to_massf(const ChemDev& cd, const double* conc, double rho, double* massf) {
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        massf[s] = conc[s] * cd.M[s] / rho;
        if (massf[s] < CH_MIN_MASSF) massf[s] = 0.0;
    }
    return phobos_sum<NSP>(massf);
}

}  // namespace gdtk
