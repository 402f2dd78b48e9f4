// tt_device.hpp -- two-temperature air on gfx950: the TwoTemperatureAir gas
// (src/gas/two_temperature_air.d, neutral species) and the TwoTemperatureAirKinetics reactor
// (src/kinetics/two_temperature_air_kinetics.d), one lane per cell.  FP64, no FMA contraction.
// The formulas and the order of the steps are the reference's; within an expression sums over
// the species are taken first and quotients by quick_div, so results agree with the reference's
// operation order to rounding.  The mechanism is in dense form (ascending lists, as prep-chem
// writes them), with explicit backward rates.
#pragma once
#include <hip/hip_runtime.h>

#include "chem_device.hpp"

namespace gdtk {

constexpr double TT_T_REF = 298.15;                  // two_temperature_air.d:24
constexpr double TT_AVOGADRO = 6.02214e23;           // physical_constants.d:18
constexpr double TT_BOLTZMANN = 1.380658e-23;        // physical_constants.d:17
constexpr double TT_SMALL_MOLE_FRACTION = 1.0e-15;   // gas_model.d:42
constexpr double TT_PI = 3.141592653589793;          // to!double(PI)

// Per-species constants of the gas and the relaxation model, computed on the host as the
// reference's constructors do (two_temperature_air.d:186-205, kinetics :387-439).
struct TTDev {
    int molecular[CH_MAX_SP];
    double Cp_tr_rot[CH_MAX_SP], del_hf[CH_MAX_SP];
    double sA[CH_MAX_SP], sB[CH_MAX_SP];      // Cp_tr_rot T_REF - del_hf, Cp_tr_rot - R
    double A_MW[CH_MAX_SP];                   // Millikan-White A (0 for atoms)
    // exp(-0.015 A_s mu_sc^(1/4) - 18.42), mu_sc the reduced mass in g/mol: the part of the
    // correlation that does not depend on T
    double K_MW[CH_MAX_SP][CH_MAX_SP];
    double cbar[CH_MAX_SP];                   // sqrt(8 k / (pi m)), m = M / N_A
    double abs_tol, rel_tol;                  // energy step
};

// GasState of a cell: T_modes[0] = Tv, u_modes[0] = uv.
template <int NSP>
struct TTCell {
    double rho, p, T, Tv, u, uv;
    double massf[NSP];
};

// The vibro-electronic energy of a weighted mixture, sum of y_s / R_s e_ve,s(T) with
// e_ve = h - Cp_tr,rot (T - T_REF) - del_hf (two_temperature_air.d:573-591, its slope
// :673-680), as one curve (TpgMix); w: weights per unit mass.
template <int NSP>
__device__ __forceinline__ void tt_ev_build(const ChemDev& cd, const TTDev& td, const double* w, double T, TpgMix& m) {
    double y[NSP], lin = 0.0, cst = 0.0;
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        y[s] = w[s] * cd.R[s];
        lin += w[s] * td.Cp_tr_rot[s];
        cst += w[s] * td.sA[s];
    }
    tpg_mix_build<NSP>(cd, y, lin, cst, T, m);
}

// :698-740 vibElecTemperature: Newton from the state's Tv; false where the reference throws.
// m: the mixture's curve, kept from one call to the next while the mass fractions stay (the six
// stages of an energy step share one build).
template <int NSP>
__device__ __forceinline__ bool tt_vib_temperature(const ChemDev& cd, const TTDev& td, const TTCell<NSP>& Q,
                                                   TpgMix& m, double& Tv_out) {
    const int MAX_ITERATIONS = 20;
    const double TOL = 1.0e-6, E_TOL = 0.01;
    double T_guess = Q.Tv;
    for (int count = 0;; ++count) {
        double e, Cv;
        if (!m.covers(T_guess)) tt_ev_build<NSP>(cd, td, Q.massf, T_guess, m);
        tpg_mix_eval(m, T_guess, e, Cv);
        const double f_guess = e - Q.uv;
        if (count == 0 && fabs(f_guess) < E_TOL) {
            Tv_out = Q.Tv;
            return true;
        }
        if (count == MAX_ITERATIONS) break;
        const double dT = quick_div(-f_guess, Cv);
        T_guess += dT;
        if (fabs(dT) < TOL) {
            Tv_out = T_guess;
            return true;
        }
    }
    return false;
}

// :275-291 update_thermo_from_rhou: T by direct inversion, Tv by Newton, p (perf_gas_mix_eos.d:43-49)
template <int NSP>
__device__ __forceinline__ bool tt_update_from_rhou(const ChemDev& cd, const TTDev& td, TTCell<NSP>& Q,
                                                    TpgMix& m) {
    double sumA = 0.0, sumB = 0.0;
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        sumA += Q.massf[s] * td.sA[s];
        sumB += Q.massf[s] * td.sB[s];
    }
    Q.T = quick_div(Q.u + sumA, sumB);
    double Tv;
    if (!tt_vib_temperature<NSP>(cd, td, Q, m, Tv)) return false;
    Q.Tv = Tv;
    double Rmix = 0.0;
#pragma unroll
    for (int s = 0; s < NSP; ++s) Rmix += Q.massf[s] * cd.R[s];
    Q.p = Q.rho * Rmix * Q.T;
    return true;
}

// reaction_mechanism.d:50-63 with rate_constant.d:72-75 (Arrhenius at T) and :391-394
// (Park at T^s Tv^(1-s)); T clamped to the temperature limits, Tv not.  The logarithm of
// Park's temperature is the weighted sum of the two, kept as a pair like theirs.  The reactions
// pass through one copy of the code.
template <int NRM>
__device__ __forceinline__ void tt_rate_constants(const ChemDev& cd, double Tin, double Tv, double* kf, double* kb) {
    double T = Tin;
    if (T < cd.T_lower) T = cd.T_lower;
    if (T > cd.T_upper) T = cd.T_upper;
    const LnPair lnT = ln_pair(T), lnTv = ln_pair(Tv);
    const double rT = quick_rcp(T);
#pragma unroll
    for (int ir = 0; ir < NRM; ++ir) {
        kf[ir] = 0.0;
        kb[ir] = 0.0;
    }
    const int nr = cd.nr;
#pragma clang loop unroll(disable)
    for (int ir = 0; ir < nr; ++ir) {
        const ReacDev& r = cd.r[ir];
        double k[2];
#pragma clang loop unroll(disable)
        for (int way = 0; way < 2; ++way) {
            const double A = way ? r.bA : r.fA, n = way ? r.bn : r.fn, C = way ? r.bC : r.fC;
            double Tk = T, rTk = rT;
            LnPair l = lnT;
            if (way ? r.b_park : r.f_park) {
                const double p = way ? r.b_s : r.f_s, q = 1.0 - p;
                const double a = p * lnT.hi, b = q * lnTv.hi;
                l.hi = a + b;
                const double bb = l.hi - a;
                l.lo = (a - (l.hi - bb)) + (b - bb) + fma(p, lnT.hi, -a) + fma(q, lnTv.hi, -b);
                l.lo = fma(p, lnT.lo, fma(q, lnTv.lo, l.lo));
                const double ex = exp(l.hi);
                Tk = fma(ex, l.lo, ex);
                rTk = quick_rcp(Tk);
            }
            const double v = arrhenius(A, n, C, Tk, rTk, l);
            if (way == 0) k[0] = v;
            else k[1] = v;
        }
#pragma unroll
        for (int j = 0; j < NRM; ++j) {
            kf[j] = (j == ir) ? k[0] : kf[j];
            kb[j] = (j == ir) ? k[1] : kb[j];
        }
    }
}

// two_temperature_air_kinetics.d:398-441 (relaxation time of molecular species isp, from the
// mole fractions and number densities of evalRate) and :444-460 + :521-543 (the exchange
// rate of u_v: Landau-Teller per molecular species plus the chemical source).  g: per species
// the net mass rate per unit mass of mixture of the chemistry step's last evaluation, which
// the source multiplies with e_ve,s(Tv).
//
// What the reference evaluates per species is summed first, since e_ve enters linearly:
//   sum over molecules of w_s (e_ve,s(T) - e_ve,s(Tv)) + sum of g_s e_ve,s(Tv),
//   w_s = massf_s / tau_s,
// are two curves, one at T with weights w and one at Tv with weights g - w (a pass of one loop
// each).  1 / tau_s with tau_s = tauMW + tauP is c_s / (tauMW c_s + 1), c_s = 1 / tauP; the
// Millikan-White exponential is exp(A_s T^(-1/3)) times a constant per pair (3 exponentials a
// rate, not 15).
template <int NSP>
__device__ __forceinline__ double tt_eval_rate(const ChemDev& cd, const TTDev& td, const TTCell<NSP>& Q,
                                               const double* g) {
    double moles[NSP], nsum = 0.0;  // mol per kg
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        moles[s] = quick_div(Q.massf[s], cd.M[s]);
        nsum += moles[s];
    }
    const double Tm13 = rcbrt(Q.T), sqrtT = sqrt(Q.T);
    const double sigma_s = 1e-20, navo = TT_AVOGADRO * Q.rho;
    double w[NSP];
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        w[s] = 0.0;
        if (!td.molecular[s]) continue;
        double total = 0.0, sum = 0.0;
#pragma unroll
        for (int c = 0; c < NSP; ++c) {
            if (moles[c] >= TT_SMALL_MOLE_FRACTION * nsum) {
                sum = fma(moles[c], td.K_MW[s][c], sum);
                total += moles[c];
            }
        }
        const double tauMW = quick_div(sum * exp(td.A_MW[s] * Tm13) * CH_P_ATM, total * Q.p);
        const double coll = sigma_s * (td.cbar[s] * sqrtT) * (navo * moles[s]);  // 1 / tauP
        w[s] = Q.massf[s] * quick_div(coll, fma(tauMW, coll, 1.0));
    }
    double rate = 0.0;
#pragma clang loop unroll(disable)
    for (int k = 0; k < 2; ++k) {
        const double Tk = (k == 0) ? Q.T : Q.Tv;
        TpgMix m;
        double e, slope;
        tt_ev_build<NSP>(cd, td, w, Tk, m);
        tpg_mix_eval(m, Tk, e, slope);
        rate += e;
#pragma unroll
        for (int s = 0; s < NSP; ++s) w[s] = g[s] - w[s];
    }
    return rate;
}

// Cash-Karp: row st of the tableau's stage weights (the last row is the fifth-order result) and
// the fourth-order weights.
__device__ constexpr double TT_CK[6][6] = {{1. / 5., 0, 0, 0, 0, 0},
                                           {3. / 40., 9. / 40., 0, 0, 0, 0},
                                           {3. / 10., -9. / 10., 6. / 5., 0, 0, 0},
                                           {-11. / 54., 5. / 2., -70. / 27., 35. / 27., 0, 0},
                                           {1631. / 55296., 175. / 512., 575. / 13824., 44275. / 110592., 253. / 4096., 0},
                                           {37. / 378., 0, 250. / 621., 125. / 594., 0, 512. / 1771.}};

// :546-706 EnergyStep: Cash-Karp on u_v at fixed total energy uTotal; every stage ends in
// update_thermo_from_rhou.  Returns 1 success, 0 failure (the state keeps the last stage,
// as in the reference), -1 where the Tv iteration fails.  The six stages are passes of one
// loop: unrolled, with the relaxation rate and the Newton iteration inlined six times, the
// kernel was 1.4 MB of code, and its waves waited for instructions.
template <int NSP>
__device__ __forceinline__ int tt_energy_step(const ChemDev& cd, const TTDev& td, TTCell<NSP>& Q, double uTotal,
                                              double h, double& hSuggest, const double* g, TpgMix& m) {
    const double b41 = 2825. / 27648., b43 = 18575. / 48384., b44 = 13525. / 55296., b45 = 277. / 14336.,
                 b46 = 1.0 / 4.0;
    const double uv0 = Q.uv;
    double k[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) k[j] = 0.0;
#pragma clang loop unroll(disable)
    for (int st = 0; st < 6; ++st) {
        const double ks = tt_eval_rate<NSP>(cd, td, Q, g);
        double sum = 0.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            k[j] = (j == st) ? ks : k[j];
            sum += TT_CK[st][j] * k[j];
        }
        Q.uv = uv0 + h * sum;
        Q.u = uTotal - Q.uv;
        if (!tt_update_from_rhou<NSP>(cd, td, Q, m)) return -1;
    }
    const double errEst = Q.uv - (uv0 + h * (b41 * k[0] + b43 * k[2] + b44 * k[3] + b45 * k[4] + b46 * k[5]));
    const double sk = td.abs_tol + td.rel_tol * fmax(fabs(uv0), fabs(Q.uv));
    const double err = fabs(errEst / sk);
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
        return 1;
    }
    scale = fmax(safe * pow(err, -alpha), minscale);
    hSuggest = scale * h;
    return 0;
}

// gas_model.d:255-271 conc2massf into the cell state
template <int NSP>
__device__ __forceinline__ void tt_conc_to_massf(const ChemDev& cd, const double* conc, TTCell<NSP>& Q) {
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        Q.massf[s] = conc[s] * cd.M[s] / Q.rho;
        if (Q.massf[s] < CH_MIN_MASSF) Q.massf[s] = 0.0;
    }
}

struct TTCounts {
    int substeps, attempts;
};

// two_temperature_air_kinetics.d:162-358 opCall: 1 success, 0 where the reference throws
// ThermochemicalReactorUpdateException (the caller restores the input state), -1 where a
// GasModelException escapes (a failed Tv iteration, a bad density).
template <int NSP, int NRM, int WALK>
__device__ __forceinline__ int tt_opcall(const ChemDev& cd, const TTDev& td, TTCell<NSP>& Q, double tInterval,
                                         double& dtSuggest, TTCounts& cnt) {
    const double DT_INCREASE_PERCENT = 10.0, DT_REDUCTION_FACTOR = 10.0, H_MIN = 1.0e-15,
                 ALLOWABLE_MASSF_ERROR = 1.0e-3;
    if (isnan(Q.rho) || !(Q.rho > 0.0)) return -1;  // massf2conc (gas_model.d:246-248)
    double conc0[NSP], concOut[NSP];
#pragma unroll
    for (int s = 0; s < NSP; ++s) {
        conc0[s] = Q.massf[s] * Q.rho / cd.M[s];
        if (conc0[s] < CH_MIN_MOLES) conc0[s] = 0.0;
        concOut[s] = 0.0;
    }
    const double uTotal = Q.u + Q.uv;
    TpgMix m;  // the mixture's e_ve curve of the current mass fractions
    m.clear();
    double kf[NRM], kb[NRM];
    tt_rate_constants<NRM>(cd, Q.T, Q.Tv, kf, kb);
    double t = 0.0, h, dtSave = 0.0;
    if (dtSuggest > tInterval) h = tInterval;
    else if (dtSuggest <= 0.0) h = estimate_step_size<NSP, NRM, WALK>(cd, kf, kb, conc0);
    else h = dtSuggest;
    int cycle = 0;
    for (; cycle < cd.maxSubcycles; ++cycle) {
        dtSave = dtSuggest;
        h = ((tInterval - t) < h) ? (tInterval - t) : h;
        int attempt = 0;
        for (; attempt < cd.maxAttempts; ++attempt) {
            ++cnt.attempts;
            double yLast[NSP];
            const bool r1 = rkf_step<NSP, NRM, WALK>(cd, kf, kb, conc0, h, concOut, dtSuggest, yLast);
            // the reaction rates of the chemistry step's last evaluation
            // (EnergyReactiveSourceTerm: production less loss in reaction order, times M, per
            // unit mass of mixture)
            double q[NSP], L[NSP], g[NSP];
            eval_split_rates<NSP, NRM, WALK>(cd, kf, kb, yLast, q, L);
#pragma unroll
            for (int s = 0; s < NSP; ++s) g[s] = quick_div((q[s] - L[s]) * cd.M[s], Q.rho);
            const int r2 = tt_energy_step<NSP>(cd, td, Q, uTotal, h, dtSuggest, g, m);
            if (r2 < 0) return -1;
            const bool ok = r1 && (r2 == 1);
            bool passes = true;
            if (ok) {
                tt_conc_to_massf<NSP>(cd, concOut, Q);
                m.clear();
                const double massfTotal = phobos_sum<NSP>(Q.massf);
                if (fabs(massfTotal - 1.0) > ALLOWABLE_MASSF_ERROR) passes = false;
            }
            if (ok && passes) {
                t += h;
#pragma unroll
                for (int s = 0; s < NSP; ++s) conc0[s] = concOut[s];
                const double hMax = h * (1.0 + DT_INCREASE_PERCENT / 100.0);
                if (dtSuggest > h) h = (dtSuggest < hMax) ? dtSuggest : hMax;
                break;
            }
            h /= DT_REDUCTION_FACTOR;
            if (h < H_MIN) return 0;
        }
        if (attempt == cd.maxAttempts) return 0;
        ++cnt.substeps;
        if (cd.tight) {
            tt_conc_to_massf<NSP>(cd, conc0, Q);
            m.clear();
            Q.u = uTotal - Q.uv;
            if (!tt_update_from_rhou<NSP>(cd, td, Q, m)) return -1;
            tt_rate_constants<NRM>(cd, Q.T, Q.Tv, kf, kb);
        }
        if (t >= tInterval) {
            if (cycle == 0) dtSave = dtSuggest;
            break;
        }
    }
    if (cycle == cd.maxSubcycles) return 0;
    tt_conc_to_massf<NSP>(cd, concOut, Q);
    const double massfTotal = phobos_sum<NSP>(Q.massf);
#pragma unroll
    for (int s = 0; s < NSP; ++s) Q.massf[s] /= massfTotal;
    dtSuggest = dtSave;
    return 1;
}

}  // namespace gdtk
