// chem.cpp -- host side of the finite-rate chemistry C ABI (include/gdtk_hip.h).
//
// gdtk_hip_chem_create restates the set-up the reference does once per run:
//   ThermallyPerfectGas + CEAThermoCurve construction   src/gas/therm_perf_gas.d:40-120,
//                                                        gas/thermo/cea_thermo_curves.d:24-55
//   ReactionMechanism (participants, net nu)            src/kinetics/reaction.d:58-143
//   ChemistryUpdate configuration                       src/kinetics/chemistry_update.d:51-136
// and gdtk_hip_chem_step is FVCell.thermochemical_increment (src/eilmer/fvcell.d:858-972)
// over a batch of cells, the granularity of the reference's GPU plug-in boundary
// GPUChem.thermochemical_increment (src/eilmer/cuda_gpu_chem.d:155-191).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/gdtk_hip.h"
#include "chem_device.hpp"
#include "chem_launch.hpp"
#include "chem_host.hpp"
#include "host_common.hpp"

namespace gdtk {

static_assert(GDTK_MAX_SPECIES == CH_MAX_SP && GDTK_MAX_REACTIONS == CH_MAX_R, "table sizes");

static std::mutex g_chem_mu;
static std::vector<std::unique_ptr<Chem>> g_chems;

Chem& get_chem(int h) {
    std::lock_guard<std::mutex> lk(g_chem_mu);
    if (h < 0 || h >= (int)g_chems.size() || !g_chems[h]) throw Error(GDTK_ERR_ARG, "bad chemistry handle");
    return *g_chems[h];
}

// One species' segment expanded about T0 (MixTable): {a0, a1, q0..q4, H0}.
static void expand_segment(const double* a, long double T0, double* out) {
    out[0] = a[0];
    out[1] = a[1];
    for (int k = 0; k < 5; ++k) {
        long double q = 0.0L, pw = 1.0L, binom = 1.0L;  // sum over m of a[2 + m] C(m, k) T0^(m - k)
        for (int m = k; m < 5; ++m) {
            q += (long double)a[2 + m] * binom * pw;
            pw *= T0;
            binom = binom * (m + 1) / (m + 1 - k);
        }
        out[2 + k] = (double)q;
    }
    long double h = -(long double)a[0] / T0 + (long double)a[1] * std::log(T0) + (long double)a[7], pw = T0;
    for (int m = 0; m < 5; ++m) {
        h += (long double)a[2 + m] * pw / (m + 1);
        pw *= T0;
    }
    out[7] = (double)h;
}

// What a species' curve is at T (cea_thermo_curves.d:56-70, 137-176, tests in its order): the
// constant-Cp extension (seg = -1 below, -2 above), segment seg alone, or the blend of seg and
// seg + 1.
static void curve_at(const CEADev& c, double T, int& seg, bool& blend) {
    blend = false;
    const int nb = c.nseg + 1;
    auto lo = [&](int i) { return c.T_breaks[i] - 0.5 * c.T_blends[i - 1]; };
    auto hi = [&](int i) { return c.T_breaks[i] + 0.5 * c.T_blends[i - 1]; };
    if (T < c.T_low) { seg = -1; return; }
    if (T > c.T_high) { seg = -2; return; }
    if (T < lo(1)) { seg = 0; return; }
    if (T > hi(nb - 2)) { seg = c.nseg - 1; return; }
    for (int i = 1; i < nb - 1; ++i) {
        seg = i - 1;
        if (T >= lo(i) && T <= hi(i)) { blend = true; return; }
        seg = i;
        if (i < c.nseg - 1 && T > hi(i) && T < lo(i + 1)) return;
    }
}

// The regions of the summed curves (MixTable): the line cut at every species' range edges, each
// piece's coefficients from what the species' curves are at its midpoint.
static void build_mix_table(ChemDev& cd) {
    MixTable& t = cd.mix;
    std::vector<double> cut;
    for (int i = 0; i < cd.nsp; ++i) {
        const CEADev& c = cd.cea[i];
        cut.push_back(c.T_low);
        cut.push_back(c.T_high);
        for (int k = 0; k < c.nseg - 1; ++k) {
            cut.push_back(c.T_breaks[k + 1] - 0.5 * c.T_blends[k]);
            cut.push_back(c.T_breaks[k + 1] + 0.5 * c.T_blends[k]);
        }
    }
    std::sort(cut.begin(), cut.end());
    cut.erase(std::unique(cut.begin(), cut.end()), cut.end());
    const double inf = std::numeric_limits<double>::infinity();
    t.nreg = (int)cut.size() + 1;
    for (int r = 0; r < t.nreg; ++r) {
        t.lo[r] = (r == 0) ? -inf : cut[r - 1];
        t.hi[r] = (r == t.nreg - 1) ? inf : cut[r];
        const double mid = (r == 0) ? std::nextafter(t.hi[r], -inf)
                         : (r == t.nreg - 1) ? std::nextafter(t.lo[r], inf) : 0.5 * (t.lo[r] + t.hi[r]);
        // the region's lower edge (z >= 0); the forms need T0 > 0
        const double T0 = std::max((r == 0) ? mid : t.lo[r], 1.0);
        t.T0[r] = T0;
        t.iT0[r] = 1.0 / T0;
        t.flat[r] = 1;
        for (int i = 0; i < cd.nsp; ++i) {
            const CEADev& c = cd.cea[i];
            int seg = 0;
            bool blend = false;
            curve_at(c, mid, seg, blend);
            double* a = t.c[r][0][i];
            if (seg < 0) {
                a[2] = ((seg == -1) ? c.Cp_low : c.Cp_high) / c.R;
                a[7] = (seg == -1) ? (c.h_low - c.Cp_low * (c.T_low - T0)) / c.R
                                   : (c.h_high + c.Cp_high * (T0 - c.T_high)) / c.R;
                continue;
            }
            expand_segment(c.coeffs[seg], T0, a);
            if (!blend) continue;
            // (1 - wB) A + wB B, wB = (T - w0) / width = w + z / width
            double B[8];
            expand_segment(c.coeffs[seg + 1], T0, B);
            const double width = c.T_blends[seg], w = (T0 - (c.T_breaks[seg + 1] - 0.5 * width)) / width;
            for (int j = 0; j < 8; ++j) {
                const double A = a[j];
                a[j] = (1.0 - w) * A + w * B[j];
                t.c[r][1][i][j] = (B[j] - A) / width;
            }
            t.flat[r] = 0;
        }
    }
}

// Gas record -> the gas part of the device table (molecular masses, species gas constants,
// CEA curves with their end-point values), with the checks of the reference's readers.
void build_tpg_gas(const gdtk_tpg_gas& g, ChemDev& cd) {
    std::memset(&cd, 0, sizeof(cd));
    if (g.nsp < 1 || g.nsp > CH_MAX_SP) throw Error(GDTK_ERR_ARG, "nsp must be 1..8");
    cd.nsp = g.nsp;
    for (int i = 0; i < g.nsp; ++i) {
        if (!(g.M[i] > 0.0)) throw Error(GDTK_ERR_ARG, "molecular mass must be positive");
        cd.M[i] = g.M[i];
        cd.R[i] = CH_R_UNIVERSAL / g.M[i];  // therm_perf_gas.d:62-64
        CEADev& c = cd.cea[i];
        const int ns = g.nseg[i];
        if (ns < 2 || ns > 3) throw Error(GDTK_ERR_ARG, "CEA curves need 2 or 3 segments");
        c.nseg = ns;
        for (int k = 0; k <= ns; ++k) c.T_breaks[k] = g.T_breaks[i][k];
        for (int k = 0; k < ns - 1; ++k) c.T_blends[k] = g.T_blends[i][k];
        for (int s = 0; s < ns; ++s)
            for (int j = 0; j < 9; ++j) c.coeffs[s][j] = g.coeffs[i][s][j];
        for (int k = 0; k < ns; ++k)
            if (!(c.T_breaks[k] < c.T_breaks[k + 1])) throw Error(GDTK_ERR_ARG, "CEA breaks must increase");
        // cea_thermo_curves.d:45-54
        c.R = cd.R[i];
        c.T_low = c.T_breaks[0];
        c.T_high = c.T_breaks[ns];
        c.Cp_low = cea_Cp(c, c.T_low);
        c.Cp_high = cea_Cp(c, c.T_high);
        c.h_low = cea_h(c, c.T_low);
        c.h_high = cea_h(c, c.T_high);
        c.s_low = cea_s(c, c.T_low);
        c.s_high = cea_s(c, c.T_high);
    }
    build_mix_table(cd);
}

// Gas and mechanism records -> the device table, with the checks the reference's input
// readers make (species indices, segment counts) and the options the kernels implement.
void build_chemdev(const gdtk_tpg_gas& g, const gdtk_mechanism& m, ChemDev& cd, bool two_temperature) {
    build_tpg_gas(g, cd);
    if (m.nr < 0 || m.nr > CH_MAX_R) throw Error(GDTK_ERR_ARG, "nr must be 0..32");
    cd.nr = m.nr;
    for (int ir = 0; ir < m.nr; ++ir) {
        const gdtk_reaction& r = m.r[ir];
        ReacDev& d = cd.r[ir];
        if (r.nreac < 1 || r.nreac > 3 || r.nprod < 1 || r.nprod > 3 || r.neff < 0 || r.neff > CH_MAX_SP)
            throw Error(GDTK_ERR_ARG, "reaction participant counts out of range");
        d.collider = r.collider ? 1 : 0;
        d.nreac = r.nreac;
        d.nprod = r.nprod;
        for (int k = 0; k < r.nreac; ++k) {
            if (r.reac_sp[k] < 0 || r.reac_sp[k] >= g.nsp || r.reac_nu[k] < 1 || r.reac_nu[k] > 3)
                throw Error(GDTK_ERR_ARG, "bad reactant (species index, or coefficient outside 1..3)");
            d.reac_sp[k] = r.reac_sp[k];
            d.reac_nu[k] = r.reac_nu[k];
        }
        for (int k = 0; k < r.nprod; ++k) {
            if (r.prod_sp[k] < 0 || r.prod_sp[k] >= g.nsp || r.prod_nu[k] < 1 || r.prod_nu[k] > 3)
                throw Error(GDTK_ERR_ARG, "bad product (species index, or coefficient outside 1..3)");
            d.prod_sp[k] = r.prod_sp[k];
            d.prod_nu[k] = r.prod_nu[k];
        }
        d.neff = d.collider ? r.neff : 0;
        for (int k = 0; k < d.neff; ++k) {
            if (r.eff_sp[k] < 0 || r.eff_sp[k] >= g.nsp) throw Error(GDTK_ERR_ARG, "bad efficiency species");
            d.eff_sp[k] = r.eff_sp[k];
            d.eff[k] = r.eff[k];
        }
        d.f_from_eq = r.f_from_eq ? 1 : 0;
        d.b_from_eq = r.b_from_eq ? 1 : 0;
        if (d.f_from_eq && d.b_from_eq) throw Error(GDTK_ERR_ARG, "both rate constants from K_c");
        d.fA = r.fA; d.fn = r.fn; d.fC = r.fC;
        d.bA = r.bA; d.bn = r.bn; d.bC = r.bC;
        if ((r.f_park || r.b_park) && !two_temperature)
            throw Error(GDTK_ERR_UNSUPPORTED, "Park two-temperature rate constants need the two-temperature reactor");
        d.f_park = r.f_park ? 1 : 0;
        d.b_park = r.b_park ? 1 : 0;
        d.f_s = r.f_s;
        d.b_s = r.b_s;
        // Dense form when every list is in strictly ascending species order.
        auto ascending = [](const int* sp, int k) {
            for (int q = 1; q < k; ++q)
                if (!(sp[q - 1] < sp[q])) return false;
            return true;
        };
        d.sorted = ascending(r.reac_sp, r.nreac) && ascending(r.prod_sp, r.nprod) &&
                   (!d.collider || ascending(r.eff_sp, r.neff));
        if (d.sorted) {
            for (int k = 0; k < r.nreac; ++k) d.reac_d[r.reac_sp[k]] = r.reac_nu[k];
            for (int k = 0; k < r.nprod; ++k) d.prod_d[r.prod_sp[k]] = r.prod_nu[k];
            for (int k = 0; k < d.neff; ++k) {
                d.eff_set |= 1u << r.eff_sp[k];
                d.eff_d[r.eff_sp[k]] = r.eff[k];
            }
        }
        // reaction.d:100-143: participants and net coefficients (first listing of a species)
        for (int s = 0; s < g.nsp; ++s) {
            int nu1 = 0, nu2 = 0, in = 0;
            for (int k = 0; k < r.nreac; ++k)
                if (r.reac_sp[k] == s) { nu1 = r.reac_nu[k]; in = 1; break; }
            for (int k = 0; k < r.nprod; ++k)
                if (r.prod_sp[k] == s) { nu2 = r.prod_nu[k]; in = 1; break; }
            d.nu[s] = nu2 - nu1;
            d.part[s] = in;
        }
    }
    // The rows of the branch-free rate walk, when every reaction has its dense form.
    cd.all_sorted = 1;
    for (int ir = 0; ir < m.nr; ++ir) cd.all_sorted &= cd.r[ir].sorted;
    for (int ir = 0; ir < CH_MAX_R; ++ir) cd.rr[ir] = RateRow{};
    if (cd.all_sorted) {
        for (int ir = 0; ir < m.nr; ++ir) {
            const ReacDev& d = cd.r[ir];
            RateRow& w = cd.rr[ir];
            w.flags = d.collider ? 1 : 0;
            for (int s = 0; s < g.nsp; ++s) {
                const bool listed = d.collider && ((d.eff_set >> s) & 1u);
                w.eff[s] = listed ? d.eff_d[s] : 0.0;
                w.code[s] = d.reac_d[s] | (d.prod_d[s] << 2) | ((d.nu[s] & 15) << 4) | (listed ? 256 : 0);
            }
        }
    }
    cd.walk = mechanism_walk(cd);
    if (!(m.T_lower < m.T_upper)) throw Error(GDTK_ERR_ARG, "tempLimits lower must be below upper");
    cd.T_lower = m.T_lower;
    cd.T_upper = m.T_upper;
    if (m.method != GDTK_ODE_ALPHA_QSS && m.method != GDTK_ODE_RKF) throw Error(GDTK_ERR_ARG, "bad ODE method");
    if (m.tightTempCoupling && m.method != GDTK_ODE_ALPHA_QSS && !two_temperature)
        throw Error(GDTK_ERR_UNSUPPORTED, "tightTempCoupling is implemented for the alpha-QSS step only");
    if (m.maxIters < 1 || m.maxSubcycles < 1 || m.maxAttempts < 1) throw Error(GDTK_ERR_ARG, "bad step control");
    cd.method = m.method;
    cd.eps1 = m.eps1;
    cd.eps2 = m.eps2;
    cd.delta = m.delta;
    cd.maxIters = m.maxIters;
    cd.errTol = m.errTol;
    cd.maxSubcycles = m.maxSubcycles;
    cd.maxAttempts = m.maxAttempts;
    cd.T_frozen = m.T_frozen;
    cd.tight = m.tightTempCoupling ? 1 : 0;
}

template <class T>
static void h2d(DevArr<T>& d, const T* h, size_t count, hipStream_t s) {
    d.reserve(count);
    if (count) HIPCHK(hipMemcpyAsync(d.p, h, count * sizeof(T), hipMemcpyHostToDevice, s));
}
template <class T>
static void d2h(T* h, const DevArr<T>& d, size_t count, hipStream_t s) {
    if (count) HIPCHK(hipMemcpyAsync(h, d.p, count * sizeof(T), hipMemcpyDeviceToHost, s));
}

}  // namespace gdtk

using namespace gdtk;

extern "C" {

int gdtk_hip_chem_create(const gdtk_tpg_gas* gas, const gdtk_mechanism* mech, int* chem) {
    return guarded([&] {
        if (!gas || !mech || !chem) throw Error(GDTK_ERR_ARG, "null argument");
        int ndev = 0;
        HIPCHK(hipGetDeviceCount(&ndev));
        if (ndev < 1) throw Error(GDTK_ERR_HIP, "no HIP device");
        auto c = std::make_unique<Chem>();
        build_chemdev(*gas, *mech, c->host, false);
        c->nsp = c->host.nsp;
        c->nr = c->host.nr;
        if (!chem_supported(c->nsp, c->nr)) throw Error(GDTK_ERR_UNSUPPORTED, "mechanism size not supported");
        int devid = 0;
        HIPCHK(hipGetDevice(&devid));
        HIPCHK(hipDeviceGetAttribute(&c->num_cu, hipDeviceAttributeMultiprocessorCount, devid));
        HIPCHK(hipMalloc(&c->dev, sizeof(ChemDev)));
        HIPCHK(hipMemcpy(c->dev, &c->host, sizeof(ChemDev), hipMemcpyHostToDevice));
        HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
        for (auto& e : c->ev) HIPCHK(hipEventCreate(&e));
        std::lock_guard<std::mutex> lk(g_chem_mu);
        g_chems.push_back(std::move(c));
        *chem = (int)g_chems.size() - 1;
        return GDTK_OK;
    });
}

int gdtk_hip_chem_destroy(int chem) {
    return guarded([&] {
        std::lock_guard<std::mutex> lk(g_chem_mu);
        if (chem < 0 || chem >= (int)g_chems.size() || !g_chems[chem]) throw Error(GDTK_ERR_ARG, "bad chemistry handle");
        HIPCHK(hipStreamSynchronize(g_chems[chem]->stream));
        g_chems[chem].reset();
        return GDTK_OK;
    });
}

int gdtk_hip_chem_step(int chem, int n, const double* rho, double* T, double* u, double* p, double* massf,
                       double* dt_chem, double dt, int* status, double* stats) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        if (n < 0) throw Error(GDTK_ERR_ARG, "negative cell count");
        if (n > 0 && (!rho || !T || !u || !p || !massf || !dt_chem || !status)) throw Error(GDTK_ERR_ARG, "null array");
        hipStream_t s = c.stream;
        const size_t N = (size_t)n, NS = (size_t)c.nsp * N;
        h2d(c.s_rho, rho, N, s);
        h2d(c.s_T, (const double*)T, N, s);
        h2d(c.s_u, (const double*)u, N, s);
        h2d(c.s_p, (const double*)p, N, s);
        h2d(c.s_massf, (const double*)massf, NS, s);
        h2d(c.s_dtc, (const double*)dt_chem, N, s);
        c.s_status.reserve(N);
        c.step_device(n, dt, c.s_rho.p, c.s_T.p, c.s_u.p, c.s_p.p, c.s_massf.p, c.s_dtc.p, c.s_T.p, c.s_u.p, c.s_p.p,
                      c.s_massf.p, c.s_dtc.p, c.s_status.p, s);
        d2h(T, c.s_T, N, s);
        d2h(u, c.s_u, N, s);
        d2h(p, c.s_p, N, s);
        d2h(massf, c.s_massf, NS, s);
        d2h(dt_chem, c.s_dtc, N, s);
        d2h(status, c.s_status, N, s);
        HIPCHK(hipStreamSynchronize(s));
        if (stats) {
            double v[8];
            c.read_stats(v, 8);
            stats[0] = v[0];
            stats[1] = v[1];
            stats[2] = v[2];
            stats[3] = v[4] + v[5] + v[6];
        }
        int failed = 0;
        for (int i = 0; i < n; ++i) failed += (status[i] != 0);
        return failed;
    });
}

int gdtk_hip_chem_step_device(int chem, int n, const double* rho, const double* T, const double* u, const double* p,
                              const double* massf, const double* dt_chem, double dt, double* T_out, double* u_out,
                              double* p_out, double* massf_out, double* dt_chem_out, int* status, void* stream) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        if (n < 0) throw Error(GDTK_ERR_ARG, "negative cell count");
        if (n > 0 && (!rho || !T || !u || !p || !massf || !dt_chem || !T_out || !u_out || !p_out || !massf_out ||
                      !dt_chem_out || !status))
            throw Error(GDTK_ERR_ARG, "null array");
        hipStream_t s = static_cast<hipStream_t>(stream);  // NULL: the default stream
        c.step_device(n, dt, rho, T, u, p, massf, dt_chem, T_out, u_out, p_out, massf_out, dt_chem_out, status, s);
        return GDTK_OK;
    });
}

int gdtk_hip_chem_stats(int chem, double* stats, int nstats) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        if (!stats || nstats < 1) throw Error(GDTK_ERR_ARG, "null stats");
        return c.read_stats(stats, nstats);
    });
}

int gdtk_hip_chem_substeps(int chem, int n, int* substeps) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        if (n != c.last_n || !substeps) throw Error(GDTK_ERR_ARG, "n must be the cell count of the last step");
        HIPCHK(hipEventSynchronize(c.ev[3]));
        // Cells that were not integrated (frozen, invalid) report 0 substeps.
        std::vector<int> f((size_t)n);
        HIPCHK(hipMemcpy(f.data(), c.last_w.flag, (size_t)n * sizeof(int), hipMemcpyDeviceToHost));
        HIPCHK(hipMemcpy(substeps, c.last_w.nsub, (size_t)n * sizeof(int), hipMemcpyDeviceToHost));
        for (int i = 0; i < n; ++i)
            if (f[i] != CF_INTEGRATE && f[i] != CF_HEAVY) substeps[i] = 0;
        return GDTK_OK;
    });
}

int gdtk_hip_chem_set_tuning(int chem, int key, int value) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        switch (key) {
        case GDTK_CHEM_TUNE_PERSISTENT: c.tuning.persistent = (value < 0) ? -1 : (value ? 1 : 0); break;
        case GDTK_CHEM_TUNE_CHUNK:
            if (value < 1 || value > 4096) throw Error(GDTK_ERR_ARG, "chunk must be 1..4096");
            c.tuning.chunk = value;
            break;
        case GDTK_CHEM_TUNE_REFILL:
            if (value < 1 || value > 4096) throw Error(GDTK_ERR_ARG, "refill period must be 1..4096");
            c.tuning.refill_period = value;
            break;
        case GDTK_CHEM_TUNE_BLOCKS_PER_CU:
            if (value < 0 || value > 64) throw Error(GDTK_ERR_ARG, "blocks per CU must be 0..64");
            c.tuning.blocks_per_cu = value;
            break;
        case GDTK_CHEM_TUNE_HEAVY_RATIO:
            if (value < 0 || value > 1000000) throw Error(GDTK_ERR_ARG, "heavy ratio must be 0..1e6");
            c.tuning.heavy_ratio = value;
            break;
        default: throw Error(GDTK_ERR_ARG, "unknown tuning key");
        }
        return GDTK_OK;
    });
}

int gdtk_hip_chem_autotune(int chem, int n, const double* rho, const double* T, const double* u, const double* p,
                           const double* massf, const double* dt_chem, double dt, double* out, int nout) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        if (n <= 0 || !rho || !T || !u || !p || !massf || !dt_chem) throw Error(GDTK_ERR_ARG, "bad arguments");
        const size_t N = (size_t)n, NS = (size_t)c.nsp * N;
        // Scratch outputs: the inputs are left untouched.
        DevArr<double> To, uo, po, mo, dto;
        DevArr<int> so;
        To.alloc(N); uo.alloc(N); po.alloc(N); mo.alloc(NS); dto.alloc(N); so.alloc(N);
        struct Cand { int persistent, chunk, refill, bpc; };
        std::vector<Cand> cands = {{0, 64, 1, 0}};
        for (int chunk : {32, 64, 256})
            for (int refill : {1, 4, 16}) cands.push_back({1, chunk, refill, 0});
        ChemTuning saved = c.tuning;
        double best = 1e300;
        ChemTuning best_t = saved;
        int k = 0;
        hipStream_t s = c.stream;
        for (const Cand& cd : cands) {
            c.tuning = ChemTuning{cd.persistent, cd.chunk, cd.refill, cd.bpc, saved.heavy_ratio};
            c.step_device(n, dt, rho, T, u, p, massf, dt_chem, To.p, uo.p, po.p, mo.p, dto.p, so.p, s);
            double v[8];
            c.read_stats(v, 8);
            const double ms = v[4] + v[5] + v[6];
            if (out && 5 * (k + 1) <= nout) {
                out[5 * k + 0] = cd.persistent;
                out[5 * k + 1] = cd.chunk;
                out[5 * k + 2] = cd.refill;
                out[5 * k + 3] = cd.bpc;
                out[5 * k + 4] = ms;
            }
            ++k;
            if (ms < best) {
                best = ms;
                best_t = c.tuning;
            }
        }
        c.tuning = best_t;
        HIPCHK(hipStreamSynchronize(s));
        return k;
    });
}

int gdtk_hip_tpg_update(int chem, int mode, int n, double* rho, double* p, double* T, double* u, double* a,
                        const double* massf) {
    return guarded([&] {
        Chem& c = get_chem(chem);
        if (mode < 0 || mode > 2) throw Error(GDTK_ERR_ARG, "mode must be 0 (pT), 1 (rhou) or 2 (rhoT)");
        if (n < 0) throw Error(GDTK_ERR_ARG, "negative cell count");
        if (n > 0 && (!rho || !p || !T || !u || !a || !massf)) throw Error(GDTK_ERR_ARG, "null array");
        hipStream_t s = c.stream;
        const size_t N = (size_t)n, NS = (size_t)c.nsp * N;
        h2d(c.s_rho, (const double*)rho, N, s);
        h2d(c.s_p, (const double*)p, N, s);
        h2d(c.s_T, (const double*)T, N, s);
        h2d(c.s_u, (const double*)u, N, s);
        h2d(c.s_a, (const double*)a, N, s);
        h2d(c.s_massf, massf, NS, s);
        c.s_status.reserve(N);
        HIPCHK(launch_tpg_update(c.dev, c.nsp, mode, n, c.s_rho.p, c.s_p.p, c.s_T.p, c.s_u.p, c.s_a.p, c.s_massf.p,
                                 c.s_status.p, s));
        d2h(rho, c.s_rho, N, s);
        d2h(p, c.s_p, N, s);
        d2h(T, c.s_T, N, s);
        d2h(u, c.s_u, N, s);
        d2h(a, c.s_a, N, s);
        std::vector<int> st(N);
        if (N) HIPCHK(hipMemcpyAsync(st.data(), c.s_status.p, N * sizeof(int), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        int failed = 0;
        for (int v : st) failed += (v != 0);
        return failed;
    });
}

}  // extern "C"
