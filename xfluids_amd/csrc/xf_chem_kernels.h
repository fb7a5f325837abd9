// Stiff finite-rate chemistry on the device: constant-volume production and
// loss rates and the CHEMEQ2 quasi-steady-state integrator, temperature
// carried as y[0].
//
// Reference: evalcore (q/p form) src/solver_Reaction/ProductionRates.h:117-176,
// evalcv :459-479, xfrsign/Alpha :227-244, Chemeq2 :488-638,
// ChemeODEQ2SolverKernel1 src/solver_Reaction/Reaction_kernels.hpp:46-73.
//
// Restructured without changing any result bit:
//  * get_Gibson(T, n) and log(p/p_atm), log(T) do not depend on the reaction
//    and are evaluated once per rate evaluation instead of NR*NS times;
//  * terms with a zero stoichiometric coefficient or third-body efficiency
//    add +0 (or multiply by pown(x, 0) = 1) in the reference and are skipped;
//  * rates are accumulated into q, d reaction by reaction; every species'
//    sum still runs over reactions in increasing order;
//  * the predictor loop writes y directly and the corrector loop is fused
//    with the convergence loop (y1 is the predicted y read before overwrite).
// Safety bound: at most CHEM_MAXSUB predictor passes per cell; a cell that
// reaches it raises XF_ERR_CHEM.  The reference loop is unbounded.
#pragma once
#include "xf_thermo.h"
#include "gen/xf_mech_gen.h"
#include <utility>

namespace xf {

constexpr int CHEM_MAXSUB = 200000;
// the bits a chemistry launch may set, which it therefore does not test: the pass bound,
// and the NaN check of the cells it has written (a NaN of an earlier launch has been
// latched by the Reaction's UpdateStates, which runs in between)
constexpr int CHEM_BITS = EBIT_CHEM | EBIT_NAN;

__device__ __forceinline__ double pown_i(double x, int n)
{
    // the products of the loop below, written out for the usual orders
    if (n == 1) return x;
    if (n == 2) return x * x;
    if (n == 3) return (x * x) * x;
    if (n == 0) return 1.0;
    double r = x;
    for (int k = 1; k < n; k++) r *= x;
    return r;
}

// What one reaction reads besides its record: T, the shared reciprocal of T
// and whether it qualifies for the corrected quotient, the logarithms
struct RxnCtx {
    double m_tmp, rT, logT, logP, logStandConc;
    bool t_ok;
};

// One reaction's contribution to the production and loss rates (evalcore,
// ProductionRates.h:117-176), from its record R and third-body efficiencies
// eff(s) in the device tables: the general form, whose values rxn_fast (a compiled
// mechanism, a lane per cell) and wave_rates (a cell per wave) reproduce bit for bit
// within their ranges.
// Species loops run over compile-time n and test the record's masks, which
// skips exactly the zero-coefficient terms (each adds +0 or multiplies by 1 in
// the reference, so skipping changes no bit).
template <int NS, class Eff>
__device__ __forceinline__ void rxn_rates(const DevRxn R, Eff eff, const RxnCtx &c, const double *gk,
                                          const double *m_cm, double &Kf_out, double &Kck_out)
{
    const double A = R.A, B = R.B, EaR = R.EaR;
    const unsigned md = R.md, mt = R.mt, mf = R.mf, mb = R.mb;
    const unsigned long long pd = R.pd, pf = R.pf, pb = R.pb;
    const int tind = R.third_ind;
    // EaR / T from the shared reciprocal: Markstein's corrected quotient
    // fma(fma(-T, q0, a), y, q0), q0 = a y, y = RN(1/T), is the correctly
    // rounded a / T while a, T lie in [2^-500, 2^500] (the remainder is exact
    // and nothing underflows); a = 0 keeps q0, the signed zero of a / T
    double ET;
    const double aE = fabs(EaR);
    if (c.t_ok && (EaR == 0.0 || (aE >= 0x1p-500 && aE <= 0x1p500))) {
        const double q0 = EaR * c.rT;
        ET = EaR == 0.0 ? q0 : fma(fma(-c.m_tmp, q0, EaR), c.rT, q0);
    } else {
        ET = EaR / c.m_tmp;
    }
    double Kf = A * dexp(B * c.logT - ET);
    double DeltaGibbs = 0.0;
    int m_dn = 0;
#pragma unroll
    for (int n = 0; n < NS; n++) {
        if ((md >> n) & 1u) {
            const int nu = (int)((pd >> (4 * n)) & 15ull) - 8;
            DeltaGibbs += nu * (c.logP - gk[n]);
            m_dn += nu;
        }
    }
    double Kck = dmin(dexp(DeltaGibbs - m_dn * c.logStandConc), 1.0E+40);
    double tb = 1.0;
    if (1 == tind) {
        tb = 0.0;
        // every efficiency of the row first (one burst of scalar loads when
        // they come from the tables)
        double e[NS];
#pragma unroll
        for (int it = 0; it < NS; it++) e[it] = eff(it);
#pragma unroll
        for (int it = 0; it < NS; it++)
            if ((mt >> it) & 1u) tb += e[it] * m_cm[it];
    }
    Kf *= tb;
    Kck *= Kf;
#pragma unroll
    for (int it = 0; it < NS; it++)
        if ((mf >> it) & 1u) Kf *= pown_i(m_cm[it], (int)((pf >> (4 * it)) & 15ull));
#pragma unroll
    for (int it = 0; it < NS; it++)
        if ((mb >> it) & 1u) Kck *= pown_i(m_cm[it], (int)((pb >> (4 * it)) & 15ull));
    Kf_out = Kf, Kck_out = Kck;
}

// the reaction's terms of the production and loss rates of every species
template <int NS>
__device__ __forceinline__ void rxn_accum(unsigned mf, unsigned mb, unsigned long long pf, unsigned long long pb,
                                          double Kf, double Kck, double *qi, double *pi)
{
#pragma unroll
    for (int n = 0; n < NS; n++) {
        if (((mf | mb) >> n) & 1u) {
            const int nf = (int)((pf >> (4 * n)) & 15ull), nb = (int)((pb >> (4 * n)) & 15ull);
            qi[n] += nb * Kf + nf * Kck;
            pi[n] += nf * Kf + nb * Kck;
        }
    }
}

template <int NS, class Eff>
__device__ __forceinline__ void rxn_step(const DevRxn R, Eff eff, const RxnCtx &c, const double *gk,
                                         const double *m_cm, double *qi, double *pi)
{
    double Kf, Kck;
    rxn_rates<NS>(R, eff, c, gk, m_cm, Kf, Kck);
    rxn_accum<NS>(R.mf, R.mb, R.pf, R.pb, Kf, Kck, qi, pi);
}

// The rate evaluation is bound by FP64 issue at two waves per SIMD (one lane per
// cell, ~4250 instructions per pass and cell before, 97 KB of code against the 64
// KB instruction cache): the fast path below drops what a compiled mechanism and
// an ordinary state make exact no-ops, and needs no scratch memory.  k_chem on a
// 128^3 mixing layer past its start-up went from 1417 to 997 us, k_chem_queue on a
// 256^2 channel from 149 to 106 us.
//
// Reaction r of compiled mechanism K on the fast path of evalcv_dev: rxn_step's
// values with every test on the record resolved at compile time.  lg = log p - g
// per species.  Terms with a zero factor are left out (0 * K adds a zero while K
// is finite; the caller checks that at the end), the first term of a sum that
// starts at 0 is taken as it is, and the two exponentials run together.
template <int NS, int K, int r>
__device__ __forceinline__ void rxn_fast(const RxnCtx &c, const double *lg, const double *m_cm, double *qi,
                                         double *pi)
{
    constexpr DevRxn R = MechSpec<K>::rx(r);
    constexpr double aE = R.EaR < 0.0 ? -R.EaR : R.EaR;
    double arg[2];
    if constexpr (R.EaR != 0.0) {
        double ET;
        if constexpr (aE >= 0x1p-500 && aE <= 0x1p500) ET = dquot(R.EaR, c.m_tmp, c.rT);
        else ET = R.EaR / c.m_tmp;
        arg[0] = R.B != 0.0 ? R.B * c.logT - ET : -ET;
    } else {
        arg[0] = R.B * c.logT;
    }
    double DG = 0.0;
    int m_dn = 0;
    bool first = true;
#pragma unroll
    for (int n = 0; n < NS; n++) {
        if ((R.md >> n) & 1u) {
            const int nu = (int)((R.pd >> (4 * n)) & 15ull) - 8;
            DG = first ? nu * lg[n] : DG + nu * lg[n];
            first = false;
            m_dn += nu;
        }
    }
    arg[1] = m_dn != 0 ? DG - m_dn * c.logStandConc : DG;
    double Kf, Kck;
    if constexpr (R.B == 0.0 && R.EaR == 0.0) {
        Kf = R.A; // A exp(0)
        Kck = dexp(arg[1]);
    } else {
        double e[2];
        dexp_n<2>(arg, e);
        Kf = R.A * e[0], Kck = e[1];
    }
    Kck = dmin(Kck, 1.0E+40);
    if constexpr (R.third_ind == 1) {
        double tb = 0.0;
        bool one = true;
#pragma unroll
        for (int it = 0; it < NS; it++)
            if ((R.mt >> it) & 1u) {
                const double x = MechSpec<K>::eff(r, it) * m_cm[it];
                tb = one ? x : tb + x;
                one = false;
            }
        Kf *= tb;
    }
    Kck *= Kf;
#pragma unroll
    for (int it = 0; it < NS; it++)
        if ((R.mf >> it) & 1u) Kf *= pown_i(m_cm[it], (int)((R.pf >> (4 * it)) & 15ull));
#pragma unroll
    for (int it = 0; it < NS; it++)
        if ((R.mb >> it) & 1u) Kck *= pown_i(m_cm[it], (int)((R.pb >> (4 * it)) & 15ull));
#pragma unroll
    for (int n = 0; n < NS; n++) {
        if (((R.mf | R.mb) >> n) & 1u) {
            const int nf = (int)((R.pf >> (4 * n)) & 15ull), nb = (int)((R.pb >> (4 * n)) & 15ull);
            qi[n] += nf == 0 ? nb * Kf : (nb == 0 ? nf * Kck : nb * Kf + nf * Kck);
            pi[n] += nb == 0 ? nf * Kf : (nf == 0 ? nb * Kck : nf * Kf + nb * Kck);
        }
    }
}
template <int NS, int K, int... r>
__device__ __forceinline__ void rxns_fast(std::integer_sequence<int, r...>, const RxnCtx &c, const double *lg,
                                          const double *m_cm, double *qi, double *pi)
{
    (rxn_fast<NS, K, r>(c, lg, m_cm, qi, pi), ...);
}

// evalcv from the species sums on: the temperature's q and d from the species'
// rates; e_k = (h1 - T) R_k
template <int NS>
__device__ __forceinline__ void evalcv_energy(const DevThermo *__restrict__ th, const double *h1, double m_tmp,
                                              double _dens, double cv, double *q, double *d)
{
    double *qi = q + 1, *pi = d + 1;
    double q0 = 0.0, d0 = 0.0;
    cdouble *Wk = as_const(th->Wi), *Rk = as_const(th->Ri);
#pragma unroll
    for (int n = 0; n < NS; n++) {
        const double wd = Wk[n] * _dens;
        qi[n] *= wd;
        pi[n] *= wd;
        const double ei = (h1[n] - m_tmp) * Rk[n];
        q0 -= qi[n] * ei, d0 -= pi[n] * ei;
    }
    const double _Cv = 1.0 / cv;
    q[0] = q0 * _Cv, d[0] = d0 * _Cv;
}

// What evalcv reads of the species at y[0] = T, for waves whose every lane has T and
// pressure where the fast fits and quotients are exact: enthalpies and Gibbs energies g
// (Ri = 1; LG: log p - g in their place), the mixture's Cv and the reactions' context;
// false otherwise.
template <int NS, bool LG>
__device__ __forceinline__ bool evalcv_species(const DevThermo *__restrict__ th, const double *y, double m_p,
                                               double *h1, double *gk, double &cv, RxnCtx &c)
{
    const double m_tmp = y[0];
    const double logP = dlog_pos(m_p * (1.0 / 101325.0));
    // mix_cv: the species' part inside, with the range's coefficients
    double _W = 0.0;
    cv = 0.0;
    cdouble *Rk = as_const(th->Ri), *iWk = as_const(th->_Wi);
    auto species = [&](auto fam) {
        constexpr bool NASA = decltype(fam)::value;
        const bool p_ok = m_p >= 0x1p-300 && m_p <= 0x1p300;
        const double top = fast_top(th);
        auto values = [&](cdouble *cf, auto t) {
            c.logT = t.lT, c.rT = t.iT;
            if (t.cold) c.logT = dlog_pos(m_tmp), c.rT = ddiv_core(1.0, m_tmp);
#pragma unroll
            for (int n = 0; n < NS; n++) {
                h1[n] = h_fast<NASA>(cf + FITC * n, t.T, t.iT, t.lT, 1.0);
                if (t.cold) h1[n] = t.below(h1[n], cp_fast<NASA>(cf + FITC * n, t.T, t.iT, 1.0));
                double g = 0.0;
                g += s_fast<NASA>(cf + FITC * n, t.T, t.iT, t.lT);
                g += dquot(-h1[n], m_tmp, c.rT);
                gk[n] = LG ? logP - g : g;
                cv += y[1 + n] * cp_fast<NASA>(cf + FITC * n, t.T, t.iT, Rk[n]);
            }
        };
        // the usual waves by one vote, and the colder ones' copy behind it: with a vote of
        // its own for each condition a step of a 256^2 channel, one lane per cell, takes
        // 505 us instead of 497
        if (__builtin_expect(__all(m_tmp >= 200.0 && m_tmp <= top && p_ok), 1)) {
            fast_ranges<NASA, false>(th, m_tmp, true, values);
            return true;
        }
        if (!__all(m_tmp >= 0x1p-100 && m_tmp <= top && p_ok)) return false;
        fast_ranges<NASA, true>(th, m_tmp, true, values);
        return true;
    };
    if (!(th->thermo ? species(std::true_type{}) : species(std::false_type{}))) return false;
#pragma unroll
    for (int n = 0; n < NS; n++) _W += y[1 + n] * iWk[n];
    cv -= Ru * _W;
    c.m_tmp = m_tmp, c.logP = logP, c.t_ok = true;
    c.logStandConc = dlog_pos(ddiv_core(m_p, R0 * m_tmp));
    return true;
}

// evalcv on the fast path with compiled mechanism SPEC.  Returns false, with nothing
// of use in q and d, where evalcv_species does or when a rate is not
// finite (a non-finite Kf or Kck reaches some species' sum, and with it the
// temperature's).
template <int NS, int SPEC>
__device__ __forceinline__ bool evalcv_fast(const DevThermo *__restrict__ th, const double *y, double *q, double *d,
                                            double m_dens, double _dens, double m_p)
{
    double h1[NS], lg[NS], m_cm[NS], cv;
    RxnCtx c;
    cdouble *iWk = as_const(th->_Wi);
    if (!evalcv_species<NS, true>(th, y, m_p, h1, lg, cv, c)) return false;
#pragma unroll
    for (int n = 0; n < NS; n++) m_cm[n] = y[1 + n] * iWk[n] * m_dens * 1.0E-3;
    double *qi = q + 1, *pi = d + 1;
#pragma unroll
    for (int n = 0; n < NS; n++) qi[n] = 0.0, pi[n] = 0.0;
    rxns_fast<NS, SPEC>(std::make_integer_sequence<int, MechSpec<SPEC>::NR>{}, c, lg, m_cm, qi, pi);
    evalcv_energy<NS>(th, h1, y[0], _dens, cv, q, d);
    return __all(fabs(q[0]) < __longlong_as_double(0x7ff0000000000000LL) &&
                 fabs(d[0]) < __longlong_as_double(0x7ff0000000000000LL));
}

// evalcv (y[0] = T): q, d of length NS + 1.  SPEC >= 0: the reactions of
// compiled mechanism SPEC, unrolled with their records as constants (the
// caller has checked that the device tables hold exactly those records), on
// the fast path; the loop over the records in the device tables for SPEC < 0
// and wherever the fast path does not hold, with the same bits.  The loop's species
// values come from evalcv_species too: with each lane's own range and vector loads of
// the coefficients a launch on 128^3 cells took 52 ms (13 passes a cell), now 45.
template <int NS, int SPEC = -1>
__device__ __forceinline__ void evalcv_dev(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc,
                                           const double *y, double *q, double *d, double m_dens, double m_p)
{
    const double m_tmp = y[0];
    const double _dens = 1.0 / m_dens;
    if constexpr (SPEC >= 0) {
        static_assert(MechSpec<SPEC>::NS == NS, "mechanism specialisation for another species count");
        if (evalcv_fast<NS, SPEC>(th, y, q, d, m_dens, _dens, m_p)) return;
    }
    // species Gibbs energy and internal-energy ingredients at T (Ri = 1)
    double h1[NS], gk[NS], cv;
    RxnCtx c;
    if (SPEC >= 0 || !evalcv_species<NS, false>(th, y, m_p, h1, gk, cv, c)) {
        const TPre t = th->thermo ? tpre<true>(m_tmp, 1) : tpre<true>(m_tmp, 0);
#pragma unroll
        for (int n = 0; n < NS; n++) {
            h1[n] = h_k(th, t, 1.0, n);
            double temp = 0.0;
            temp += s_k(th, t, 1.0, n);
            temp += (-h1[n] / m_tmp);
            gk[n] = temp;
        }
        cv = mix_cv<NS>(th, y + 1, t);
        c.m_tmp = m_tmp;
        // log T: the fit's log max(T, 200) when T >= 200 (the same call on the same value)
        c.logT = m_tmp >= 200.0 ? t.lT : dlog(m_tmp);
        c.logP = dlog(m_p * (1.0 / 101325.0));
        c.logStandConc = dlog(m_p / (R0 * m_tmp));
        c.rT = 1.0 / m_tmp;
        c.t_ok = __all(m_tmp >= 0x1p-500 && m_tmp <= 0x1p500);
    }
    double m_cm[NS];
#pragma unroll
    for (int n = 0; n < NS; n++) m_cm[n] = y[1 + n] * th->_Wi[n] * m_dens * 1.0E-3;
    double *qi = q + 1, *pi = d + 1;
#pragma unroll
    for (int n = 0; n < NS; n++) qi[n] = 0.0, pi[n] = 0.0;
    const int NR = mc->NR;
    for (int r = 0; r < NR; r++) {
        // the uniform record, read in one burst of scalar loads
        const DevRxn R = mc->rx[r];
        const double *er = mc->third + r * NS;
        rxn_step<NS>(R, [er](int it) { return er[it]; }, c, gk, m_cm, qi, pi);
    }
    evalcv_energy<NS>(th, h1, m_tmp, _dens, cv, q, d);
}

// evalcv with the work of one cell spread over the 64 lanes of a wave, every
// input uniform across the wave and every output left uniform: lane n < NS
// evaluates species n's enthalpy and Gibbs energy, lane r < NR reaction r's
// forward and reverse rates; both are broadcast, and every lane then sums
// the species' production and loss over the reactions in increasing order
// and finishes the temperature terms exactly as evalcv_dev.  The operations
// on every value are evalcv_dev's, so the results are its bits (the table
// form of the rates, which equals every compiled mechanism's).
template <int NS>
__device__ __forceinline__ void evalcv_coop(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc,
                                            const double *y, double *q, double *d, double m_dens, double m_p)
{
    const int ln = threadIdx.x & 63;
    const double m_tmp = y[0];
    const double _dens = 1.0 / m_dens;
    const TPre t = th->thermo ? tpre<true>(m_tmp, 1) : tpre<true>(m_tmp, 0);
    double h1[NS], gk[NS];
    {
        double h = 0.0, gv = 0.0;
        if (ln < NS) {
            h = h_k(th, t, 1.0, ln);
            double temp = 0.0;
            temp += s_k(th, t, 1.0, ln);
            temp += (-h / m_tmp);
            gv = temp;
        }
#pragma unroll
        for (int n = 0; n < NS; n++) h1[n] = __shfl(h, n), gk[n] = __shfl(gv, n);
    }
    const double logStandConc = dlog(m_p / (R0 * m_tmp));
    // log T: the fit's log max(T, 200) when T >= 200 (the same call on the same value)
    const double logT = m_tmp >= 200.0 ? t.lT : dlog(m_tmp);
    const double logP = dlog(m_p * (1.0 / 101325.0));
    double m_cm[NS];
#pragma unroll
    for (int n = 0; n < NS; n++) m_cm[n] = y[1 + n] * th->_Wi[n] * m_dens * 1.0E-3;
    RxnCtx c;
    c.m_tmp = m_tmp, c.logT = logT, c.logP = logP, c.logStandConc = logStandConc;
    c.rT = 1.0 / m_tmp;
    c.t_ok = m_tmp >= 0x1p-500 && m_tmp <= 0x1p500;
    const int NR = mc->NR;
    double Kf = 0.0, Kck = 0.0;
    if (ln < NR) {
        const DevRxn R = mc->rx[ln];
        const double *er = mc->third + ln * NS;
        rxn_rates<NS>(R, [er](int it) { return er[it]; }, c, gk, m_cm, Kf, Kck);
    }
    double *qi = q + 1, *pi = d + 1;
#pragma unroll
    for (int n = 0; n < NS; n++) qi[n] = 0.0, pi[n] = 0.0;
    for (int r = 0; r < NR; r++) {
        const DevRxn &R = mc->rx[r];
        rxn_accum<NS>(R.mf, R.mb, R.pf, R.pb, __shfl(Kf, r), __shfl(Kck, r), qi, pi);
    }
    double q0 = 0.0, d0 = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) {
        qi[n] *= th->Wi[n] * _dens;
        pi[n] *= th->Wi[n] * _dens;
        const double ei = (h1[n] - m_tmp) * th->Ri[n];
        q0 -= qi[n] * ei, d0 -= pi[n] * ei;
    }
    const double cv = mix_cv<NS>(th, y + 1, t);
    const double _Cv = 1.0 / cv;
    q[0] = q0 * _Cv, d[0] = d0 * _Cv;
}

__device__ __forceinline__ double alpha_of(double r)
{
    return (180.0 + r * (60.0 + r * (11.0 + r))) / (360.0 + r * (60.0 + r * (12.0 + r)));
}

// The predictor and corrector divide seven times per component, which as IEEE
// divisions were 770 of a pass's 3460 vector instructions, chained through the carry
// register, with a branch per component around the error norm.  For the species they
// take the unscaled sequence, all components in one block.  Its quotient is the
// IEEE-rounded one while divisor and dividend stay clear of the ends of the range:
// the divisors are at least ymin, 1 or 1e-30 where the ratios r and the rates are not
// negative, and in_range bounds all of them.  A dividend so small that the remainder
// underflows leaves a quotient below 2^-890, whose last bits reach nothing: it is only
// ever added to ymin or more, or competes with eps >= 1e-10.  The temperature's rates
// may have either sign, and it keeps the IEEE division.  k_chem on the 128^3 mixing
// layer went on from 997 to 947 us, k_chem_queue on the channel from 106 to 102; at one
// pass a cell a launch on 128^3 takes 480 us now, 771 before both.
//
// a non-negative number up to 2^160: its upper word is at most this one
constexpr unsigned CHEM_IN_RANGE = (1023u + 160u) << 20;
__device__ __forceinline__ void in_range(unsigned &top, double a)
{
    const unsigned h = (unsigned)__double2hiint(a); // negative, infinite and NaN: larger
    top = h > top ? h : top;
}
// a / b: FAST by ddiv_core
template <bool FAST> __device__ __forceinline__ double chem_div(double a, double b)
{
    return FAST ? ddiv_core(a, b) : a / b;
}
template <bool FAST> __device__ __forceinline__ double chem_alpha(double r)
{
    return chem_div<FAST>(180.0 + r * (60.0 + r * (11.0 + r)), 360.0 + r * (60.0 + r * (12.0 + r)));
}

// Chemeq2 state of one cell, advanced one rate evaluation at a time so that
// a lane can also work through a queue of cells (k_chem_queue).  Every
// advance is: before() -> evalcv_dev(y) -> after().  The first advance of a
// cell is the start-up (clip and renormalise Y, initial step from the rates,
// ProductionRates.h:488-530); each later one is a predictor/corrector pass
// (ProductionRates.h:531-638).  The sequence of operations per cell is the
// reference's; only the place of the rate evaluation in the code is shared.
//
// Where the saved state (ys, qs, ds) and rtau live is a policy: registers for
// the one-lane-per-cell kernel, LDS for the queue kernel, whose persistent
// one-wave blocks would otherwise spill them to scratch memory at two waves
// per SIMD.  Only the storage differs; the arithmetic is the same.
template <int NL> struct ChemRegs {
    double a[4][NL];
    __device__ __forceinline__ double &at(int k, int i) { return a[k][i]; }
};
// arrays k = 0..3 of lane `lane`: p[(k * NL + i) * 64], lane-contiguous rows
// (consecutive lanes hit consecutive banks)
template <int NL> struct ChemLds {
    double *p;
    __device__ __forceinline__ double &at(int k, int i) { return p[(k * NL + i) * 64]; }
};

template <int NS, class St = ChemRegs<NS + 1>, int SPEC = -1> struct ChemLane {
    static constexpr int NL = NS + 1;
    double y[NL], q[NL], d[NL];
    St st;
    double dt, dtg, dtmin, epsmax, ts, tn, rho, m_p;
    int passes;
    bool started;
    __device__ __forceinline__ double &ys(int i) { return st.at(0, i); }
    __device__ __forceinline__ double &qs(int i) { return st.at(1, i); }
    __device__ __forceinline__ double &ds(int i) { return st.at(2, i); }
    __device__ __forceinline__ double &rtau(int i) { return st.at(3, i); }

    __device__ __forceinline__ void begin(double dtg_, double rho_, double p_)
    {
        dtg = dtg_, rho = rho_, m_p = p_;
        dtmin = 1.0e-7, epsmax = 1.0;
        started = false;
        passes = 0;
    }

    // returns -1 when the pass count reaches the safety bound (no evaluation
    // is needed then), 0 otherwise
    __device__ __forceinline__ int before()
    {
        const double ymin = 1.0e-20;
        if (!started) {
            double sumy = 0.0;
#pragma unroll
            for (int i = 1; i < NL; i++) y[i] = dmax(y[i], ymin), sumy += y[i];
            sumy = 1.0 / sumy;
#pragma unroll
            for (int i = 1; i < NL; i++) y[i] *= sumy;
            return 0;
        }
        if (++passes > CHEM_MAXSUB) return -1;
        unsigned top = 0;
        predict<false>(0, 1, top);
        predict<true>(1, NL, top);
        if (__any(top > CHEM_IN_RANGE)) predict<false>(1, NL, top);
        tn = ts + dt;
        return 0;
    }

    // components lo .. hi - 1; FAST: top collects the words that in_range bounds
    template <bool FAST> __device__ __forceinline__ void predict(int lo, int hi, unsigned &top)
    {
        const double ymin = 1.0e-20;
#pragma unroll
        for (int i = lo; i < hi; i++) {
            const double rt = chem_div<FAST>(dt * ds(i), ys(i));
            rtau(i) = rt;
            const double alpha = chem_alpha<FAST>(rt);
            const double scr = chem_div<FAST>(dt * (qs(i) - ds(i)), 1.0 + alpha * rt);
            if (FAST) in_range(top, rt), in_range(top, ys(i)), in_range(top, qs(i));
            y[i] = dmax(ys(i) + scr, ymin);
        }
    }
    // the corrector with the convergence test: the new values, and eps raised to the
    // components' errors
    template <bool FAST>
    __device__ __forceinline__ void correct(int lo, int hi, double *yn, double &eps, unsigned &top)
    {
        const double ymin = 1.0e-20;
#pragma unroll
        for (int i = lo; i < hi; i++) {
            const double yp = y[i];
            const double rtaub = 0.5 * (rtau(i) + chem_div<FAST>(dt * d[i], yp));
            const double alpha = chem_alpha<FAST>(rtaub);
            const double ysi = ys(i);
            const double qt = (1.0 - alpha) * qs(i) + alpha * q[i];
            const double scr = chem_div<FAST>(qt * dt - rtaub * ysi, 1.0 + alpha * rtaub);
            const double scr2 = dmax(ysi + scr, 0.0);
            double scr1 = fabs(scr2 - yp);
            yn[i] = dmax(scr2, ymin);
            scr1 = chem_div<FAST>(scr1, yn[i]);
            const double err =
                0.5 * (scr1 + dmin(chem_div<FAST>(fabs(q[i] - d[i]), q[i] + d[i] + 1.0e-30), scr1));
            eps = (0.25 * (ysi + yn[i])) > ymin ? dmax(err, eps) : eps;
            if (FAST) {
                in_range(top, yp), in_range(top, rtaub), in_range(top, yn[i]);
                in_range(top, q[i]), in_range(top, d[i]);
            }
        }
    }

    // after the rate evaluation at y: 1 = reached dtg, 0 = continue
    __device__ __forceinline__ int after()
    {
        const double tfd = 1.0 + 1.0e-10, epscl = 1.0e4;
        if (!started) {
            const double epsmin = 1.0e-4, sqreps = 0.05;
            double scrtch = 1e-25;
#pragma unroll
            for (int i = 0; i < NL; i++) {
                const double ascr = fabs(q[i]);
                const double sb = 0.1 * epsmin * ascr - d[i];
                const double scr2 = (sb >= 0.0 ? 1.0 : -1.0) * fabs(1.0 / y[i]);
                const double scr1 = scr2 * d[i];
                scrtch = dmax(-fabs(ascr - d[i]) * scr2, dmax(scr1, scrtch));
            }
            dt = dmin(sqreps / scrtch, dtg);
            dtmin *= dt;
            ts = 0.0, tn = 0.0;
#pragma unroll
            for (int i = 0; i < NL; i++) ys(i) = y[i], qs(i) = q[i], ds(i) = d[i];
            started = true;
            return 0;
        }
        double eps0 = 1e-10, yn[NL];
        unsigned top = 0;
        correct<false>(0, 1, yn, eps0, top);
        double eps = eps0;
        correct<true>(1, NL, yn, eps, top);
        if (__any(top > CHEM_IN_RANGE)) {
            eps = eps0;
            correct<false>(1, NL, yn, eps, top);
        }
#pragma unroll
        for (int i = 0; i < NL; i++) y[i] = yn[i];
        eps = eps * epscl;
        if (eps < epsmax) {
            if (dtg <= (tn * tfd)) return 1;
        } else {
            tn = ts;
        }
        const double dto = dt;
        double rteps = 0.5 * (eps + 1.0);
        rteps = 0.5 * (rteps + eps / rteps);
        rteps = 0.5 * (rteps + eps / rteps);
        dt = dmin(dt * (1.0 / rteps + 0.005), tfd * (dtg - tn));
        if (eps > epsmax) {
            dt = dmin(dt, 0.34 * dto);
            if (dt <= dtmin) epsmax *= 10.0;
            return 0; // back to the predictor from the same saved state
        }
        epsmax = 1.0;
        ts = tn;
#pragma unroll
        for (int i = 0; i < NL; i++) ys(i) = y[i], qs(i) = q[i], ds(i) = d[i];
        return 0;
    }

    // one advance: 1 = done, 0 = continue, -1 = safety bound
    __device__ __forceinline__ int advance(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc)
    {
        if (before() < 0) return -1;
        evalcv_dev<NS, SPEC>(th, mc, y, q, d, rho, m_p);
        return after();
    }
    // the same advance by a whole wave on one cell (state uniform across
    // the wave): the rate evaluation spread over the lanes
    __device__ __forceinline__ int advance_coop(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc)
    {
        if (before() < 0) return -1;
        evalcv_coop<NS>(th, mc, y, q, d, rho, m_p);
        return after();
    }
};

// Everything of a cell's CHEMEQ2 run between two passes, so that a cell the
// queue lanes hand over continues on a whole wave (k_chem_coop) from exactly
// where it stopped: y, q, d, ys, qs, ds, rtau, the step state, the start
// energy, the cell and its case.
template <int NS> struct ChemSpill {
    static constexpr int NL = NS + 1;
    static constexpr int NV = 7 * NL + 9;
    double v[NV];
    long long id, tl;
    int passes, started, k, pad;
};

template <int NS, class St, int SPEC>
__device__ __forceinline__ void chem_spill_save(ChemSpill<NS> &r, ChemLane<NS, St, SPEC> &L, double e0, long long id,
                                                long long tl, int k)
{
    constexpr int NL = NS + 1;
#pragma unroll
    for (int i = 0; i < NL; i++) {
        r.v[i] = L.y[i], r.v[NL + i] = L.q[i], r.v[2 * NL + i] = L.d[i];
        r.v[3 * NL + i] = L.ys(i), r.v[4 * NL + i] = L.qs(i), r.v[5 * NL + i] = L.ds(i), r.v[6 * NL + i] = L.rtau(i);
    }
    double *w = r.v + 7 * NL;
    w[0] = L.dt, w[1] = L.dtg, w[2] = L.dtmin, w[3] = L.epsmax, w[4] = L.ts, w[5] = L.tn, w[6] = L.rho, w[7] = L.m_p;
    w[8] = e0;
    r.id = id, r.tl = tl, r.passes = L.passes, r.started = L.started ? 1 : 0, r.k = k;
}

template <int NS, class St, int SPEC>
__device__ __forceinline__ double chem_spill_load(const ChemSpill<NS> &r, ChemLane<NS, St, SPEC> &L)
{
    constexpr int NL = NS + 1;
#pragma unroll
    for (int i = 0; i < NL; i++) {
        L.y[i] = r.v[i], L.q[i] = r.v[NL + i], L.d[i] = r.v[2 * NL + i];
        L.ys(i) = r.v[3 * NL + i], L.qs(i) = r.v[4 * NL + i], L.ds(i) = r.v[5 * NL + i], L.rtau(i) = r.v[6 * NL + i];
    }
    const double *w = r.v + 7 * NL;
    L.dt = w[0], L.dtg = w[1], L.dtmin = w[2], L.epsmax = w[3], L.ts = w[4], L.tn = w[5], L.rho = w[6], L.m_p = w[7];
    L.passes = r.passes, L.started = r.started != 0;
    return w[8];
}

// Chemeq2 on one cell, its saved state at lds (lane-strided, ChemLds).
// Returns predictor passes, or -1 at the safety bound.
template <int NS, int SPEC>
__device__ int chemeq2_dev(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc, double *y, double dtg,
                           double rho, double m_p, double *lds)
{
    ChemLane<NS, ChemLds<NS + 1>, SPEC> L;
    L.st.p = lds;
#pragma unroll
    for (int i = 0; i < NS + 1; i++) L.y[i] = y[i];
    L.begin(dtg, rho, m_p);
    int st;
    while ((st = L.advance(th, mc)) == 0) {
    }
#pragma unroll
    for (int i = 0; i < NS + 1; i++) y[i] = L.y[i];
    return st < 0 ? -1 : L.passes;
}

// get_Cope (Mixing_device.h:145-154) at one temperature
template <int NS>
__device__ __forceinline__ double mix_e(const DevThermo *__restrict__ th, const double *yi, double T)
{
    double e = 0.0;
    cdouble *Rk = as_const(th->Ri);
    auto sum = [&](auto fam) {
        constexpr bool NASA = decltype(fam)::value;
        // (twice a cell: the general form below serves the colder waves)
        if (__all(T >= 200.0 && T <= fast_top(th))) {
            fast_ranges<NASA, false>(th, T, NASA, [&](cdouble *c, auto t) {
#pragma unroll
                for (int n = 0; n < NS; n++)
                    e += (h_fast<NASA>(c + FITC * n, t.T, t.iT, t.lT, 1.0) - T) * Rk[n] * yi[n];
            });
            return;
        }
        const TPre t = tpre<NASA>(T, NASA ? 1 : 0);
#pragma unroll
        for (int n = 0; n < NS; n++) {
            const double ei = (h_k(th, t, 1.0, n) - T) * th->Ri[n];
            e += ei * yi[n];
        }
    };
    if (th->thermo) sum(std::true_type{});
    else sum(std::false_type{});
    return e;
}

// The mass fractions a cell's chemistry starts from: the y array of the
// Reaction's UpdateStates (ChemeODEQ2SolverKernel1 reads it,
// Reaction_kernels.hpp:58-60) -- Y_k = U_{5+k} / rho and the remainder, or for
// a GhostSpecies mixture the stored renormalised planes and 0
template <int NS>
__device__ __forceinline__ void chem_y0(const double *U, const double *ypl, int ghost, long long N, long long id,
                                        double rho1, double *yi)
{
    if (ghost) {
        yi[NS - 1] = 0.0;
#pragma unroll
        for (int k = 0; k < NS - 1; k++) yi[k] = ypl[k * N + id];
    } else {
        yi[NS - 1] = 1.0;
#pragma unroll
        for (int k = 0; k < NS - 1; k++) {
            yi[k] = U[(5 + k) * N + id] * rho1;
            yi[NS - 1] += -yi[k];
        }
    }
}

// One interior cell of ChemeODEQ2SolverKernel1.
template <int NS, int SPEC>
__device__ __forceinline__ int chem_cell(const Geom &g, const DevThermo *__restrict__ th,
                                         const DevMech *__restrict__ mc, Fields &f, long long N, long long id,
                                         double dtc, double *lds)
{
    // the cell's CHEMEQ2 state held directly (no copy of y in and out)
    ChemLane<NS, ChemLds<NS + 1>, SPEC> L;
    L.st.p = lds;
    L.y[0] = f.T[id];
    const double rho = f.U[id]; // rho = U[0] (Getrhoyi)
    const double rho1 = 1.0 / rho;
    chem_y0<NS>(f.U, f.y, g.ghost, N, id, rho1, L.y + 1);
    const double e0 = mix_e<NS>(th, L.y + 1, L.y[0]);
    L.begin(dtc, rho, f.p[id]);
    int st;
    while ((st = L.advance(th, mc)) == 0) {
    }
    const double e1 = mix_e<NS>(th, L.y + 1, L.y[0]);
#pragma unroll
    for (int n = 0; n < NS - 1; n++) f.U[(5 + n) * N + id] = L.y[1 + n] * rho;
    f.T[id] = L.y[0];
    f.U[4 * N + id] += (e1 - e0) * rho;
    return st < 0 ? -1 : L.passes;
}

// EstimateNAN after the Reaction (flag 4, src/XFLUIDS.cpp:639;
// EstimateFluidNANKernel, src/Fluids.cpp:47-87) on the cell the chemistry has
// just written: U[0] < 0 or any component NaN/Inf.  The reference also reads
// the third stage's LU there, which that stage's own check passed and nothing
// has changed since.
__device__ __forceinline__ bool cell_bad(const double *U, long long N, long long id, int E)
{
    bool bad = U[id] < 0;
    for (int n = 0; n < E; n++) {
        const double a = U[n * N + id];
        bad = bad || isnan(a) || isinf(a);
    }
    return bad;
}

// two waves per SIMD for the 9-species state (<= 256 registers per lane)
template <int NS> struct ChemOccupancy {
    static constexpr int waves = NS <= 3 ? 3 : 2;
};

// LDS of one one-wave block: ys, qs, ds and rtau of its 64 lanes, 20 KiB at
// NS = 9, so the 8 blocks of two waves per SIMD fill the CU's 160 KiB
template <int NS> struct ChemQueueLds {
    static constexpr int doubles = 4 * (NS + 1) * 64;
};

// one lane per interior cell, one-wave blocks; check = 1 (a time step's
// Reaction) also runs the post-Reaction NaN check on the cell.  The saved
// CHEMEQ2 state (ys, qs, ds, rtau) lives in LDS: in registers, with the rate
// evaluation's, it needs ~380 per lane and the kernel ran one wave per SIMD.
template <int NS, int SPEC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(ChemOccupancy<NS>::waves)))
k_chem(Geom g, const DevThermo *__restrict__ th, const DevMech *__restrict__ mc, Fields f, int record, int check)
{
    __shared__ double lds[ChemQueueLds<NS>::doubles];
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long total = (long long)g.X_inner * g.Y_inner * g.Z_inner;
    if (t >= total) return;
    if (step_halted(f.err, ~CHEM_BITS)) return;
    const int i = g.Bx + (int)(t % g.X_inner);
    const int j = g.By + (int)((t / g.X_inner) % g.Y_inner);
    const int k = g.Bz + (int)(t / ((long long)g.X_inner * g.Y_inner));
    const long long id = (long long)g.Xmax * g.Ymax * k + (long long)g.Xmax * j + i;
    const int passes = chem_cell<NS, SPEC>(g, th, mc, f, g.N, id, f.dt[DT_CHEM], lds + (threadIdx.x & 63));
    if (record) f.substeps[t] = passes;
    int bits = passes < 0 ? EBIT_CHEM : 0;
    if (passes < 0) report_cell(f.err, EBIT_CHEM, id);
    if (check && cell_bad(f.U, g.N, id, NS + 4)) {
        report_cell(f.err, EBIT_NAN, id);
        bits |= EBIT_NAN;
    }
    if (bits) report_pass(f.err, bits, 4);
}

// Interior cell t (0 <= t < total) -> padded-grid id
__device__ __forceinline__ long long chem_cell_id(const Geom &g, long long t)
{
    const int i = g.Bx + (int)(t % g.X_inner);
    const int j = g.By + (int)((t / g.X_inner) % g.Y_inner);
    const int k = g.Bz + (int)(t / ((long long)g.X_inner * g.Y_inner));
    return (long long)g.Xmax * g.Ymax * k + (long long)g.Xmax * j + i;
}

// The part of one case the chemistry step touches.  `off` is the index of
// the case's first interior cell in the concatenated cell list of an
// ensemble (0 for a single case).
struct ChemCase {
    long long off;
    Geom g;
    double *U, *T, *p, *dt;
    int *substeps, *err;
    double *y; // GhostSpecies mass-fraction planes (g.ghost), else unused
};

// Write-back of a finished cell (ChemeODEQ2SolverKernel1's tail,
// Reaction_kernels.hpp:60-73): Ns-1 partial densities, T, the energy
// change; the pass count; the pass bound and post-Reaction NaN check.
template <int NS, class St, int SPEC>
__device__ __forceinline__ void chem_store(const DevThermo *__restrict__ th, const ChemCase &cc, long long id,
                                           long long tl, ChemLane<NS, St, SPEC> &L, double e0, int st, int record,
                                           int check)
{
    const long long N = cc.g.N;
    const double rho = L.rho;
    const double e1 = mix_e<NS>(th, L.y + 1, L.y[0]);
#pragma unroll
    for (int n = 0; n < NS - 1; n++) cc.U[(5 + n) * N + id] = L.y[1 + n] * rho;
    cc.T[id] = L.y[0];
    cc.U[4 * N + id] += (e1 - e0) * rho;
    if (record) cc.substeps[tl] = st < 0 ? -1 : L.passes;
    int bits = st < 0 ? EBIT_CHEM : 0;
    if (st < 0) report_cell(cc.err, EBIT_CHEM, id);
    if (check && cell_bad(cc.U, N, id, NS + 4)) {
        report_cell(cc.err, EBIT_NAN, id);
        bits |= EBIT_NAN;
    }
    if (bits) report_pass(cc.err, bits, 4);
}

// Cells that the queue's lanes hand to whole waves: records, their count
// (count[0], may exceed cap: the lanes that found the list full kept their
// cells) and the waves' pick counter (count[1]); a cell is handed over once
// it has run `after` passes.  cap = 0: no hand-over.
struct ChemSpillBuf {
    void *rec;
    unsigned *count;
    int cap, after;
};

// Work-queue driver: persistent lanes draining the interior cells of one or
// several cases.  Cells of very different stiffness take from 1 to ~10^3
// passes; with one lane per cell a wave runs as long as its stiffest cell
// while the other lanes idle.  Here every lane that has finished a cell takes
// the next one from a device counter (one atomic per wave, handed out by lane
// rank), so the lanes of a wave stay busy with the same code until the queue
// is empty; a cell that starts and the cells that continue share one rate
// evaluation per iteration.  A cell still running after sp.after passes is
// handed to the whole-wave kernel (k_chem_coop) while the list has
// room: a few very stiff cells would otherwise keep single lanes busy, one
// serial rate evaluation after another, long after the rest.  Each cell's
// arithmetic is exactly that of the per-cell driver.  Termination: the
// counter only grows, a wave stops once every lane has drawn an index >=
// total and holds no cell, and a cell is bounded by CHEM_MAXSUB passes.  The
// counters must be zero at launch.
template <int NS, int SPEC, class Cases>
__device__ __forceinline__ void chem_queue_run(const Cases &cases, long long total, const DevThermo *__restrict__ th,
                                               const DevMech *__restrict__ mc, unsigned long long *queue, int record,
                                               int check, double *lds, ChemSpillBuf sp)
{
    const int lane = threadIdx.x & 63;
    ChemLane<NS, ChemLds<NS + 1>, SPEC> L;
    L.st.p = lds + lane;
    // a lane keeps only its cell's case index, id and interior index across
    // passes; the case record is read again where it is needed (for an
    // ensemble it differs per lane, and holding it would cost ~40 registers)
    long long tl = -1, id = 0;
    int ck = 0;
    double e0 = 0.0;
    bool active = false, done = false, can_spill = sp.cap > 0;
    for (;;) {
        // every lane without a cell draws until it has one or the queue is empty; the
        // cells of a case whose step has halted are passed over
        while (const unsigned long long want = __ballot(!active && !done)) {
            const int cnt = __popcll(want);
            const int leader = __ffsll((long long)want) - 1;
            unsigned long long base = 0;
            if (lane == leader) base = atomicAdd(queue, (unsigned long long)cnt);
            base = __shfl(base, leader);
            if (!active && !done) {
                const int rank = __popcll(want & ((1ull << lane) - 1ull));
                const long long t = (long long)(base + (unsigned long long)rank);
                ChemCase cc{};
                if (t < total) {
                    ck = cases.find_k(t);
                    cc = cases.get(ck);
                }
                if (t < total && !lane_halted(cc.err, ~CHEM_BITS)) {
                    tl = t - cc.off;
                    const long long N = cc.g.N;
                    id = chem_cell_id(cc.g, tl);
                    L.y[0] = cc.T[id];
                    const double rho = cc.U[id];
                    const double rho1 = 1.0 / rho;
                    chem_y0<NS>(cc.U, cc.y, cc.g.ghost, N, id, rho1, L.y + 1);
                    e0 = mix_e<NS>(th, L.y + 1, L.y[0]);
                    L.begin(cc.dt[DT_CHEM], rho, cc.p[id]);
                    active = true;
                } else if (t >= total) {
                    done = true;
                } else if (rank == cnt - 1) {
                    // the wave's last index lies in a halted case: the counter goes on
                    // behind it (every index up to there is one of that case's cells)
                    atomicMax(queue, (unsigned long long)(cc.off + (long long)cc.g.X_inner * cc.g.Y_inner * cc.g.Z_inner));
                }
            }
        }
        if (!__any(active)) break;
        if (active) {
            // starting cells and running cells share this one evaluation
            const int st = L.advance(th, mc);
            if (st != 0) {
                chem_store<NS>(th, cases.get(ck), id, tl, L, e0, st, record, check);
                active = false;
            } else if (can_spill && L.passes >= sp.after) {
                const unsigned idx = atomicAdd(sp.count, 1u);
                if (idx < (unsigned)sp.cap) {
                    chem_spill_save(((ChemSpill<NS> *)sp.rec)[idx], L, e0, id, tl, ck);
                    active = false;
                } else {
                    can_spill = false; // the list is full: keep this cell here
                }
            }
        }
    }
}

// The cells the queue handed over, one whole wave per cell (evalcv_coop):
// persistent one-wave blocks take records from the list until it is
// drained, and write each cell back as the queue would have.
template <int NS, class Cases>
__device__ __forceinline__ void chem_coop_run(const Cases &cases, const DevThermo *__restrict__ th,
                                              const DevMech *__restrict__ mc, ChemSpillBuf sp, int record, int check)
{
    const int ln = threadIdx.x & 63;
    const ChemSpill<NS> *rec = (const ChemSpill<NS> *)sp.rec;
    const unsigned n = min(sp.count[0], (unsigned)sp.cap);
    for (;;) {
        unsigned idx = 0;
        if (ln == 0) idx = atomicAdd(sp.count + 1, 1u);
        idx = __shfl(idx, 0);
        if (idx >= n) break;
        ChemLane<NS, ChemRegs<NS + 1>, -1> L;
        const double e0 = chem_spill_load(rec[idx], L);
        const ChemCase cc = cases.get(rec[idx].k);
        int st;
        while ((st = L.advance_coop(th, mc)) == 0) {
        }
        if (ln == 0) chem_store<NS>(th, cc, rec[idx].id, rec[idx].tl, L, e0, st, record, check);
    }
}

struct OneCase {
    ChemCase c;
    __device__ __forceinline__ int find_k(long long) const { return 0; }
    __device__ __forceinline__ ChemCase get(int) const { return c; }
};

// cases[k].off ascending; the case holding cell t by binary search
struct ManyCases {
    const ChemCase *cases;
    int n;
    __device__ __forceinline__ int find_k(long long t) const
    {
        int lo = 0, hi = n - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (cases[mid].off <= t) lo = mid;
            else hi = mid - 1;
        }
        return lo;
    }
    __device__ __forceinline__ ChemCase get(int k) const { return cases[k]; }
};


__device__ __forceinline__ OneCase one_case(const Geom &g, const Fields &f)
{
    OneCase one;
    one.c.off = 0;
    one.c.g = g;
    one.c.U = f.U, one.c.T = f.T, one.c.p = f.p, one.c.dt = f.dt;
    one.c.substeps = f.substeps, one.c.err = f.err;
    one.c.y = f.y;
    return one;
}

// the queue counter is queue[0..1] (64 bits); the hand-over counters follow
// (queue[2] records, queue[3] waves' picks)
template <int NS, int SPEC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(ChemOccupancy<NS>::waves)))
k_chem_queue(Geom g, const DevThermo *__restrict__ th, const DevMech *__restrict__ mc, Fields f, int record,
             int check, void *spill, int spill_cap, int spill_after)
{
    const OneCase one = one_case(g, f);
    __shared__ double lds[ChemQueueLds<NS>::doubles];
    const ChemSpillBuf sp{spill, f.queue + 2, spill_cap, spill_after};
    chem_queue_run<NS, SPEC>(one, (long long)g.X_inner * g.Y_inner * g.Z_inner, th, mc, (unsigned long long *)f.queue,
                             record, check, lds, sp);
}

// one queue over the cells of every case of an ensemble (shared mechanism)
template <int NS, int SPEC>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(ChemOccupancy<NS>::waves)))
k_chem_queue_multi(const ChemCase *__restrict__ cases, int ncases, long long total, const DevThermo *__restrict__ th,
                   const DevMech *__restrict__ mc, unsigned long long *queue, int record, int check, void *spill,
                   int spill_cap, int spill_after)
{
    ManyCases many{cases, ncases};
    __shared__ double lds[ChemQueueLds<NS>::doubles];
    const ChemSpillBuf sp{spill, (unsigned *)queue + 2, spill_cap, spill_after};
    chem_queue_run<NS, SPEC>(many, total, th, mc, queue, record, check, lds, sp);
}

// the handed-over cells of one case / of an ensemble, one wave per cell
template <int NS>
__global__ void __launch_bounds__(64) k_chem_coop(Geom g, const DevThermo *__restrict__ th,
                                                  const DevMech *__restrict__ mc, Fields f, int record, int check,
                                                  void *spill, int spill_cap)
{
    const OneCase one = one_case(g, f);
    chem_coop_run<NS>(one, th, mc, ChemSpillBuf{spill, f.queue + 2, spill_cap, 0}, record, check);
}
template <int NS>
__global__ void __launch_bounds__(64) k_chem_coop_multi(const ChemCase *__restrict__ cases, int ncases,
                                                        const DevThermo *__restrict__ th,
                                                        const DevMech *__restrict__ mc, unsigned long long *queue,
                                                        int record, int check, void *spill, int spill_cap)
{
    ManyCases many{cases, ncases};
    chem_coop_run<NS>(many, th, mc, ChemSpillBuf{spill, (unsigned *)queue + 2, spill_cap, 0}, record, check);
}

// ---------------------------------------------------------------------------
// One cell per wave (XF_CHEM_WAVE).  With few cells (a 1-D tube) the chemistry
// launch lasts as long as the stiffest cell's serial chain of passes, about
// 4500 instructions each on one lane.  Here the wave of a cell spreads every
// pass over its lanes: lane i < NS + 1 holds solution component i (0 = T,
// 1 + n = Y_n) and does that component's predictor and corrector; lane 1 + n
// evaluates species n's enthalpy, Gibbs energy and concentration, lane r < NR
// reaction r's rates, and lane 1 + n sums its species' production and loss
// over the reactions in order.  Every sum and maximum the reference forms over
// components or species (normalisation, step-size scratch, energy terms, Cv,
// the error norm) runs as an ordered chain over the lanes' values, so each
// value is rounded exactly as in ChemLane / evalcv_dev and the results are the
// per-cell driver's bits.  Requires NS + 1 <= 64 and NR <= 64.
//
// Bound by the latency of a pass's chains.  With the reactions' loops as branches on
// their records, a table walk at the start of every cell and 239 registers a lane, 8192
// cells (one pass each but for a few) took 98 us; as straight-line steps over packed
// records, with the lane's tables in LDS, 57, and 2000 cells (as long as the stiffest
// cell's passes) 37 instead of 56.
// ---------------------------------------------------------------------------

// Cross-lane exchanges of the cell's wave go through LDS: the lanes that own
// values write them, one barrier (a single wave: no wait on other waves), and
// every lane reads them back at the same addresses (LDS broadcasts).  Sums are
// then formed on every lane in the reference's order.
template <int NS> struct WaveShared {
    double K[2 * MAXNR]; // Kf, Kck of each reaction, side by side; 0 beyond the last
    double S[2 * MAXNS]; // log p less the Gibbs energy (general path: the energy) and concentration of each species
    double V[4 * 64];    // per-lane operands of the ordered sums
    double hc[FITC - 1][16];  // species n's fit coefficients of the current range at [.][1 + n]
    double eff[NS][MAXNR];    // reaction r's third-body efficiencies
};

// lane k's value on every lane
__device__ __forceinline__ double wave_lane(double v, int k)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k),
                            __builtin_amdgcn_readlane(__double2loint(v), k));
}

// ((init + v[lo]) + v[lo+1]) + ... of a lane-indexed LDS array with stride st
__device__ __forceinline__ double lds_sum(const double *v, int st, int lo, int hi, double init)
{
    double s = init;
    for (int k = lo; k < hi; k++) s += v[k * st];
    return s;
}
// ((init - v[lo]) - v[lo+1]) - ...
__device__ __forceinline__ double lds_sub(const double *v, int st, int lo, int hi, double init)
{
    double s = init;
    for (int k = lo; k < hi; k++) s -= v[k * st];
    return s;
}

// a lane's column of coefficients in LDS
struct FitCol {
    const double *c;
    __device__ __forceinline__ double operator[](int m) const { return c[16 * m]; }
};

// What a lane reads on every pass, loaded once per cell: species lane 1 + n
// keeps W, 1/W and R of species n and its orders in the reactions, and in LDS the fit
// coefficients of the current range (reloaded when T crosses into another range);
// reaction lane r keeps its record, and its third-body efficiencies in LDS.
template <int NS> struct WaveLane {
    double Wi = 0.0, iWi = 0.0, Ri = 0.0;
    int rc = -1; // range the coefficients hc belong to
    double *hc; // the lane's coefficients: m at hc[16 * m] (FitCol)
    DevWaveRxn R{};
    unsigned acc[MAXNR / 4];
    bool fast; // the tables qualify for the straight-line path

    __device__ __forceinline__ void load(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc,
                                         WaveShared<NS> &sh, int NR, double m_p)
    {
        const int ln = threadIdx.x & 63;
        const bool sp = ln >= 1 && ln <= NS;
        hc = &sh.hc[0][ln & 15];
        if (ln < 16) {
#pragma unroll
            for (int m = 0; m < FITC - 1; m++) hc[16 * m] = 0.0;
        }
        if (sp) Wi = th->Wi[ln - 1], iWi = th->_Wi[ln - 1], Ri = th->Ri[ln - 1];
#pragma unroll
        for (int w = 0; w < MAXNR / 4; w++) acc[w] = sp ? mc->wacc[(ln - 1) * (MAXNR / 4) + w] : 0u;
        // an idle lane's record: every order 0, no factors
        R.nu = 0x8888888888888888ull, R.ff = R.fb = 15u | 15u << 5 | 15u << 10;
        if (ln < NR) {
            R = mc->wr[ln];
#pragma unroll
            for (int it = 0; it < NS; it++) sh.eff[it][ln] = mc->third[ln * NS + it];
        }
        fast = th->fast && mc->wave_ok && m_p >= 0x1p-300 && m_p <= 0x1p300;
    }
    // the fit coefficients of range r (the same on every lane: T is the cell's)
    __device__ __forceinline__ void range(const DevThermo *__restrict__ th, int r)
    {
        r = r < 0 ? 0 : r;
        if (r != rc) {
            const int ln = threadIdx.x & 63;
            if (ln >= 1 && ln <= NS) {
                const double *c = th->Hf + (r * MAXNS + ln - 1) * FITC;
#pragma unroll
                for (int m = 0; m < FITC - 1; m++) hc[16 * m] = c[m];
            }
            rc = r;
        }
    }
};

// the lane's Kf and Kck and the species lane's sums over the reactions, for T where
// the fast fits and quotients are exact; false, with nothing of use, when a value is
// not finite.  Every lane runs every step: terms of a zero order add a zero, factors
// that a reaction lacks are 1.  No branch and no table read is
// left between the barriers, the two logarithms run on different lanes, and the two
// exponentials together.
template <int NS, int THERMO>
__device__ __forceinline__ bool wave_rates(const DevThermo *__restrict__ th, WaveLane<NS> &W, WaveShared<NS> &sh,
                                           int NR, double yv, double T, double m_dens, double m_p, double logP,
                                           double &h1, double &ycp, double &qi, double &pi)
{
    const double inf = __longlong_as_double(0x7ff0000000000000LL);
    const int ln = threadIdx.x & 63;
    const bool sp = ln >= 1 && ln <= NS;
    const double iT = ddiv_core(1.0, T);
    const double lx = dlog_pos(ln < 32 ? T : ddiv_core(m_p, R0 * T));
    const double lT = wave_lane(lx, 0), logStandConc = wave_lane(lx, 32);
    W.range(th, THERMO ? (T >= 6000.0 ? 2 : (T >= 1000.0 ? 1 : 0)) : (T > 1000.0 ? 0 : 1));
    const FitCol hc{W.hc};
    h1 = h_fast<THERMO != 0>(hc, T, iT, lT, 1.0);
    double g = 0.0;
    g += s_fast<THERMO != 0>(hc, T, iT, lT);
    g += dquot(-h1, T, iT);
    const double lg = logP - g, conc = yv * W.iWi * m_dens * 1.0E-3;
    if (sp) sh.S[ln - 1] = lg, sh.S[MAXNS + ln - 1] = conc;
    if (ln == 0) sh.S[MAXNS + 15] = 1.0;
    ycp = yv * cp_fast<THERMO != 0>(hc, T, iT, W.Ri);
    __syncthreads();
    // the packed orders as values of their own on every pass: the compiler would keep
    // each, unpacked, in registers for the whole cell
    auto packed = [](unsigned v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    const unsigned nu[2] = {packed((unsigned)W.R.nu), packed((unsigned)(W.R.nu >> 32))};
    double DG = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) DG += ((int)((nu[n / 8] >> (4 * (n % 8))) & 15u) - 8) * sh.S[n];
    double arg[2] = {W.R.B * lT - dquot(W.R.EaR, T, iT), DG - W.R.dn * logStandConc}, e[2];
    dexp_n<2>(arg, e);
    double Kf = W.R.A * e[0], Kck = dmin(e[1], 1.0E+40);
    double tb = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) tb += sh.eff[n][ln < MAXNR ? ln : 0] * sh.S[MAXNS + n];
    Kf *= W.R.third ? tb : 1.0;
    Kck *= Kf;
    const unsigned ff = packed(W.R.ff), fb = packed(W.R.fb);
    auto factor = [&](unsigned f) {
        const double x = sh.S[MAXNS + (f & 15u)];
        return f & 16u ? x * x : x;
    };
#pragma unroll
    for (int k = 0; k < 3; k++) Kf *= factor(ff >> (5 * k));
#pragma unroll
    for (int k = 0; k < 3; k++) Kck *= factor(fb >> (5 * k));
    if (!__all((ln >= NR || (fabs(Kf) < inf && fabs(Kck) < inf)) && (!sp || (fabs(lg) < inf && fabs(conc) < inf))))
        return false;
    if (ln < MAXNR) sh.K[2 * ln] = ln < NR ? Kf : 0.0, sh.K[2 * ln + 1] = ln < NR ? Kck : 0.0;
    __syncthreads();
    qi = 0.0, pi = 0.0;
#pragma unroll
    for (int w = 0; w < MAXNR; w += 8) {
        if (w >= NR) break;
        const unsigned a[2] = {packed(W.acc[w / 4]), packed(W.acc[w / 4 + 1])};
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const unsigned b = a[r / 4] >> (8 * (r % 4));
            const int nf = (int)(b & 15u), nb = (int)((b >> 4) & 15u);
            const double kf = sh.K[2 * (w + r)], kc = sh.K[2 * (w + r) + 1];
            qi += nb * kf + nf * kc;
            pi += nf * kf + nb * kc;
        }
    }
    return true;
}

// the same for every T and value, with the tests of rxn_rates on the record
template <int NS, int THERMO>
__device__ __forceinline__ void wave_rates_general(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc,
                                                   WaveLane<NS> &W, WaveShared<NS> &sh, int NR, double yv, double T,
                                                   double m_dens, double m_p, double logP, double &h1, double &ycp,
                                                   double &qi, double &pi)
{
    const int ln = threadIdx.x & 63;
    const bool sp = ln >= 1 && ln <= NS;
    const TPre t = tpre<true>(T, THERMO);
    W.range(th, t.r);
    h1 = 0.0, ycp = 0.0;
    if (sp) {
        double hc[9];
#pragma unroll
        for (int m = 0; m < 9; m++) hc[m] = W.hc[16 * m];
        // h_k and s_k with Ri = 1
        h1 = h_fit(hc, THERMO, t, 1.0);
        if (t.TT < 200.0) h1 += cp200_k(th, 1.0, ln - 1) * (t.TT - 200.0);
        double temp = 0.0;
        temp += s_fit(hc, THERMO, t, 1.0);
        temp += (-h1 / T);
        sh.S[ln - 1] = temp;
        sh.S[MAXNS + ln - 1] = yv * W.iWi * m_dens * 1.0E-3;
        ycp = yv * cp_fit(hc, THERMO, t, W.Ri);
    }
    const double logStandConc = dlog(m_p / (R0 * T));
    // log T: the fit's log max(T, 200) when T >= 200 (the same call on the same value)
    const double logT = T >= 200.0 ? t.lT : dlog(T);
    __syncthreads();
    if (ln < NR) {
        RxnCtx c;
        c.m_tmp = T, c.logT = logT, c.logP = logP, c.logStandConc = logStandConc;
        c.rT = T >= 200.0 ? t.iT : 1.0 / T; // the fit's 1 / max(T, 200) when T >= 200
        c.t_ok = T >= 0x1p-500 && T <= 0x1p500;
        double Kf, Kck;
        rxn_rates<NS>(mc->rx[ln], [mc, ln](int it) { return mc->third[ln * NS + it]; }, c, sh.S, sh.S + MAXNS, Kf, Kck);
        sh.K[2 * ln] = Kf, sh.K[2 * ln + 1] = Kck;
    }
    __syncthreads();
    qi = 0.0, pi = 0.0;
    if (sp) {
        // a reaction adds to species n exactly when its nu_f or nu_b is non-zero
        for (int r = 0; r < NR; r++) {
            const unsigned b = (mc->wacc[(ln - 1) * (MAXNR / 4) + r / 4] >> (8 * (r % 4))) & 255u;
            if (b) {
                const int nf = (int)(b & 15u), nb = (int)(b >> 4);
                const double kf = sh.K[2 * r], kc = sh.K[2 * r + 1];
                qi += nb * kf + nf * kc;
                pi += nf * kf + nb * kc;
            }
        }
    }
}

// evalcv (ProductionRates.h:459-479) at the distributed state: yv is
// component ln, T the cell's; returns the component's q and d
template <int NS, int THERMO>
__device__ __forceinline__ void evalcv_wave(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc,
                                            WaveLane<NS> &W, WaveShared<NS> &sh, int NR, double yv, double T,
                                            double &qv, double &dv, double m_dens, double m_p, double _dens,
                                            double logP)
{
    const int ln = threadIdx.x & 63;
    double h1, ycp, qi, pi;
    if (!(W.fast && T >= 200.0 && T <= 1.0e5 &&
          wave_rates<NS, THERMO>(th, W, sh, NR, yv, T, m_dens, m_p, logP, h1, ycp, qi, pi)))
        wave_rates_general<NS, THERMO>(th, mc, W, sh, NR, yv, T, m_dens, m_p, logP, h1, ycp, qi, pi);
    if (ln >= 1 && ln <= NS) {
        qi *= W.Wi * _dens;
        pi *= W.Wi * _dens;
        const double ei = (h1 - T) * W.Ri;
        sh.V[4 * ln + 0] = qi * ei;
        sh.V[4 * ln + 1] = pi * ei;
        sh.V[4 * ln + 2] = ycp;
        sh.V[4 * ln + 3] = yv * W.iWi;
    }
    __syncthreads();
    const double q0 = lds_sub(sh.V + 0, 4, 1, NS + 1, 0.0);
    const double d0 = lds_sub(sh.V + 1, 4, 1, NS + 1, 0.0);
    // mix_cv: sum Y_n Cp_n, sum Y_n / W_n, both in species order
    double cv = lds_sum(sh.V + 2, 4, 1, NS + 1, 0.0);
    const double _W = lds_sum(sh.V + 3, 4, 1, NS + 1, 0.0);
    __syncthreads(); // V is written again before the next read
    cv -= Ru * _W;
    const double _Cv = 1.0 / cv;
    qv = ln == 0 ? q0 * _Cv : qi;
    dv = ln == 0 ? d0 * _Cv : pi;
}

// get_Cope at the distributed state (mix_e's order)
template <int NS, int THERMO>
__device__ __forceinline__ double mix_e_wave(const DevThermo *__restrict__ th, WaveLane<NS> &W, WaveShared<NS> &sh,
                                             double yv, double T)
{
    const int ln = threadIdx.x & 63;
    double h;
    if (W.fast && T >= 200.0 && T <= 1.0e5) {
        W.range(th, THERMO ? (T >= 6000.0 ? 2 : (T >= 1000.0 ? 1 : 0)) : (T > 1000.0 ? 0 : 1));
        h = h_fast<THERMO != 0>(FitCol{W.hc}, T, ddiv_core(1.0, T), THERMO ? dlog_pos(T) : 0.0, 1.0);
    } else {
        const TPre t = THERMO ? tpre<true>(T, 1) : tpre<false>(T, 0);
        h = ln >= 1 && ln <= NS ? h_k(th, t, 1.0, ln - 1) : 0.0;
    }
    if (ln >= 1 && ln <= NS) sh.V[ln] = (h - T) * W.Ri * yv;
    __syncthreads();
    const double e = lds_sum(sh.V, 1, 1, NS + 1, 0.0);
    __syncthreads();
    return e;
}

// ChemeODEQ2SolverKernel1 + Chemeq2 for interior cell tl of case cc on one
// wave; every branch below is uniform across the wave
template <int NS, int THERMO>
__device__ __forceinline__ void chem_wave_cell(const DevThermo *__restrict__ th, const DevMech *__restrict__ mc,
                                               const ChemCase &cc, long long tl, int record, int check,
                                               WaveShared<NS> &sh)
{
    constexpr int NL = NS + 1;
    const int ln = threadIdx.x & 63;
    const bool comp = ln < NL;
    const long long N = cc.g.N;
    const long long id = chem_cell_id(cc.g, tl);
    const double rho = cc.U[id];
    const double rho1 = 1.0 / rho;
    const double m_p = cc.p[id];
    const int NR = mc->NR;
    // evalcv's 1 / rho and log(p / p_atm): constants of the cell
    const double _dens = 1.0 / rho;
    const double logP = dlog(m_p * (1.0 / 101325.0));
    // the start values: T, then Getrhoyi's fractions (chem_y0)
    double yv = 0.0;
    if (ln == 0) yv = cc.T[id];
    if (ln >= 1 && ln < NS) yv = cc.g.ghost ? cc.y[(ln - 1) * N + id] : cc.U[(4 + ln) * N + id] * rho1;
    if (cc.g.ghost) {
        if (ln == NS) yv = 0.0;
    } else {
        sh.V[ln] = yv;
        __syncthreads();
        const double rem = lds_sub(sh.V, 1, 1, NS, 1.0); // ((1 - Y_0) - Y_1) - ...
        __syncthreads();
        if (ln == NS) yv = rem;
    }
    WaveLane<NS> W;
    W.load(th, mc, sh, NR, m_p);
    const double e0 = mix_e_wave<NS, THERMO>(th, W, sh, yv, wave_lane(yv, 0));
    // Chemeq2 (ProductionRates.h:488-638), the steps of ChemLane
    const double ymin = 1.0e-20, tfd = 1.0 + 1.0e-10, epscl = 1.0e4;
    const double dtg = cc.dt[DT_CHEM];
    double dt = 0.0, dtmin = 1.0e-7, epsmax = 1.0, ts = 0.0, tn = 0.0;
    double qv = 0.0, dv = 0.0, ys = 0.0, qs = 0.0, ds = 0.0, rtau = 0.0;
    int passes = 0, st = 0;
    bool started = false;
    for (;;) {
        if (!started) {
            if (ln >= 1 && comp) yv = dmax(yv, ymin);
            sh.V[ln] = yv;
            __syncthreads();
            double sumy = lds_sum(sh.V, 1, 1, NL, 0.0);
            __syncthreads();
            sumy = 1.0 / sumy;
            if (ln >= 1 && comp) yv *= sumy;
        } else {
            if (++passes > CHEM_MAXSUB) {
                st = -1;
                break;
            }
            if (comp) {
                const double rt = dt * ds / ys;
                rtau = rt;
                const double alpha = alpha_of(rt);
                const double scr = dt * (qs - ds) / (1.0 + alpha * rt);
                yv = dmax(ys + scr, ymin);
            }
            tn = ts + dt;
        }
        evalcv_wave<NS, THERMO>(th, mc, W, sh, NR, yv, wave_lane(yv, 0), qv, dv, rho, m_p, _dens, logP);
        if (!started) {
            const double epsmin = 1.0e-4, sqreps = 0.05;
            if (comp) {
                const double ascr = fabs(qv);
                const double sb = 0.1 * epsmin * ascr - dv;
                const double scr2 = (sb >= 0.0 ? 1.0 : -1.0) * fabs(1.0 / yv);
                sh.V[4 * ln + 0] = -fabs(ascr - dv) * scr2;
                sh.V[4 * ln + 1] = scr2 * dv;
            }
            __syncthreads();
            double scrtch = 1e-25;
            for (int i = 0; i < NL; i++) scrtch = dmax(sh.V[4 * i], dmax(sh.V[4 * i + 1], scrtch));
            __syncthreads();
            dt = dmin(sqreps / scrtch, dtg);
            dtmin *= dt;
            ts = 0.0, tn = 0.0;
            ys = yv, qs = qv, ds = dv;
            started = true;
            continue;
        }
        // corrector and the error norm (the maximum in component order)
        if (comp) {
            const double yp = yv;
            const double rtaub = 0.5 * (rtau + dt * dv / yp);
            const double alpha = alpha_of(rtaub);
            const double ysi = ys;
            const double qt = (1.0 - alpha) * qs + alpha * qv;
            const double scr = (qt * dt - rtaub * ysi) / (1.0 + alpha * rtaub);
            const double scr2 = dmax(ysi + scr, 0.0);
            double scr1 = fabs(scr2 - yp);
            yv = dmax(scr2, ymin);
            double cand = 0.0, has = 0.0;
            if ((0.25 * (ysi + yv)) > ymin) {
                scr1 = scr1 / yv;
                cand = 0.5 * (scr1 + dmin(fabs(qv - dv) / (qv + dv + 1.0e-30), scr1));
                has = 1.0;
            }
            sh.V[4 * ln + 0] = cand;
            sh.V[4 * ln + 1] = has;
        }
        __syncthreads();
        double eps = 1e-10;
        for (int i = 0; i < NL; i++)
            if (sh.V[4 * i + 1] != 0.0) eps = dmax(sh.V[4 * i], eps);
        __syncthreads();
        eps = eps * epscl;
        if (eps < epsmax) {
            if (dtg <= (tn * tfd)) {
                st = 1;
                break;
            }
        } else {
            tn = ts;
        }
        const double dto = dt;
        double rteps = 0.5 * (eps + 1.0);
        rteps = 0.5 * (rteps + eps / rteps);
        rteps = 0.5 * (rteps + eps / rteps);
        dt = dmin(dt * (1.0 / rteps + 0.005), tfd * (dtg - tn));
        if (eps > epsmax) {
            dt = dmin(dt, 0.34 * dto);
            if (dt <= dtmin) epsmax *= 10.0;
            continue;
        }
        epsmax = 1.0;
        ts = tn;
        ys = yv, qs = qv, ds = dv;
    }
    // write-back (ChemeODEQ2SolverKernel1's tail), the pass count, the checks
    const double e1 = mix_e_wave<NS, THERMO>(th, W, sh, yv, wave_lane(yv, 0));
    bool bad = false;
    if (ln >= 1 && ln < NS) {
        const double v = yv * rho;
        cc.U[(4 + ln) * N + id] = v;
        bad = isnan(v) || isinf(v);
    }
    if (ln == 0) {
        cc.T[id] = yv;
        const double u4 = cc.U[4 * N + id] + (e1 - e0) * rho;
        cc.U[4 * N + id] = u4;
        if (record) cc.substeps[tl] = st < 0 ? -1 : passes;
        bad = rho < 0 || isnan(rho) || isinf(rho) || isnan(u4) || isinf(u4);
        for (int k = 1; k < 4; k++) bad = bad || isnan(cc.U[k * N + id]) || isinf(cc.U[k * N + id]);
    }
    const bool any_bad = __any(bad);
    if (ln == 0) {
        int bits = st < 0 ? EBIT_CHEM : 0;
        if (st < 0) report_cell(cc.err, EBIT_CHEM, id);
        if (check && any_bad) {
            report_cell(cc.err, EBIT_NAN, id);
            bits |= EBIT_NAN;
        }
        if (bits) report_pass(cc.err, bits, 4);
    }
}

// one interior cell per one-wave block; THERMO = the context's fit family.  Three
// waves per SIMD: at 8192 cells and nine species 57 us, two waves 60, four (which
// spill 192 bytes a lane) 67.
template <int NS, int THERMO>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
k_chem_wave(Geom g, const DevThermo *__restrict__ th, const DevMech *__restrict__ mc, Fields f, int record, int check)
{
    const long long tl = blockIdx.x;
    if (tl >= (long long)g.X_inner * g.Y_inner * g.Z_inner) return;
    if (step_halted(f.err, ~CHEM_BITS)) return;
    __shared__ WaveShared<NS> sh;
    chem_wave_cell<NS, THERMO>(th, mc, one_case(g, f).c, tl, record, check, sh);
}

// zero the work-queue counter (a kernel, so the step graph holds no memset)
static __global__ void k_queue_reset(unsigned int *q)
{
    if (threadIdx.x < 4) q[threadIdx.x] = 0u;
}

} // namespace xf
