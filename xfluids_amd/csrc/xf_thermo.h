// Species and mixture thermodynamics on the device (FP64).
//
// Same formulas and association order as the reference's
// src/solver_Ini/Thermo_device.h (NASA-9 three-range and JANAF/NASA-7
// two-range fits, T >= 200 K clamp, linear enthalpy extrapolation below
// 200 K) and src/solver_Ini/Mixing_device.h (mixture sums, damped Newton
// temperature inversion).  Restructured for the GPU: the fit range, 1/T and
// log(T) depend only on T and are evaluated once per temperature instead of
// once per species (identical values), and loops over species are unrolled
// for a compile-time species count NS.
#pragma once
#include <type_traits>
#include "xf_internal.h"
#include "xf_dev_math.h"

namespace xf {

constexpr double OT = 1.0 / 3.0; // _OT, src/include/global_setup.h:35

// Per-temperature quantities shared by all species.
struct TPre {
    double TT;   // unclamped temperature
    double T;    // max(T, 200)
    double iT;   // 1/T
    double lT;   // log(T) (only when requested)
    int r;       // fit range index (Hia[.. * 3 + r], Hc[(r * MAXNS + n) * 9 + ..])
};

template <bool NEED_LOG>
__device__ __forceinline__ TPre tpre(double T0, int thermo)
{
    TPre t;
    t.TT = T0;
    t.T = dmax(T0, 200.0);
    t.iT = 1.0 / t.T;
    t.lT = NEED_LOG ? dlog(t.T) : 0.0;
    if (thermo) {
        // NASA-9: 200-1000 -> 0, 1000-6000 -> 1, >= 6000 -> 2 (Thermo_device.h:15-20)
        t.r = (t.T >= 1000.0 && t.T < 6000.0) ? 1 : ((t.T < 1000.0) ? 0 : ((t.T >= 6000.0) ? 2 : -1));
    } else {
        // JANAF: > 1000 -> 0 (high fit), else 1 (Thermo_device.h:34-37)
        t.r = (t.T > 1000.0) ? 0 : 1;
    }
    return t;
}

// The fit formulas on the nine coefficients c of one fit range of one
// species: Hia[n * 21 + m * 3 + r] (m = 0..6) then Hib[n * 6 + m * 3 + r]
// (m = 0, 1), as the regrouped copy Hc[(r * MAXNS + n) * 9 + ...] holds them.
// c comes from the table (cp_k, h_k, s_k) or from registers a wave loaded
// once (the one-wave-per-cell chemistry): the same expressions either way.

// HeatCapacity_NASA / HeatCapacity_JANAF (Thermo_device.h:10-40)
__device__ __forceinline__ double cp_fit(const double *c, int thermo, const TPre &t, double Ri)
{
    const double T = t.T;
    if (thermo) {
        if (t.r < 0) return 0.0;
        return Ri * ((c[0] * t.iT + c[1]) * t.iT + c[2] + (c[3] + (c[4] + (c[5] + c[6] * T) * T) * T) * T);
    }
    return Ri * (c[0] + (c[1] + (c[2] + (c[3] + c[4] * T) * T) * T) * T);
}

// get_Enthalpy_NASA / get_Enthalpy_JANAF (Thermo_device.h:62-102) without the
// extrapolation below 200 K (h_k adds it)
__device__ __forceinline__ double h_fit(const double *c, int thermo, const TPre &t, double Ri)
{
    const double T = t.T;
    double hi = 0.0;
    if (thermo) {
        if (t.r >= 0)
            hi = Ri * (-c[0] / T + c[1] * t.lT + (c[2] + (0.5 * c[3] + (c[4] * OT + (0.25 * c[5] + 0.2 * c[6] * T) * T) * T) * T) * T +
                       c[7]);
    } else {
        hi = Ri * (T * (c[0] + T * (c[1] * 0.5 + T * (c[2] * OT + T * (c[3] * 0.25 + c[4] * T * 0.2)))) + c[5]);
    }
    return hi;
}

// get_Entropy_NASA / get_Entropy_JANAF (Thermo_device.h:132-161)
__device__ __forceinline__ double s_fit(const double *c, int thermo, const TPre &t, double Ri)
{
    const double T = t.T;
    if (thermo) {
        if (t.r < 0) return 0.0;
        return Ri * ((-0.5 * c[0] * t.iT - c[1]) * t.iT + c[2] * t.lT +
                     (c[3] + (0.5 * c[4] + (c[5] * OT + c[6] * 0.25 * T) * T) * T) * T + c[8]);
    }
    return Ri * (c[0] * t.lT + (c[1] + (0.5 * c[2] + (c[3] * OT + c[4] * 0.25 * T) * T) * T) * T + c[6]);
}

// species n's coefficients of range t.r in the table (range 0 when t.r < 0,
// where the NASA formulas return before reading them)
__device__ __forceinline__ const double *fit_coeffs(const DevThermo *__restrict__ th, int r, int n)
{
    return th->Hc + ((r < 0 ? 0 : r) * MAXNS + n) * 9;
}

__device__ __forceinline__ double cp_k(const DevThermo *__restrict__ th, const TPre &t, double Ri, int n)
{
    return cp_fit(fit_coeffs(th, t.r, n), th->thermo, t, Ri);
}

// Cp of species n at exactly 200 K (used by the low-temperature extrapolation)
__device__ __forceinline__ double cp200_k(const DevThermo *__restrict__ th, double Ri, int n)
{
    TPre t;
    t.TT = 200.0;
    t.T = 200.0;
    t.iT = 1.0 / t.T;
    t.lT = 0.0;
    t.r = th->thermo ? 0 : 1;
    return cp_k(th, t, Ri, n);
}

__device__ __forceinline__ double h_k(const DevThermo *__restrict__ th, const TPre &t, double Ri, int n)
{
    double hi = h_fit(fit_coeffs(th, t.r, n), th->thermo, t, Ri);
    if (t.TT < 200.0) {
        const double Cpi = cp200_k(th, Ri, n);
        hi += Cpi * (t.TT - 200.0);
    }
    return hi;
}

__device__ __forceinline__ double s_k(const DevThermo *__restrict__ th, const TPre &t, double Ri, int n)
{
    return s_fit(fit_coeffs(th, t.r, n), th->thermo, t, Ri);
}

// Table data that no kernel writes, as the compiler's constant address space: a
// read at a wave-uniform address is then a scalar load wherever it stands (the
// compiler drops that for an ordinary pointer once control flow diverges).
typedef const double __attribute__((address_space(4))) cdouble;
__device__ __forceinline__ cdouble *as_const(const double *p) { return (cdouble *)(unsigned long long)p; }
// DevThermo::fast as a scalar load
__device__ __forceinline__ bool table_fast(const DevThermo *__restrict__ th)
{
    return *(const int __attribute__((address_space(4))) *)(unsigned long long)&th->fast != 0;
}

// ---- the fits on a clamped temperature, 200 K <= T <= 1e5 K on every lane of the
// wave (FastT below): the same expressions with the fit family as a constant and one
// exact shortcut.  -c0 / T takes the corrected
// quotient of the shared reciprocal (DevThermo::fast says that every coefficient
// is 0 or within [2^-300, 2^300], so nothing leaves the quotient's range; c0 = 0
// gives a zero, which adds nothing).  No branch on the family, the range or
// T < 200 is left inside the species loops (a wave with colder lanes runs a copy of
// its own, FastT), so the species' chains overlap: a
// Newton iteration at nine species is one basic block instead of some thirty,
// and k_states<9> at 8192 cells (a launch as long as its longest Newton chain)
// went from 44.7 to 24.5 us, on a 128^3 mixing layer from 223 to 181 us.
template <bool NASA, class P> __device__ __forceinline__ double cp_fast(P c, double T, double iT, double Ri)
{
    if (NASA) return Ri * ((c[0] * iT + c[1]) * iT + c[2] + (c[3] + (c[4] + (c[5] + c[6] * T) * T) * T) * T);
    return Ri * (c[0] + (c[1] + (c[2] + (c[3] + c[4] * T) * T) * T) * T);
}
template <bool NASA, class P>
__device__ __forceinline__ double h_fast(P c, double T, double iT, double lT, double Ri)
{
    if (NASA)
        return Ri * (dquot(-c[0], T, iT) + c[1] * lT + (c[2] + (c[9] + (c[10] + (c[11] + c[12] * T) * T) * T) * T) * T +
                     c[7]);
    return Ri * (T * (c[0] + T * (c[9] + T * (c[10] + T * (c[11] + c[4] * T * 0.2)))) + c[5]);
}
template <bool NASA, class P>
__device__ __forceinline__ double s_fast(P c, double T, double iT, double lT)
{
    if (NASA)
        return ((c[13] * iT - c[1]) * iT + c[2] * lT + (c[3] + (c[14] + (c[15] + c[16] * T) * T) * T) * T + c[8]);
    return (c[0] * lT + (c[1] + (c[14] + (c[15] + c[16] * T) * T) * T) * T + c[6]);
}

// The per-temperature values of the fast fits: T = max(T0, 200) and what follows from
// it.  COLD: some lane of the wave is below 200 K.
template <bool COLD> struct FastT {
    static constexpr bool cold = COLD;
    double T0, T, iT, lT;
    // a species' enthalpy h at T as that at T0, by the linear extrapolation below 200 K;
    // Cp its heat capacity at T
    __device__ __forceinline__ double below(double h, double Cp) const
    {
        return COLD && T0 < 200.0 ? h + Cp * (T0 - 200.0) : h;
    }
};
// the highest temperature of the fast fits: 1e5 K, or a NaN, which no temperature is
// below, where the table does not qualify
__device__ __forceinline__ double fast_top(const DevThermo *__restrict__ th)
{
    return th->fast ? 1.0e5 : __longlong_as_double(0x7ff8000000000000LL);
}
template <bool NASA, bool COLD, class F>
__device__ __forceinline__ void fast_ranges(const DevThermo *__restrict__ th, double T0, bool need_log, F body)
{
    FastT<COLD> t;
    t.T0 = T0;
    t.T = COLD ? dmax(T0, 200.0) : T0;
    t.iT = ddiv_core(1.0, t.T);
    t.lT = need_log ? dlog_pos(t.T) : 0.0;
    // the ranges of tpre at T >= 200
    const int r = NASA ? (t.T >= 6000.0 ? 2 : (t.T >= 1000.0 ? 1 : 0)) : (t.T > 1000.0 ? 0 : 1);
#pragma unroll 1
    for (int q = 0; q < (NASA ? 3 : 2); q++) {
        int ru = q; // hidden from the compiler, which would put r for q in the address
        asm volatile("" : "+s"(ru));
        if (r == q) body(as_const(th->Hf + ru * (MAXNS * FITC)), t);
    }
}
// body(c, t) with the coefficients of the lane's fit range at c + FITC * species, c the
// same on every lane that runs it together (scalar loads shared by the wave): once for a
// wave in one range, once per range for a wave that straddles a limit.  False, with
// nothing run, unless every active lane with run set has T <= top (fast_top, read once
// by the caller).  The body is there twice, so that a wave at 200 K and above, the usual
// one, spends nothing on colder ones.  With a loop over the species and vector loads of
// the coefficients for the colder ones k_states took 438 us on a stream of 150 K at 64^3
// and nine species (126 now), and a Reaction of one pass a cell 216 (89 now).
template <bool NASA, class F>
__device__ __forceinline__ bool fast_fits(const DevThermo *__restrict__ th, double top, double T, bool run,
                                          bool need_log, F body)
{
    if (__builtin_expect(__all(!run || (T >= 200.0 && T <= top)), 1)) {
        fast_ranges<NASA, false>(th, T, need_log, body);
        return true;
    }
    if (!__all(!run || T <= top)) return false;
    fast_ranges<NASA, true>(th, T, need_log, body);
    return true;
}

// get_CopR (Mixing_device.h:49-56)
template <int NS>
__device__ __forceinline__ double mix_R(const DevThermo *__restrict__ th, const double *yi)
{
    double R = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) R += yi[n] * th->_Wi[n];
    return R * Ru;
}

// get_CopCp (Mixing_device.h:61-68)
template <int NS>
__device__ __forceinline__ double mix_cp(const DevThermo *__restrict__ th, const double *yi, const TPre &t)
{
    double cp = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) cp += yi[n] * cp_k(th, t, th->Ri[n], n);
    return cp;
}

// get_CopCv (Mixing_device.h:73-86)
template <int NS>
__device__ __forceinline__ double mix_cv(const DevThermo *__restrict__ th, const double *yi, const TPre &t)
{
    double cv = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) cv += yi[n] * cp_k(th, t, th->Ri[n], n);
    double _W = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) _W += yi[n] * th->_Wi[n];
    cv -= Ru * _W;
    return cv;
}

// get_CopGamma(thermal, yi, Cp, T) (Mixing_device.h:114-126)
template <int NS>
__device__ __forceinline__ double mix_gamma_cp(const DevThermo *__restrict__ th, const double *yi, double Cp)
{
    double _W = 0.0;
#pragma unroll
    for (int n = 0; n < NS; n++) _W += yi[n] * th->_Wi[n];
    const double CopW = 1.0 / _W;
    const double g = Cp / (Cp - Ru / CopW);
    return (g > 1.0) ? g : -1.0;
}

// sub_FuncT + get_T (Mixing_device.h:159-193).  R = get_CopR is loop
// invariant and hoisted (same value every iteration).  A launch on few cells
// lasts as long as its longest Newton chain (the step of T is limited, so a cell
// behind a shock takes tens of iterations), a launch on many is bound by the
// FP64 issue of the sums; the fast fits shorten both.  With the products of the
// coefficients and the fits' constants in the table k_states takes 61 us instead of
// 63 at 80 x 40 x 40 and five species, and with converged lanes kept on 54; at
// 60 x 40 x 36 52 instead of 63.
//
// The step of T from the sums
__device__ __forceinline__ double newton_step(double h, double Cp, double R, double T, double e)
{
    const double func_T = h - R * T - e;
    const double dfunc_T = Cp - R;
    double df = dmin(func_T / (dfunc_T + 1.0e-30), 1e-3 * T);
    df = dmax(df, -1e-2 * T);
    return df;
}

// The last few chains of a wave, a group of lanes per cell and a species per lane: the
// terms of the sums side by side, added in the species' order on every lane.  A wave
// that is nearly alone on its SIMD waits some ten cycles for each instruction, so a
// chain is as long as its instructions: with the tail k_states at 80 x 40 x 40 and five
// species takes 45.5 us instead of 54.3, at 8192 cells and nine species 16.7 instead of
// 20.0.  Blocks of 256 lanes.
template <int NS> struct NewtonTail {
    static constexpr int L = NS > 8 ? 16 : 8; // lanes per cell
    static constexpr int CELLS = 64 / L;
    static constexpr int FROM = 4; // iterations before it: shorter chains end sooner without
    struct Shared {
        double y[4][CELLS * L];   // mass fractions of the groups' cells
        double2 x[4][64];         // a species' terms of h and Cp
    };
};
// runs the cells of the lanes in `left` (at most CELLS, every lane of the wave active)
// from iteration it on, until each has converged or one leaves the interval of the
// straight-line fits or falls below 200 K; returns the iteration reached
template <int NS, bool NASA>
__device__ __forceinline__ int newton_tail(const DevThermo *__restrict__ th, typename NewtonTail<NS>::Shared &sh,
                                           const double *yi, double e, double R, unsigned long long left, int it,
                                           double &T, double &root, bool &run)
{
    using TL = NewtonTail<NS>;
    constexpr int L = TL::L;
    static_assert(NS <= L, "a lane per species");
    const int lane = threadIdx.x & 63, wv = (threadIdx.x >> 6) & 3;
    const int rank = __popcll(left & ((1ull << lane) - 1ull)); // of a running lane's cell
    auto order = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // group g takes the g-th running lane (groups without one the last)
    const int g = lane / L, n = lane % L, cells = __popcll(left);
    int owner = 0;
    {
        unsigned long long m = left;
        for (int k = 0; k < TL::CELLS; k++) {
            const int l = __ffsll((long long)m) - 1;
            if (k <= g && l >= 0) owner = l;
            m &= m - 1;
        }
    }
    if (run) {
#pragma unroll
        for (int k = 0; k < NS; k++) sh.y[wv][rank * L + k] = yi[k];
    }
    order();
    const int cell = min(g, cells - 1);
    const double y = n < NS ? sh.y[wv][cell * L + n] : 0.0;
    const double Ri = n < NS ? th->Ri[n] : 0.0, eg = __shfl(e, owner), Rg = __shfl(R, owner);
    double Tg = __shfl(T, owner), rg = Tg;
    bool go = true;
    int range = -1;
    double c[13];
    for (; it < 101; it++) {
        if (!__all(!go || (Tg >= 200.0 && Tg <= 1.0e5))) break;
        const int r = NASA ? (Tg >= 6000.0 ? 2 : (Tg >= 1000.0 ? 1 : 0)) : (Tg > 1000.0 ? 0 : 1);
        if (__any(r != range)) {
            range = r;
            const double *p = th->Hf + (r * MAXNS + (n < NS ? n : 0)) * FITC;
#pragma unroll
            for (int m = 0; m < 13; m++) c[m] = p[m];
        }
        const double iT = ddiv_core(1.0, Tg), lT = NASA ? dlog_pos(Tg) : 0.0;
        sh.x[wv][lane] = make_double2(h_fast<NASA>((const double *)c, Tg, iT, lT, Ri) * y,
                                      y * cp_fast<NASA>((const double *)c, Tg, iT, Ri));
        order();
        double h = 0.0, Cp = 0.0;
#pragma unroll
        for (int k = 0; k < NS; k++) {
            const double2 x = sh.x[wv][g * L + k];
            h += x.x;
            Cp += x.y;
        }
        order();
        const double df = newton_step(h, Cp, Rg, Tg, eg);
        Tg = Tg - df;
        rg = go ? Tg : rg;
        go = go && !(fabs(df) <= 1.0e-6);
        if (!__any(go)) {
            it++;
            break;
        }
    }
    // back to the cells' lanes
    const double Tb = __shfl(rg, (rank * L) & 63);
    const int gb = __shfl(go ? 1 : 0, (rank * L) & 63);
    if (run) T = Tb, root = Tb, run = gb != 0;
    return it;
}

template <int NS, bool NASA, bool TAIL>
__device__ __forceinline__ double get_T_fam(const DevThermo *__restrict__ th, const double *yi, double e, double T0,
                                            typename NewtonTail<NS>::Shared *sh)
{
    double T = T0, root = T0;
    const double R = mix_R<NS>(th, yi);
    const double top = fast_top(th);
    cdouble *Rk = as_const(th->Ri);
    bool run = true;
    double h, Cp;
    auto sums = [&](cdouble *c, auto t) {
#pragma unroll
        for (int n = 0; n < NS; n++) {
            const double Ri = Rk[n], Cpn = cp_fast<NASA>(c + FITC * n, t.T, t.iT, Ri);
            h += t.below(h_fast<NASA>(c + FITC * n, t.T, t.iT, t.lT, Ri), Cpn) * yi[n];
            Cp += yi[n] * Cpn;
        }
    };
    // the step of T from the sums; the lanes that go on
    auto step = [&]() {
        const double df = newton_step(h, Cp, R, T, e);
        T = T - df;
        root = run ? T : root;
        run = run && !(fabs(df) <= 1.0e-6);
        return (unsigned long long)__ballot(run);
    };
    // a lane that has converged goes on about its root, past the result: with the last
    // few cells alone active a wave runs at half speed on an otherwise idle chip
    int it = 1;
    for (; it < 101 && __all(!run || (T >= 200.0 && T <= top)); it++) {
        h = 0.0, Cp = 0.0;
        fast_ranges<NASA, false>(th, T, NASA, sums);
        const unsigned long long left = step();
        if (!left) return root;
        if constexpr (TAIL) {
            if (it >= NewtonTail<NS>::FROM && __popcll(left) <= NewtonTail<NS>::CELLS && __ballot(1) == ~0ull &&
                __all(!run || (T >= 200.0 && T <= top))) {
                it = newton_tail<NS, NASA>(th, *sh, yi, e, R, left, it + 1, T, root, run) - 1;
                if (!__any(run)) return root;
            }
        }
    }
    // a loop of its own from the first lane below 200 K (or above the fits' interval) on,
    // so that the usual waves' stays short
    for (; it < 101; it++) {
        h = 0.0, Cp = 0.0;
        if (__all(!run || T <= top)) {
            fast_ranges<NASA, true>(th, T, NASA, sums);
        } else {
            const TPre t = tpre<NASA>(T, NASA ? 1 : 0);
#pragma unroll 1
            for (int n = 0; n < NS; n++) {
                double y = yi[0];
#pragma unroll
                for (int q = 1; q < NS; q++) y = q == n ? yi[q] : y;
                h += h_k(th, t, th->Ri[n], n) * y;
                Cp += y * cp_k(th, t, th->Ri[n], n);
            }
        }
        if (!step()) break;
    }
    return root;
}
template <int NS, bool TAIL>
__device__ __forceinline__ double get_T(const DevThermo *__restrict__ th, const double *yi, double e, double T0)
{
    typename NewtonTail<NS>::Shared *sh = nullptr;
    if constexpr (TAIL) {
        __shared__ typename NewtonTail<NS>::Shared s;
        sh = &s;
    }
    return th->thermo ? get_T_fam<NS, true, TAIL>(th, yi, e, T0, sh) : get_T_fam<NS, false, TAIL>(th, yi, e, T0, sh);
}

} // namespace xf
