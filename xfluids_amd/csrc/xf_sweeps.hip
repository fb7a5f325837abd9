// Sweep kernels of one species count and scheme, every direction, precision form
// and tile shape, and their launches (SweepLaunch, xf_context.h).  Compiled with
// -DXF_NS=<species> -DXF_SCH=<scheme> for every pair the library has.
#include "xf_context.h"

namespace xf {

template <int NS, bool COP, int SCH> struct SweepKernels {
    template <int DIR, int PREC, int SHAPE>
    static void one_t(xf_ctx *c, const double *Ug, int mode, int stage, const double *Ua, const double *Ub, double *Uo)
    {
        constexpr int E = COP ? NS + 4 : 5;
        static_assert(SweepShape<DIR, E, SHAPE>::TS == (DIR == 0 ? (SHAPE == 0 ? 64 : 32)
                                                                 : (SHAPE == 0 ? 16 : (SHAPE == 1 ? 32 : 8))),
                      "tile_faces");
        unsigned gr[5];
        sweep_grid(c->g, DIR, SHAPE, tile_blocks(c->g, DIR, SHAPE), gr);
        static const char *names[3] = {"sweep_x", "sweep_y", "sweep_z"};
        ProfScope ps(c, names[DIR]);
        hipLaunchKernelGGL((k_sweep<NS, COP, DIR, SCH, PREC, SHAPE>), dim3(gr[0], gr[1], gr[2]), dim3(256), 0, c->stream,
                           c->g, c->d_th, Ug, c->f, c->d.ncop_gamma, mode, stage, Ua, Ub, Uo, (int)gr[3], (int)gr[4]);
    }
    template <int DIR, int PREC, int SHAPE>
    static void multi_t(const xf_ctx *c0, hipStream_t st, const EnsCase *cases, int ncases, long long blocks, int mode,
                        int stage, int sg, int sa, int sb, int so)
    {
        hipLaunchKernelGGL((k_sweep_multi<NS, COP, DIR, SCH, PREC, SHAPE>), dim3((unsigned)blocks), dim3(256), 0, st,
                           cases, ncases, c0->d_th, c0->d.ncop_gamma, mode, stage, sg, sa, sb, so);
    }
    // f(DIR, PREC, SHAPE as integral constants) for the run-time values
    template <int DIR, int PREC, class F> static void on_shape(int shape, F f)
    {
        using std::integral_constant;
        constexpr integral_constant<int, DIR> d{};
        constexpr integral_constant<int, PREC> p{};
        if (SweepShapes<DIR>::count > 2 && shape == 2)
            f(d, p, integral_constant<int, (SweepShapes<DIR>::count > 2 ? 2 : 0)>{});
        else if (shape == 1)
            f(d, p, integral_constant<int, 1>{});
        else
            f(d, p, integral_constant<int, 0>{});
    }
    template <int DIR, class F> static void on_precision(int prec, int shape, F f)
    {
        if (prec == XF_MIXED) on_shape<DIR, XF_MIXED>(shape, f);
        else if (prec == XF_FUSED_FP64) on_shape<DIR, XF_FUSED_FP64>(shape, f);
        else on_shape<DIR, XF_PLAIN_FP64>(shape, f);
    }
    template <class F> static void on(int dir, int prec, int shape, F f)
    {
        if (dir == 0) on_precision<0>(prec, shape, f);
        if (dir == 1) on_precision<1>(prec, shape, f);
        if (dir == 2) on_precision<2>(prec, shape, f);
    }
};

template <int NS, bool COP, int SCH>
void SweepLaunch<NS, COP, SCH>::sweep(xf_ctx *c, int dir, const double *Ug, int mode, int stage, const double *Ua,
                                      const double *Ub, double *Uo)
{
    using K = SweepKernels<NS, COP, SCH>;
    K::on(dir, c->d.precision, c->shape[dir], [&](auto d, auto p, auto s) {
        K::template one_t<d(), p(), s()>(c, Ug, mode, stage, Ua, Ub, Uo);
    });
}

template <int NS, bool COP, int SCH>
void SweepLaunch<NS, COP, SCH>::multi(const xf_ctx *c0, hipStream_t st, const EnsCase *cases, int ncases,
                                      long long blocks, int dir, int shape, int mode, int stage, int sg, int sa, int sb,
                                      int so)
{
    using K = SweepKernels<NS, COP, SCH>;
    K::on(dir, c0->d.precision, shape, [&](auto d, auto p, auto s) {
        K::template multi_t<d(), p(), s()>(c0, st, cases, ncases, blocks, mode, stage, sg, sa, sb, so);
    });
}

template struct SweepLaunch<XF_NS, (XF_NS > 1), XF_SCH>;

} // namespace xf
