// Context of one case and the per-species-count kernel dispatch table,
// shared by the C-ABI translation unit (xf_api.hip) and the translation units
// that instantiate the kernels for each compile-time species count
// (xf_ops_ns*.hip, and xf_sweeps.hip per count and scheme), so that those compile
// in parallel.
#pragma once
#include "xf_sweep_kernels.h"
#include "xf_chem_kernels.h"
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <vector>

using namespace xf;

namespace xf {

struct EvPair {
    const char *name;
    hipEvent_t a, b;
};

struct Ops {
    // UpdateStates on U; bcs != 0 (packed BC codes) also fills the ghost cells;
    // where: the stage a failure is reported in (1..3 RK stage, 4 Reaction)
    void (*states)(xf_ctx *, double *U, int full, int bcs, int where);
    void (*sweep)(xf_ctx *, int dir, const double *Ug, int mode, int stage, const double *Ua, const double *Ub,
                  double *Uo);
    // check = 1: the post-Reaction NaN check of a time step on each cell
    void (*chem)(xf_ctx *, int record, int check);
    void (*prepare)(xf_ctx *);
    // shared queue over the cells of several cases (ensembles)
    // spec: compiled mechanism whose records the tables hold, or -1
    void (*chem_multi)(hipStream_t, const ChemCase *, int ncases, long long total, const DevThermo *,
                       const DevMech *, unsigned long long *queue, int blocks, int record, int check, int spec,
                       void *spill, int spill_cap, int spill_after);
    // bytes of one hand-over record (ChemSpill<NS>)
    size_t (*spill_bytes)();
    int (*multi_blocks)(long long total, int spec);
    // viscous terms of GetLU: transport coefficients and centre gradients of
    // the state Ug, then the wall flux of one direction (before its sweep)
    void (*visc_prep)(xf_ctx *, const double *Ug);
    void (*visc_flux)(xf_ctx *, int dir, const double *Ug);
    // one launch over every case of an ensemble (case table on the device;
    // sel codes pick U, U1 or U2 per case; the scheme and precision are those of
    // the template case c0)
    // fold: some case's blocks are too many for the sweeps to fold
    void (*states_multi)(const xf_ctx *c0, hipStream_t, const EnsCase *, int ncases, long long blocks, int full,
                         int fill, int where, int sel, bool fold);
    void (*sweep_multi)(const xf_ctx *c0, hipStream_t, const EnsCase *, int ncases, long long blocks, int dir, int shape,
                        int mode, int stage, int sel_g, int sel_a, int sel_b, int sel_o);
    // the sweeps compute the wall flux themselves when Geom::visc_fused is set
    bool visc_in_sweep;
};

// dispatch tables, one translation unit each
Ops ops_ns1();
Ops ops_ns2();
Ops ops_ns3();
Ops ops_ns4();
Ops ops_ns5();
Ops ops_ns9();
Ops ops_ns10();
Ops ops_ns11();

} // namespace xf

struct xf_ctx {
    xf_case_desc d;
    Geom g;
    int E, NCOP;
    long long N, Ninner;
    hipStream_t stream = nullptr;
    Fields f{};
    double *U2 = nullptr; // RK stage-2 output of the fused path
    double *xbuf = nullptr; // cells in the host's order on their way in or out (xf_upload_state)
    DevThermo h_th{};
    DevThermo *d_th = nullptr;
    DevMech h_mc{};
    DevMech *d_mc = nullptr;
    DevTransport *d_tr = nullptr;
    bool thermo_set = false, mech_set = false, transport_set = false;
    Ops ops{};
    bool has_ops = false;
    int chem_blocks = 0; // resident one-wave blocks of the work-queue chemistry kernel
    // cells the queue hands to whole waves after spill_after passes (at most
    // spill_cap of them per launch; 0 = never).  Switched off: the one run of
    // the hand-over on the GPU did not finish and no cause has been shown, so
    // xf_set_chem_handover refuses any other value and nothing is allocated.
    void *spill = nullptr;
    int spill_cap = 0, spill_after = 0;
    // compiled mechanism the device tables match (MechSpec<mech_spec>), or -1;
    // spec_allowed = false keeps the generic loop (xf_set_chem_specialization)
    int mech_spec = -1;
    bool spec_allowed = true;
    int shape[3] = {0, 0, 0}; // sweep tile shape per direction (SweepShape)
    bool shape_set[3] = {false, false, false}; // chosen by the caller or the autotuner
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int last_code = 0, last_id = -1;
    int last_step = 0, last_where = 0; // step (Iteration) and stage of the last failure
    int step_count = 0, target_reached = 0; // device clock as of the last error read
    bool prof = false;
    std::string prof_filter; // ",name,name," or empty for all
    std::vector<EvPair> evs;
    std::map<std::string, std::pair<double, int>> times;
};

#define XF_HIP(call)                                                                                                   \
    do {                                                                                                               \
        hipError_t e_ = (call);                                                                                        \
        if (e_ != hipSuccess) {                                                                                        \
            fprintf(stderr, "xfluids_amd: HIP error %s at %s:%d\n", hipGetErrorString(e_), __FILE__, __LINE__);       \
            return XF_EHIP;                                                                                            \
        }                                                                                                              \
    } while (0)

namespace xf {

inline unsigned nblk(long long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// faces along the sweep of a tile of shape `shape` in direction dir (the shapes of
// SweepShape); it has 256 / that many pencils
inline int tile_faces(int dir, int shape)
{
    return dir == 0 ? (shape == 0 ? 64 : 32) : (shape == 0 ? 16 : (shape == 1 ? 32 : 8));
}

// tile grid of a sweep in direction dir with tile shape `shape` (TS faces by
// TW = 256 / TS pencils): x tiles along the sweep axis of x, pencil rows, third axis;
// then the cells a tile covers along the sweep and (y, z) its columns.  launch: the
// blocks of the whole launch (tile_blocks, over all cases of an ensemble).  As a rule
// a direction takes full tiles and a remainder.  Its cells are spread evenly over the
// same number of tiles instead where that would leave waves with a few active lanes:
// those run at half speed or less.  Along the sweep when the remainder is at most
// TS / 16 cells (64 cells in x as 63 + 1 took 129 us at 64^3 and nine species, as
// 32 + 32 110), and in every launch of under two blocks per CU (one species: 15.2 us
// at 64^2 and 65^2, 7.8 at 63^2; evenly 7.8 at each).  With fuller remainders even
// tiles cost 1-2 %, and even columns, whose rows then straddle cache lines, up to 5 %.
inline void sweep_grid(const Geom &g, int dir, int shape, long long launch, unsigned out[5])
{
    const int TS = tile_faces(dir, shape), TW = 256 / TS;
    // (0 tiles of no cells, where a direction has none: the launch then fails)
    auto tiles = [](int n, int most) { return most > 0 ? (unsigned)((n + most - 1) / most) : 0u; };
    const int inner = dir == 0 ? g.X_inner : (dir == 1 ? g.Y_inner : g.Z_inner);
    const unsigned along = tiles(inner, TS - 1), across = tiles(dir == 0 ? g.Y_inner * g.Z_inner : g.X_inner, TW);
    out[0] = dir == 0 ? along : across;
    out[1] = dir == 0 ? across : along;
    out[2] = dir == 0 ? 1 : (unsigned)(dir == 1 ? g.Z_inner : g.Y_inner);
    const bool small = launch < 512;
    const int rest = inner - (int)(along - 1) * (TS - 1);
    out[3] = small || rest <= TS / 16 ? tiles(inner, (int)along) : TS - 1;
    out[4] = small && dir != 0 ? tiles(g.X_inner, (int)across) : TW;
}
// its blocks, which do not depend on the launch's
inline long long tile_blocks(const Geom &g, int dir, int shape)
{
    unsigned gr[5];
    sweep_grid(g, dir, shape, 0, gr);
    return (long long)gr[0] * gr[1] * gr[2];
}

// The tile shape a context or an ensemble starts with (xf_set_tile_shape and
// xf_autotune change it): the one with the fewest blocks, blocks(shape) those of its
// launch, since every block runs the same instructions whatever part of its lanes has
// a face; ties take the lower number.  8 x 32 tiles in y and z stage 13 cells for every
// 7 they finish and must save more than a quarter of the blocks.  Measured at nine
// species (x 64 x 4 / 32 x 8): 128^3 624 / 544 us with 12288 / 10240 blocks, 64^3 130 /
// 84 with 2048 / 1536, 100^3 289 / 281 with 5000 each; y (16 x 16 / 32 x 8 / 8 x 32):
// 128^3 541 / 578 / 852 with 9216 / 10240 / 9728; three species at 97 x 48 x 48 50.8 /
// 43.7 / 59.6 with 1344 / 1248 / 1344.  Where 8 x 32 tiles save a quarter (64 cases of
// 128 x 16, y 16 x 16 / 8 x 32, microseconds a step): one species 289 / 285, three 427 /
// 406, nine 1089 / 1104; where they save nothing (nine cases of 256 x 256) 377 / 386, 651 /
// 655 and 2122 / 2298.  An ensemble of a 64 x 7 and eight 256 x 256
// channels: 2122 us a step with the shapes of all its cases (x 32 x 8, y 16 x 16), 2284
// with those of the first one alone (y 8 x 32).
template <class F> int fewest_blocks(int dir, F blocks)
{
    double best = 0.0;
    int shape = 0;
    for (int s = 0; s < (dir == 0 ? 2 : 3); s++) {
        const double cost = (double)blocks(s) * (s == 2 ? 1.35 : 1.0);
        if (s == 0 || cost < best) best = cost, shape = s;
    }
    return shape;
}

struct ProfScope {
    xf_ctx *c;
    const char *name;
    hipEvent_t a{}, b{};
    bool on;
    ProfScope(xf_ctx *c_, const char *n) : c(c_), name(n)
    {
        on = c->prof && (c->prof_filter.empty() || c->prof_filter.find("," + std::string(n) + ",") != std::string::npos);
        if (on) {
            (void)hipEventCreate(&a);
            (void)hipEventCreate(&b);
            (void)hipEventRecord(a, c->stream);
        }
    }
    ~ProfScope()
    {
        if (on) {
            (void)hipEventRecord(b, c->stream);
            c->evs.push_back({name, a, b});
        }
    }
};

// Launches of the sweeps of one species count and scheme (every direction,
// precision form and tile shape): defined in xf_sweeps.hip, which the build
// compiles once per pair, so that the many instances compile in parallel
template <int NS, bool COP, int SCH> struct SweepLaunch {
    static void sweep(xf_ctx *c, int dir, const double *Ug, int mode, int stage, const double *Ua, const double *Ub,
                      double *Uo);
    static void multi(const xf_ctx *c0, hipStream_t st, const EnsCase *cases, int ncases, long long blocks, int dir,
                      int shape, int mode, int stage, int sg, int sa, int sb, int so);
};

template <int NS, bool COP> struct Launch {
    static void states(xf_ctx *c, double *U, int full, int bcs, int where)
    {
        ProfScope ps(c, "states");
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(nblk(c->N)), dim3(256), 0, c->stream, c->g, c->d_th, U, c->f,
                               c->d.ncop_gamma, full, bcs, where);
        };
        if (COP && nblk(c->N) <= STATES_TAIL) launch(k_states<NS, COP, COP>);
        else launch(k_states<NS, COP, false>);
        if constexpr (COP) {
            if (c->g.ghost)
                hipLaunchKernelGGL((k_rhoyi_writeback<NS>), dim3(nblk(c->N)), dim3(256), 0, c->stream, c->g, U,
                                   c->f);
        }
        if (state_blocks(c->g) > FOLD_BLOCKS)
            hipLaunchKernelGGL(k_states_fold, dim3(12), dim3(1024), 0, c->stream, c->f.spart, state_blocks(c->g),
                               c->f.red, c->f.err);
    }
    static void sweep(xf_ctx *c, int dir, const double *Ug, int mode, int stage, const double *Ua, const double *Ub,
                      double *Uo)
    {
        if (c->d.scheme == XF_WENO5Z) SweepLaunch<NS, COP, XF_WENO5Z>::sweep(c, dir, Ug, mode, stage, Ua, Ub, Uo);
        else if (c->d.scheme == XF_WENOCU6) SweepLaunch<NS, COP, XF_WENOCU6>::sweep(c, dir, Ug, mode, stage, Ua, Ub, Uo);
        else SweepLaunch<NS, COP, XF_WENO5JS>::sweep(c, dir, Ug, mode, stage, Ua, Ub, Uo);
    }
    // calls f(std::integral_constant<int, K>) for the compiled mechanism K
    // == spec if one exists for this species count, else with K = -1 (the
    // generic loop over the device tables)
    template <int K, class F> static void spec_switch(int spec, F &f)
    {
        if constexpr (K < XF_NMECH_SPEC) {
            if constexpr (COP && MechSpec<K>::NS == NS) {
                if (spec == K) {
                    f(std::integral_constant<int, K>{});
                    return;
                }
            }
            spec_switch<K + 1>(spec, f);
        } else {
            f(std::integral_constant<int, -1>{});
        }
    }
    static void chem(xf_ctx *c, int record, int check)
    {
        if constexpr (COP) {
            ProfScope ps(c, "chem");
            auto launch = [&](auto K) {
                constexpr int S = decltype(K)::value;
                if (c->d.chem_driver == XF_CHEM_QUEUE) {
                    const int cap = c->spill_after > 0 ? c->spill_cap : 0;
                    hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(64), 0, c->stream, c->f.queue);
                    hipLaunchKernelGGL((k_chem_queue<NS, S>), dim3(c->chem_blocks), dim3(64), 0, c->stream, c->g,
                                       c->d_th, c->d_mc, c->f, record, check, c->spill, cap, c->spill_after);
                    if (cap > 0)
                        hipLaunchKernelGGL((k_chem_coop<NS>), dim3(coop_blocks(cap)), dim3(64), 0, c->stream, c->g,
                                           c->d_th, c->d_mc, c->f, record, check, c->spill, cap);
                } else if (c->d.chem_driver == XF_CHEM_WAVE) {
                    if (c->d.thermo)
                        hipLaunchKernelGGL((k_chem_wave<NS, 1>), dim3((unsigned)c->Ninner), dim3(64), 0, c->stream,
                                           c->g, c->d_th, c->d_mc, c->f, record, check);
                    else
                        hipLaunchKernelGGL((k_chem_wave<NS, 0>), dim3((unsigned)c->Ninner), dim3(64), 0, c->stream,
                                           c->g, c->d_th, c->d_mc, c->f, record, check);
                } else {
                    hipLaunchKernelGGL((k_chem<NS, S>), dim3(nblk(c->Ninner, 64)), dim3(64), 0, c->stream, c->g,
                                       c->d_th, c->d_mc, c->f, record, check);
                }
            };
            spec_switch<0>(c->mech_spec, launch);
        }
    }
    // persistent lanes of the queue driver: as many one-wave blocks as stay
    // resident, never more than the cells need (queried outside any stream
    // capture, again once the mechanism has picked the kernel)
    static void prepare(xf_ctx *c)
    {
        if constexpr (COP) {
            int per_cu = 0, ncu = 0, dev = 0;
            (void)hipGetDevice(&dev);
            (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
            auto query = [&](auto K) {
                constexpr int S = decltype(K)::value;
                (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_chem_queue<NS, S>, 64, 0);
            };
            spec_switch<0>(c->mech_spec, query);
            const long long want = (c->Ninner + 63) / 64;
            const long long nb = (long long)std::max(per_cu, 1) * std::max(ncu, 1);
            c->chem_blocks = (int)std::max(1LL, std::min(nb, want));
        }
    }
    static void chem_multi(hipStream_t st, const ChemCase *cases, int ncases, long long total, const DevThermo *th,
                           const DevMech *mc, unsigned long long *queue, int blocks, int record, int check, int spec,
                           void *spill, int spill_cap, int spill_after)
    {
        if constexpr (COP) {
            const int cap = spill_after > 0 ? spill_cap : 0;
            auto launch = [&](auto K) {
                constexpr int S = decltype(K)::value;
                hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(64), 0, st, (unsigned int *)queue);
                hipLaunchKernelGGL((k_chem_queue_multi<NS, S>), dim3(blocks), dim3(64), 0, st, cases, ncases, total,
                                   th, mc, queue, record, check, spill, cap, spill_after);
            };
            spec_switch<0>(spec, launch);
            if (cap > 0)
                hipLaunchKernelGGL((k_chem_coop_multi<NS>), dim3(coop_blocks(cap)), dim3(64), 0, st, cases, ncases, th,
                                   mc, queue, record, check, spill, cap);
        }
    }
    // persistent one-wave blocks of the hand-over kernel: a wave per cell
    // while the list lasts, no more than 2048
    static unsigned coop_blocks(int cap) { return (unsigned)std::min(cap, 2048); }
    static size_t spill_bytes() { return COP ? sizeof(ChemSpill<NS>) : 0; }
    static int multi_blocks(long long total, int spec)
    {
        int per_cu = 0, ncu = 0, dev = 0;
        if constexpr (COP) {
            (void)hipGetDevice(&dev);
            (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
            auto query = [&](auto K) {
                constexpr int S = decltype(K)::value;
                (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_chem_queue_multi<NS, S>,
                                                                   64, 0);
            };
            spec_switch<0>(spec, query);
        }
        const long long want = (total + 63) / 64;
        const long long nb = (long long)std::max(per_cu, 1) * std::max(ncu, 1);
        return (int)std::max(1LL, std::min(nb, want));
    }
    static void visc_prep(xf_ctx *c, const double *Ug)
    {
        if constexpr (COP) {
            ProfScope ps(c, "visc_prep");
            const Geom &g = c->g;
            if (c->d.precision == XF_MIXED)
                hipLaunchKernelGGL((k_transport<NS, 1>), dim3(nblk(c->N)), dim3(256), 0, c->stream, g, c->d_th,
                                   c->d_tr, Ug, c->f, c->d.visc_heat, c->d.visc_diffu);
            else
                hipLaunchKernelGGL((k_transport<NS, 0>), dim3(nblk(c->N)), dim3(256), 0, c->stream, g, c->d_th,
                                   c->d_tr, Ug, c->f, c->d.visc_heat, c->d.visc_diffu);
            const int i0 = g.DimX ? g.Bx - 2 : 0, nx = g.DimX ? g.X_inner + 4 : 1;
            const int j0 = g.DimY ? g.By - 2 : 0, ny = g.DimY ? g.Y_inner + 4 : 1;
            const int k0 = g.DimZ ? g.Bz - 2 : 0, nz = g.DimZ ? g.Z_inner + 4 : 1;
            const int *bc = c->d.BC;
            // the mixed form stores the gradients (and the transport
            // coefficients) as FP32 planes
            const int ns = c->d.visc_diffu ? NS : 0;
            const unsigned blocks = nblk((long long)nx * ny * nz) + 2u * ns;
            auto deriv = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, c->stream, g, c->f, i0, nx, j0, ny, k0, nz, bc[0],
                                   bc[1], bc[2], bc[3], bc[4], bc[5], ns, (int)nblk(c->N));
            };
            if (c->d.precision == XF_MIXED) deriv(k_vel_deriv<XF_MIXED>);
            else deriv(k_vel_deriv<XF_PLAIN_FP64>);
        }
    }
    template <int DIR> static void visc_flux_d(xf_ctx *c, const double *Ug)
    {
        const Geom &g = c->g;
        const long long plane = (long long)(g.X_inner + (DIR == 0)) * (g.Y_inner + (DIR == 1));
        const long long nz = g.Z_inner + (DIR == 2);
        // z: (chunks of 256 faces of a plane) x (face planes), as the kernel maps them
        const unsigned blocks = DIR == 2 ? nblk(plane) * (unsigned)nz : nblk(plane * nz);
        static const char *names[3] = {"visc_x", "visc_y", "visc_z"};
        ProfScope ps(c, names[DIR]);
        if (c->d.precision == XF_MIXED)
            hipLaunchKernelGGL((k_visc_flux<NS, DIR, XF_MIXED>), dim3(blocks), dim3(256), 0, c->stream, g, Ug, c->f);
        else
            hipLaunchKernelGGL((k_visc_flux<NS, DIR, XF_PLAIN_FP64>), dim3(blocks), dim3(256), 0, c->stream, g, Ug,
                               c->f);
    }
    static void visc_flux(xf_ctx *c, int dir, const double *Ug)
    {
        if constexpr (COP) {
            if (dir == 0) visc_flux_d<0>(c, Ug);
            if (dir == 1) visc_flux_d<1>(c, Ug);
            if (dir == 2) visc_flux_d<2>(c, Ug);
        }
    }
    static void states_multi(const xf_ctx *c0, hipStream_t st, const EnsCase *cases, int ncases, long long blocks,
                             int full, int fill, int where, int sel, bool fold)
    {
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, st, cases, ncases, c0->d_th,
                               c0->d.ncop_gamma, full, fill, where, sel);
        };
        if (COP && blocks <= STATES_TAIL) launch(k_states_multi<NS, COP, COP>);
        else launch(k_states_multi<NS, COP, false>);
        if (fold) hipLaunchKernelGGL(k_states_fold_multi, dim3((unsigned)(12 * ncases)), dim3(1024), 0, st, cases);
    }
    static void sweep_multi(const xf_ctx *c0, hipStream_t st, const EnsCase *cases, int ncases, long long blocks,
                            int dir, int shape, int mode, int stage, int sg, int sa, int sb, int so)
    {
        if (c0->d.scheme == XF_WENO5Z)
            SweepLaunch<NS, COP, XF_WENO5Z>::multi(c0, st, cases, ncases, blocks, dir, shape, mode, stage, sg, sa, sb, so);
        else if (c0->d.scheme == XF_WENOCU6)
            SweepLaunch<NS, COP, XF_WENOCU6>::multi(c0, st, cases, ncases, blocks, dir, shape, mode, stage, sg, sa, sb, so);
        else
            SweepLaunch<NS, COP, XF_WENO5JS>::multi(c0, st, cases, ncases, blocks, dir, shape, mode, stage, sg, sa, sb, so);
    }
    static Ops ops()
    {
        return Ops{&states,    &sweep,     &chem,         &prepare,     &chem_multi,         &spill_bytes,
                   &multi_blocks, &visc_prep, &visc_flux, &states_multi, &sweep_multi, visc_in_sweep<NS>()};
    }
};

} // namespace xf
