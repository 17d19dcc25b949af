// mgo_kernels.hip - gfx950 kernels of the Graph-ODE engine (FP64 throughout).
//
// One lane per (node, age group): a wavefront holds 64/G nodes; a node's 10 compartments of one age
// group live in the lane's registers. Cross-age-group terms (force of infection, test-and-trace demand,
// ICU occupancy, the step's error norm) are group reductions over the node's G consecutive lanes through LDS
// slots and shuffles; the G x G contact row of the lane stays in registers. There is no dense
// contraction, so everything runs on the FP64 vector ALUs.
//
// Kernels per half-day cycle (GraphSimulation::advance, cpp/memilio/mobility/graph_simulation.h:101-120):
//   node_phase<G,K>    per node lane: SystemIntegrator::advance to t+dt with integrator K; writes the
//                      departure row and takes the departing travelers off (departure cycles) or writes the
//                      pre-return state and the return coefficients (return cycles)
//   edge_phase<G>      per node lane: the arriving travelers, one sum over the node's in-edges in the
//                      reference's edge order (deterministic, no atomics); or the returns in closed form,
//                      marking the nodes on which the negative-value fix-up can act
//   walk_phase<G>      per node of the instances whose returns need the edge walk (GENERAL), one wavefront each
//   settle_phase<G>    per instance (up to 64 blocks): marked nodes walk their edges with the fix-up, in passes
//                      over the nodes whose inputs changed; sequential replay where these do not settle. Then
//                      the instance's next cycle: step size, edge action and output day
//
// The file is compiled once per shard (MGO_SHARD, see memilio_amd/build.py), in parallel: shard 0 holds the
// launch dispatch and the kernels without a G, shards 1..8 the kernels of that G, shards 9..12 the node kernel
// over mixed G of integrator kind MGO_SHARD - 9, shard 13 the edge kernels over mixed G, shard 14 the percentile sorts.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdint>
#include <type_traits>

#include "../../include/mgo.h"
#include "mgo_internal.h"
#include "mgo_npi.h"

namespace mgo
{

#define MGO_PI 3.14159265358979323846

// Fused multiply-adds are written out: every instantiation of a body (age groups, with or without the optional
// model features, per-G or mixed) then rounds alike, and a run's results do not depend on the kernel that a
// batch's other runs bring with them.
#pragma clang fp contract(off)

// Segment and edge-structure descriptors do not change during a launch and are read from the constant address
// space: the pointers they hold are then known to be global. Read as ordinary memory they are generic, and every
// access through them is a FLAT instruction, which occupies the LDS path too and is waited for with it.
using Seg = const __attribute__((address_space(4))) SegDev;
using Est = const __attribute__((address_space(4))) EdgeStructDev;

__device__ __forceinline__ Seg* segment(const LaunchDev& ld, int seg)
{
    return (Seg*)(ld.segs + seg);
}
__device__ __forceinline__ Est& edge_struct(Seg& c, int k)
{
    return *(Est*)(c.estructs + k);
}
// pointers held by other records (instances, node parameters) are cast to global where they are used
using gdouble = __attribute__((address_space(1))) double;

// orders a wavefront's LDS accesses across its lanes (LDS instructions of a wavefront complete in order)
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// cpp/memilio/math/smoother.h:46-60
__device__ __forceinline__ double smoother_cosine(double x, double xl, double xr, double yl, double yr)
{
    if (x <= xl) {
        return yl;
    }
    if (x >= xr) {
        return yr;
    }
    return fma(0.5 * (yl - yr), cospi((x - xl) / (xr - xl)), 0.5 * (yl + yr));
}

// Blocks are dispatched round-robin over the 8 XCDs; map the hardware block id so that each XCD gets a
// contiguous range of nodes (instances stay within one XCD's L2 for the edge gathers). The host pads
// the grid to a multiple of 8.
__device__ __forceinline__ int xcd_block()
{
    const int per = int(gridDim.x) >> 3;
    const int b   = int(blockIdx.x);
    return (b & 7) * per + (b >> 3);
}

template <int G>
__device__ __forceinline__ double group_sum(double v, int base)
{
    double s = __shfl(v, base);
#pragma unroll
    for (int j = 1; j < G; ++j) {
        s = s + __shfl(v, base + j);
    }
    return s;
}

template <int G>
__device__ __forceinline__ double group_max(double v, int base)
{
    double s = __shfl(v, base);
#pragma unroll
    for (int j = 1; j < G; ++j) {
        s = fmax(s, __shfl(v, base + j));
    }
    return s;
}

template <int G>
__device__ __forceinline__ double group_min(double v, int base)
{
    double s = __shfl(v, base);
#pragma unroll
    for (int j = 1; j < G; ++j) {
        s = fmin(s, __shfl(v, base + j));
    }
    return s;
}

// predicate over the node's G lanes from one wavefront ballot (lanes of a node are active together)
template <int G>
__device__ __forceinline__ bool group_all(bool v, int base)
{
    const unsigned long long m = (~__ballot(!v) >> base) & ((1ull << G) - 1);
    return m == ((1ull << G) - 1);
}

// x^p for the step-size controllers' factors (x > 0, |p| < 1): exp2(p log2 x) within a few ulp of pow, at
// about half of its cost (pow carries log(x) in extended precision for arbitrary exponents)
__device__ __forceinline__ double step_pow(double x, double p)
{
    return exp2(p * log2(x));
}

// 1/x for a population x >= 1e-12: the hardware reciprocal refined by two Newton steps (within an ulp of the
// correctly rounded quotient, half the instructions of the IEEE division sequence)
__device__ __forceinline__ double recip_pop(double x)
{
    double r       = __builtin_amdgcn_rcp(x);
    double e       = fma(-x, r, 1.0);
    r              = fma(r, e, r);
    e              = fma(-x, r, 1.0);
    return fma(r, e, r);
}

// compartments of a lane in registers
template <int M>
struct Comps {
    static constexpr int N = M == PLAIN ? 8 : NC;
    static constexpr int S = 0, E = 1, INS = 2;
    static constexpr int INSC = 3; // FEATURES and NPIS only, like ISYC
    static constexpr int ISY  = M == PLAIN ? 3 : 4;
    static constexpr int ISYC = 5;
    static constexpr int ISEV = M == PLAIN ? 4 : 6;
    static constexpr int ICR  = M == PLAIN ? 5 : 7;
    static constexpr int R    = M == PLAIN ? 6 : 8;
    static constexpr int D    = M == PLAIN ? 7 : 9;
    // register of compartment i of the state layout, or -1
    __device__ static constexpr int of(int i)
    {
        return M != PLAIN ? i : (i < mgo::INSC) ? i : (i == mgo::INSC || i == mgo::ISYC) ? -1 : (i == mgo::ISY) ? 3 : i - 2;
    }
};

// Per-lane context of one node lane, loaded once per kernel.
template <int G, int M>
struct Lane {
    // rates (see LaneCoef); isev: the sum of ISev's
    double e, ins_isy, ins_r, isy_isev, isy_r, isev_icr, isev_r, isev_d, isev, icr_d, icr_r;
    double rel, risk, tp;
    double crow[G]; // contact row times tp at the last evaluated time (constant without dampings)
    // features
    double ttr, maxrisk, cps, dps, tisev, ttc, ttc_hi, icu_cap;
    const gdouble* damp_time;
    const gdouble* damp_mat;
    int damp_cnt;
    double row_lo, row_hi; // crow holds for row_lo <= t <= row_hi (dampings)
    int flags;
    int node;
    int age;
    int base;         // first lane of the node's group
    int inst;
    double* wx;       // LDS: the wavefront's exchange slots, one double per lane (force of infection, error norm)
    double* ws;       // LDS: the wavefront's stage-season slots, (5 + G - 1) / G planes of BLOCK doubles
    double* cold;     // LDS: the lane's Cold values, planes of BLOCK doubles
};

// Scalars of a lane that a step attempt reads at most a few times: kept in LDS, since the registers of two
// wavefronts per SIMD hold the stage vectors (in registers, 25 values per attempt went through scratch memory).
enum Cold : int {
    COLD_ABS = 0,
    COLD_REL,
    COLD_DT_MAX,
    COLD_DT_MIN,
    COLD_DT_RESTORE,
    COLD_TMAX,   // end of the piece
    COLD_SPAN,   // its length
    COLD_SEASON, // season of the next k1
    COLD_START_DAY,
    COLD_SEASONALITY,
    COLD_DAYS,   // two integers: next output day, end of the output days (both counted from day0)
    COLD_COUNTS, // two integers: steps, attempts
    NUM_COLD
};

// LDS of a node kernel: exchange slots, stage-season planes, cold planes
template <int G>
constexpr int node_lds()
{
    return BLOCK * (1 + (5 + G - 1) / G + NUM_COLD);
}

// Effective contact row C(t)_age,. = B - D(t) o (B - M) (contact_matrix.h:190-194, damping.h:381-396), times tp, of
// a node with dampings. D changes only within the day before a damping's time: outside of it the row and its
// interval are kept, so that most right-hand sides do without the chain of loads from the damping cache (their
// latency, in every right-hand side, was most of the node kernel's time on damped nodes).
template <int G, int M>
__device__ __forceinline__ void contact_row(Seg& c, Lane<G, M>& L, double t)
{
    if (t >= L.row_lo && t <= L.row_hi) {
        return;
    }
    const double* B   = c.cbase + (size_t(L.node) * G + L.age) * G;
    const gdouble* tk = L.damp_time;
    int k             = 1;
    while (k < L.damp_cnt - 1 && !(tk[k] > t)) {
        ++k;
    }
    const double xr    = tk[k];
    const double xl    = xr - 1.0;
    const gdouble* Dl  = L.damp_mat + (size_t(k - 1) * G + L.age) * G;
    const gdouble* Dr  = L.damp_mat + (size_t(k) * G + L.age) * G;
    const double* Dd   = c.cdelta + (size_t(L.node) * G + L.age) * G;
    const bool left    = t <= xl;
    const bool right   = t >= xr;
    const double cs    = (left || right) ? 0.0 : cospi((t - xl) / (xr - xl));
    L.row_lo           = left ? tk[k - 1] : INFINITY;
    L.row_hi           = left ? xl : -INFINITY;
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const double d = left ? Dl[j] : (right ? Dr[j] : fma(0.5 * (Dl[j] - Dr[j]), cs, 0.5 * (Dl[j] + Dr[j])));
        L.crow[j]      = L.tp * fma(-d, Dd[j], B[j]);
    }
}

// Seasonal factor 1 + k sin(pi ((StartDay + t) / 182.5 + 0.5)) of the lane's node at time t
// (model.h:115-117). sinpi reduces its argument exactly; sin needs a reduction by pi whose code (and registers)
// was a tenth of the kernel.
template <int G, int M>
__device__ __forceinline__ double season_at(const Lane<G, M>& L, double t)
{
    return fma(L.cold[COLD_SEASONALITY * BLOCK], sinpi(fma(L.cold[COLD_START_DAY * BLOCK] + t, 1.0 / 182.5, 0.5)), 1.0);
}

// Seasonal factors of the five later stages of a step, spread over the node's G lanes: lane a evaluates
// stages j = a, a + G, ... (j < 5) at t + c_j h, and every lane reads a stage's factor from the lane that
// owns it (one sin per lane and step attempt for G >= 5 instead of five).
template <int G, int M>
__device__ __forceinline__ void stage_seasons(const Lane<G, M>& L, double t, double h, double c2, double c3,
                                              double c4, double c5, double c6)
{
#pragma unroll
    for (int q = 0; q < (5 + G - 1) / G; ++q) {
        const int j    = L.age + q * G;
        const double c = (j == 0) ? c2 : (j == 1) ? c3 : (j == 2) ? c4 : (j == 3) ? c5 : c6;
        L.ws[q * BLOCK + threadIdx.x % WAVE] = (j < 5) ? season_at(L, fma(c, h, t)) : 1.0;
    }
    wave_sync();
}

template <int J, int G, int M>
__device__ __forceinline__ double stage_season(const Lane<G, M>& L)
{
    return L.ws[(J / G) * BLOCK + L.base + J % G];
}

// Force-of-infection coefficient of the lane's age group: season * tp * sum_j C_gj(t) w_j(pop),
// w_j = divN_j * (rel_j pop[INS_j] + risk_j pop[ISy_j]) (model.h:99-145, factored over j). Also returns
// the ICU-adjusted ISev->ICr / ISev->D coefficients (model.h:147-152, 196-204).
template <int G, int M>
__device__ __forceinline__ double force_of_infection(Seg& c, Lane<G, M>& L, const double (&pop)[Comps<M>::N], double t,
                                                     double season, double& c_icr, double& c_d)
{
    using X     = Comps<M>;
    double risk = L.risk;
    if (M != PLAIN && (L.flags & NF_TTC_ACTIVE)) {
        const double ttr = group_sum<G>(L.ttr * pop[X::INS], L.base);
        risk             = smoother_cosine(ttr, L.ttc, L.ttc_hi, L.risk, L.maxrisk);
    }
    const double Nj = ((pop[X::S] + pop[X::E]) + (pop[X::INS] + pop[X::ISY])) + ((pop[X::ISEV] + pop[X::ICR]) + pop[X::R]);
    const double divN = (Nj < 1e-12) ? 0.0 : recip_pop(Nj);
    const double w    = divN * fma(L.rel, pop[X::INS], risk * pop[X::ISY]);
    if (M != PLAIN && (L.flags & NF_DAMPED)) {
        contact_row(c, L, t);
    }
    // w of the node's G lanes through the wavefront's LDS slots: one write, G reads (a wavefront's LDS
    // instructions complete in order; the lanes of a node are active together)
    L.wx[threadIdx.x % WAVE] = w;
    wave_sync();
    double wg[G];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        wg[j] = L.wx[L.base + j];
    }
    wave_sync();
    double lam = L.crow[0] * wg[0], lam1 = 0.0; // two chains: half the latency
    if constexpr (G > 1) {
        lam1 = L.crow[1] * wg[1];
    }
#pragma unroll
    for (int j = 2; j < G; ++j) {
        double& l = (j & 1) ? lam1 : lam;
        l         = fma(L.crow[j], wg[j], l);
    }
    lam += lam1;
    c_icr = L.isev_icr;
    c_d   = L.isev_d;
    if (M != PLAIN && (L.flags & NF_ICU_ACTIVE)) {
        const double icu  = group_sum<G>(pop[X::ICR], L.base);
        const double crit = smoother_cosine(icu, 0.90 * L.icu_cap, L.icu_cap, L.cps, 0.0);
        c_icr             = crit / L.tisev;
        c_d               = (L.dps + (L.cps - crit)) / L.tisev;
    }
    return season * lam;
}

// Right-hand side of the node ODE, pop == y (osecir::Model::get_flows + FlowModel::get_derivatives,
// flow_model.h:112-125,219-235). A flow that leaves one compartment and enters another is computed once where two
// uses need it and fused into the sums elsewhere.
template <int G, int M>
__device__ __forceinline__ void rhs(Seg& c, Lane<G, M>& L, const double (&y)[Comps<M>::N], double t, double season,
                                    double (&dy)[Comps<M>::N])
{
    using X = Comps<M>;
    double c_icr, c_d;
    const double f0   = y[X::S] * force_of_infection(c, L, y, t, season, c_icr, c_d);
    const double f1   = L.e * y[X::E];
    const double f2   = L.ins_isy * y[X::INS];
    const double f6   = L.isy_isev * y[X::ISY];
    double isev       = L.isev;
    double to_isev    = f6;
    double to_r       = fma(L.ins_r, y[X::INS], fma(L.isy_r, y[X::ISY], fma(L.isev_r, y[X::ISEV], L.icr_r * y[X::ICR])));
    if constexpr (M != PLAIN) {
        if (L.flags & NF_ICU_ACTIVE) {
            isev = (c_icr + L.isev_r) + c_d;
        }
        const double f4 = L.ins_isy * y[X::INSC];
        const double f8 = L.isy_isev * y[X::ISYC];
        to_isev += f8;
        to_r        = fma(L.ins_r, y[X::INSC], fma(L.isy_r, y[X::ISYC], to_r));
        dy[X::INSC] = fma(-L.ins_r, y[X::INSC], -f4);
        dy[X::ISYC] = fma(-L.isy_r, y[X::ISYC], f4 - f8);
    }
    dy[X::S]    = -f0;
    dy[X::E]    = f0 - f1;
    dy[X::INS]  = fma(-L.ins_r, y[X::INS], f1 - f2);
    dy[X::ISY]  = fma(-L.isy_r, y[X::ISY], f2 - f6);
    dy[X::ISEV] = fma(-isev, y[X::ISEV], to_isev);
    dy[X::ICR]  = fma(-L.icr_r, y[X::ICR], fma(-L.icr_d, y[X::ICR], c_icr * y[X::ISEV]));
    dy[X::R]    = to_r;
    dy[X::D]    = fma(c_d, y[X::ISEV], L.icr_d * y[X::ICR]);
}

// ------------------------------------------------------------------------------- Cash-Karp 5(4)
// Cash & Karp, ACM TOMS 16 (1990) 201-222; the same ratios odeint's runge_kutta_cash_karp54 uses.
namespace ck
{
constexpr double C2 = 1.0 / 5.0, C3 = 3.0 / 10.0, C4 = 3.0 / 5.0, C5 = 1.0, C6 = 7.0 / 8.0;
constexpr double A21 = 1.0 / 5.0;
constexpr double A31 = 3.0 / 40.0, A32 = 9.0 / 40.0;
constexpr double A41 = 3.0 / 10.0, A42 = -9.0 / 10.0, A43 = 6.0 / 5.0;
constexpr double A51 = -11.0 / 54.0, A52 = 5.0 / 2.0, A53 = -70.0 / 27.0, A54 = 35.0 / 27.0;
constexpr double A61 = 1631.0 / 55296.0, A62 = 175.0 / 512.0, A63 = 575.0 / 13824.0, A64 = 44275.0 / 110592.0,
                 A65 = 253.0 / 4096.0;
constexpr double B1 = 37.0 / 378.0, B3 = 250.0 / 621.0, B4 = 125.0 / 594.0, B6 = 512.0 / 1771.0;
constexpr double E1 = 37.0 / 378.0 - 2825.0 / 27648.0, E3 = 250.0 / 621.0 - 18575.0 / 48384.0,
                 E4 = 125.0 / 594.0 - 13525.0 / 55296.0, E5 = -277.0 / 14336.0, E6 = 512.0 / 1771.0 - 1.0 / 4.0;
} // namespace ck

// One Cash-Karp step from (y, k1 = f(y, t)) with step h: 5th-order solution in yo, embedded error in er.
template <int G, int M>
__device__ __forceinline__ void cash_karp_stages(Seg& c, Lane<G, M>& L, const double (&y)[Comps<M>::N],
                                                 const double (&k1)[Comps<M>::N], double t, double h,
                                                 double (&yo)[Comps<M>::N], double (&er)[Comps<M>::N], bool want_err)
{
    constexpr int N = Comps<M>::N;
    stage_seasons(L, t, h, ck::C2, ck::C3, ck::C4, ck::C5, ck::C6);
    double k2[N], k3[N], k4[N], k5[N], yt[N];
    {
        const double a1 = ck::A21 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a1, k1[i], y[i]);
        }
    }
    rhs(c, L, yt, fma(ck::C2, h, t), stage_season<0>(L), k2);
    {
        const double a1 = ck::A31 * h, a2 = ck::A32 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a2, k2[i], fma(a1, k1[i], y[i]));
        }
    }
    rhs(c, L, yt, fma(ck::C3, h, t), stage_season<1>(L), k3);
    {
        const double a1 = ck::A41 * h, a2 = ck::A42 * h, a3 = ck::A43 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a3, k3[i], fma(a2, k2[i], fma(a1, k1[i], y[i])));
        }
    }
    rhs(c, L, yt, fma(ck::C4, h, t), stage_season<2>(L), k4);
    {
        const double a1 = ck::A51 * h, a2 = ck::A52 * h, a3 = ck::A53 * h, a4 = ck::A54 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a4, k4[i], fma(a3, k3[i], fma(a2, k2[i], fma(a1, k1[i], y[i]))));
        }
    }
    rhs(c, L, yt, fma(ck::C5, h, t), stage_season<3>(L), k5);
    {
        const double a1 = ck::A61 * h, a2 = ck::A62 * h, a3 = ck::A63 * h, a4 = ck::A64 * h, a5 = ck::A65 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a5, k5[i], fma(a4, k4[i], fma(a3, k3[i], fma(a2, k2[i], fma(a1, k1[i], y[i])))));
        }
    }
    double(&k6)[N] = k2; // k2 is no longer needed
    rhs(c, L, yt, fma(ck::C6, h, t), stage_season<4>(L), k6);
    {
        const double b1 = ck::B1 * h, b3 = ck::B3 * h, b4 = ck::B4 * h, b6 = ck::B6 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yo[i] = fma(b6, k6[i], fma(b4, k4[i], fma(b3, k3[i], fma(b1, k1[i], y[i]))));
        }
    }
    if (want_err) {
        const double e1 = ck::E1 * h, e3 = ck::E3 * h, e4 = ck::E4 * h, e5 = ck::E5 * h, e6 = ck::E6 * h;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            er[i] = fma(e6, k6[i], fma(e5, k5[i], fma(e4, k4[i], fma(e3, k3[i], e1 * k1[i]))));
        }
    }
}

// ------------------------------------------------------------------------------- RKF45 (RKIntegratorCore)
// adapt_rk.h:71-137 default tableau
namespace rkf
{
constexpr double C2 = 0.25, C3 = 3 / 8.0, C4 = 12 / 13.0, C5 = 1.0, C6 = 0.5;
constexpr double A21 = 0.25;
constexpr double A31 = 3 / 32.0, A32 = 9 / 32.0;
constexpr double A41 = 1932 / 2197.0, A42 = -7200 / 2197.0, A43 = 7296 / 2197.0;
constexpr double A51 = 439 / 216.0, A52 = -8.0, A53 = 3680 / 513.0, A54 = -845 / 4104.0;
constexpr double A61 = -8 / 27.0, A62 = 2.0, A63 = -3544 / 2565.0, A64 = 1859 / 4104.0, A65 = -11 / 40.0;
constexpr double BL1 = 25 / 216.0, BL3 = 1408 / 2565.0, BL4 = 2197 / 4104.0, BL5 = -0.2;
constexpr double BH1 = 16 / 135.0, BH3 = 6656 / 12825.0, BH4 = 28561 / 56430.0, BH5 = -9 / 50.0, BH6 = 2 / 55.0;
constexpr double D1 = BH1 - BL1, D3 = BH3 - BL3, D4 = BH4 - BL4, D5 = BH5 - BL5, D6 = BH6 - 0.0;
} // namespace rkf

template <int G, int M>
__device__ __forceinline__ void rkf45_stages(Seg& c, Lane<G, M>& L, const double (&y)[Comps<M>::N],
                                             const double (&k1)[Comps<M>::N], double t, double h,
                                             double (&yo)[Comps<M>::N], double (&er)[Comps<M>::N])
{
    constexpr int N = Comps<M>::N;
    stage_seasons(L, t, h, rkf::C2, rkf::C3, rkf::C4, rkf::C5, rkf::C6);
    double k2[N], k3[N], k4[N], k5[N], yt[N];
    {
        const double a1 = h * rkf::A21;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a1, k1[i], y[i]);
        }
    }
    rhs(c, L, yt, fma(rkf::C2, h, t), stage_season<0>(L), k2);
    {
        const double a1 = h * rkf::A31, a2 = h * rkf::A32;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a2, k2[i], fma(a1, k1[i], y[i]));
        }
    }
    rhs(c, L, yt, fma(rkf::C3, h, t), stage_season<1>(L), k3);
    {
        const double a1 = h * rkf::A41, a2 = h * rkf::A42, a3 = h * rkf::A43;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a3, k3[i], fma(a2, k2[i], fma(a1, k1[i], y[i])));
        }
    }
    rhs(c, L, yt, fma(rkf::C4, h, t), stage_season<2>(L), k4);
    {
        const double a1 = h * rkf::A51, a2 = h * rkf::A52, a3 = h * rkf::A53, a4 = h * rkf::A54;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a4, k4[i], fma(a3, k3[i], fma(a2, k2[i], fma(a1, k1[i], y[i]))));
        }
    }
    rhs(c, L, yt, fma(rkf::C5, h, t), stage_season<3>(L), k5);
    {
        const double a1 = h * rkf::A61, a2 = h * rkf::A62, a3 = h * rkf::A63, a4 = h * rkf::A64, a5 = h * rkf::A65;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            yt[i] = fma(a5, k5[i], fma(a4, k4[i], fma(a3, k3[i], fma(a2, k2[i], fma(a1, k1[i], y[i])))));
        }
    }
    double(&k6)[N] = k2; // k2 is no longer needed
    rhs(c, L, yt, fma(rkf::C6, h, t), stage_season<4>(L), k6);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        // y + dt * (K * b_low) and dt * |K * (b_high - b_low)| (adapt_rk.h:268-271)
        const double sl = fma(k5[i], rkf::BL5, fma(k4[i], rkf::BL4, fma(k3[i], rkf::BL3, k1[i] * rkf::BL1)));
        yo[i]           = fma(sl, h, y[i]);
        const double sd =
            fma(k6[i], rkf::D6, fma(k5[i], rkf::D5, fma(k4[i], rkf::D4, fma(k3[i], rkf::D3, k1[i] * rkf::D1))));
        er[i] = h * fabs(sd);
    }
}

template <int G, int M>
__device__ __forceinline__ Seg* load_lane(const LaunchDev& ld, Lane<G, M>& L, double* wx)
{
    L.wx = wx + (threadIdx.x / WAVE) * WAVE;
    L.ws = wx + BLOCK + (threadIdx.x / WAVE) * WAVE;
    L.cold = wx + BLOCK * (1 + (5 + G - 1) / G) + threadIdx.x;
    constexpr int NPW = WAVE / G;
    const int lb      = xcd_block();
    if (lb >= ld.num_blocks) {
        return nullptr;
    }
    const int seg = ld.block_seg[lb];
    if (seg < 0) {
        return nullptr;
    }
    Seg* c = segment(ld, seg);
    const int wave  = (lb - ld.block_first[seg]) * (BLOCK / WAVE) + int(threadIdx.x) / WAVE;
    const int lane  = int(threadIdx.x) % WAVE;
    const int grp   = lane / G;
    L.age           = lane - grp * G;
    L.node          = wave * NPW + grp;
    L.base          = grp * G; // lane index (within the wavefront) of the group's first lane
    if (grp >= NPW || L.node >= c->num_nodes) {
        return nullptr;
    }
    if (c->node_order) {
        L.node = c->node_order[L.node]; // same graph node of consecutive runs in one wavefront
    }
    const NodeP& np = c->nodep[L.node];
    L.flags         = np.flags;
    L.inst          = np.inst;
    L.cold[COLD_START_DAY * BLOCK]   = np.start_day;
    L.cold[COLD_SEASONALITY * BLOCK] = np.seasonality;
    double lc[NUM_LC];
    const double2* p = reinterpret_cast<const double2*>(c->lcoef + (size_t(L.node) * G + L.age) * NUM_LC);
#pragma unroll
    for (int k = 0; k < NUM_LC / 2; ++k) {
        const double2 v = p[k];
        lc[2 * k]       = v.x;
        lc[2 * k + 1]   = v.y;
    }
    L.e        = lc[LC_E];
    L.ins_isy  = lc[LC_INS_ISY];
    L.ins_r    = lc[LC_INS_R];
    L.isy_isev = lc[LC_ISY_ISEV];
    L.isy_r    = lc[LC_ISY_R];
    L.isev_icr = lc[LC_ISEV_ICR];
    L.isev_r   = lc[LC_ISEV_R];
    L.isev_d   = lc[LC_ISEV_D];
    L.isev     = (lc[LC_ISEV_ICR] + lc[LC_ISEV_R]) + lc[LC_ISEV_D];
    L.icr_d    = lc[LC_ICR_D];
    L.icr_r    = lc[LC_ICR_R];
    L.tp       = lc[LC_TP];
    L.rel      = lc[LC_REL];
    L.risk     = lc[LC_RISK];
    if constexpr (M != PLAIN) {
        L.maxrisk   = lc[LC_MAXRISK];
        L.ttr       = lc[LC_TTR];
        L.cps       = lc[LC_CPS];
        L.dps       = lc[LC_DPS];
        L.tisev     = lc[LC_TISEV];
        L.ttc       = np.ttc;
        L.ttc_hi    = np.ttc_hi;
        L.icu_cap   = np.icu;
        L.damp_time = (const gdouble*)np.damp_time;
        L.damp_mat  = (const gdouble*)np.damp_mat;
        L.damp_cnt  = np.damp_cnt;
        L.row_lo    = INFINITY;
        L.row_hi    = -INFINITY;
    }
    const double* B = c->cbase + (size_t(L.node) * G + L.age) * G;
#pragma unroll
    for (int j = 0; j < G; ++j) {
        L.crow[j] = L.tp * B[j];
    }
    return c;
}

__device__ __forceinline__ double detect_nondetection(const NodeP& np, double t)
{
    // test_commuters (model.h:717-742): nondetection applies in [start, end)
    return (t >= np.det_start && t < np.det_end) ? np.nondetect : 1.0;
}

// mobility factor of the ISy compartment of the lane's age group (model.h:687-715)
template <int G, int M>
__device__ __forceinline__ double mobility_factor(const Lane<G, M>& L, double y_ins)
{
    if (M == PLAIN || !(L.flags & NF_TTC_ACTIVE)) {
        return L.risk;
    }
    const double ttr = group_sum<G>(L.ttr * y_ins, L.base);
    return smoother_cosine(ttr, L.ttc, L.ttc_hi, L.risk, L.maxrisk);
}

// ------------------------------------------------------------------------------- clock
// One GraphSimulation::advance loop iteration per instance (graph_simulation.h:101-120) and the
// departure/return alternation of MobilityEdge::apply_mobility (metapopulation_mobility_instant.h:544-623).
__device__ __forceinline__ void clock_one(InstDev& I)
{
    I.c_active  = 0;
    I.c_action  = 0;
    I.c_out_day = -1;
    I.fx_state  = 0;
    I.fx_changed = 0;
    I.fx_pass    = 0;
    I.fx_count   = 0;
    if (I.status != 0 || !(I.t < I.tmax) || I.plain == PLAIN_LOST) {
        return;
    }
    double step = I.dt_graph;
    if (I.t + step > I.tmax) {
        step = I.tmax - I.t;
    }
    // single-model runs end exactly at tmax (Simulation::advance(tmax)); graph runs at t + dt like
    // SimulationNode::advance(t, dt)
    const double tn = (I.exact_end && step != I.dt_graph) ? I.tmax : I.t + step;
    I.c_active      = 1;
    I.c_t0          = I.t;
    I.c_t1          = tn;
    I.c_step        = step;
    if (I.estruct >= 0) {
        if (I.pending && I.ret_time <= tn) {
            if (I.toggle) {
                I.c_action = 2;
                I.c_tdep   = I.t_dep;
                I.pending  = 0;
            }
            else {
                I.status = MGO_ERR_UNSUPPORTED; // return and departure in one call: more than one pending move
            }
        }
        else if (!I.toggle) {
            if (I.pending) {
                I.status = MGO_ERR_UNSUPPORTED;
            }
            else {
                I.c_action = 1;
                I.fx_neg   = 0;
                I.pending  = 1;
                I.t_dep    = tn;
                I.ret_time = tn + step;
            }
        }
        I.toggle ^= 1;
    }
    if (I.c_action == 2) {
        I.fx_epoch += FX_EPOCH_STEP; // fix-up records of earlier return phases read as unfixed
    }
    I.t             = tn;
    const double dn = rint(tn);
    if (fabs(tn - dn) <= 1e-10) {
        const int d = int(dn) - I.day0;
        if (d >= 0 && d < I.ndays) {
            I.c_out_day = d;
        }
    }
}

// First clock of a run; later ones are advanced at the end of the settling kernel.
static __global__ void __launch_bounds__(256) clock_kernel(InstDev* inst, int n)
{
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) {
        clock_one(inst[i]);
    }
}

// daily output of local node v: [day][v][g][10]
__device__ __forceinline__ gdouble* out_ptr(const InstDev& I, int v, int age, int G, int day)
{
    return (gdouble*)I.out + (size_t(day) * I.num_nodes + v) * size_t(G * NC) + size_t(age) * NC;
}

// linear_interpolation (math/interpolation.h:44-48): y_a + w (y_b - y_a), rounded as the reference (no FMA)
__device__ __forceinline__ double lerp_ref(double ya, double yb, double w)
{
#pragma clang fp contract(off)
    return ya + w * (yb - ya);
}

// Daily value of the output day d = c_out_day at the end of a phase, from the lane's state y after the phase's
// edge action (apply_mobility changes the last value of the node's TimeSeries in place), as
// interpolate_simulation_result (analyze_result.h:235-261) takes it from the node's time points: between the
// state before the node's last step and y when that step ends at or after d (weight 1 when it ends on d);
// else y, the last value so far: then the next phase's first step encloses d and overwrites the day.
template <int G>
__device__ __forceinline__ void write_phase_end_day(Seg& c, const InstDev& I, size_t lane, int v, int age,
                                                    const double (&y)[NC])
{
    const double* pr = c.yint + lane * YINT_STRIDE;
    const double w   = pr[YINT_W];
    gdouble* op       = out_ptr(I, v, age, G, I.c_out_day);
    if (w >= 0.0) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            op[i] = lerp_ref(pr[i], y[i], w);
        }
    }
    else {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            op[i] = y[i];
        }
    }
}

// segment node of an instance's local node v
__device__ __forceinline__ size_t seg_node(const InstDev& I, int v)
{
    return size_t(I.node_base) + size_t(v) * size_t(I.node_stride);
}

// Plane arrays (SegDev::dep, arr, ypre, wst): every compartment pair is one 16-byte plane over the segment's
// lanes, so a wavefront's access to it is one contiguous run.
// ten compartments of a lane from / to planes
__device__ __forceinline__ void load_planes(const double2* p, size_t stride, size_t lane, double (&v)[NC])
{
#pragma unroll
    for (int q = 0; q < NC / 2; ++q) {
        const double2 t = p[size_t(q) * stride + lane];
        v[2 * q]        = t.x;
        v[2 * q + 1]    = t.y;
    }
}
__device__ __forceinline__ void store_planes(double2* p, size_t stride, size_t lane, const double (&v)[NC])
{
#pragma unroll
    for (int q = 0; q < NC / 2; ++q) {
        p[size_t(q) * stride + lane] = double2{v[2 * q], v[2 * q + 1]};
    }
}

// Return coefficients of the lane's node as a destination (calculate_mobility_returns,
// metapopulation_mobility_instant.h:460-471): the force of infection and the ICU-adjusted rates of the state
// pop at the departure time, frozen for the Euler step of the returning travelers (the other rates are lane
// constants).
template <int G, int M>
__device__ __forceinline__ void return_coefficients(Seg& c, Lane<G, M>& L, const InstDev& I,
                                                    const double (&pop)[Comps<M>::N])
{
    double c_icr, c_d;
    const double kappa = force_of_infection(c, L, pop, I.c_tdep, season_at(L, I.c_tdep), c_icr, c_d);
    const size_t lane  = size_t(L.node) * G + L.age;
    c.kap[lane]        = kappa;
    if (c.kicu) {
        c.kicu[lane] = double2{c_icr, c_d};
    }
}

// Coefficient at the departure time, B - D (B - M) (DampingMatrixExpression::get_matrix_at,
// contact_matrix.h:190-194), of an edge or of a sum over edges of one source. D: the source's damping factor.
__device__ __forceinline__ double damped(double b, double m, double D)
{
#pragma clang fp contract(off)
    return b - D * (b - m);
}

// Departures of the lane's node at c_t1 (metapopulation_mobility_instant.h:605-621): the departure row (the
// traveler vector per unit of coefficient: SimulationNode::m_last_state with the ISy mobility factor and the
// commuter nondetection factor), and the node's state without all its travelers. Every out-edge takes the same
// row times its coefficient, so the sum over the out-edges is the row times the sum of the coefficients (a
// constant of the graph): no walk over the out-edges.
template <int G, int M>
__device__ __forceinline__ void leave(Seg& c, const Lane<G, M>& L, InstDev& I, double fac, double nd, double D,
                                      double (&y)[NC])
{
#pragma clang fp contract(off)
    Est& es = edge_struct(c, I.estruct);
    const size_t lane       = size_t(L.node) * G + L.age;
    double row[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        row[i] = y[i];
    }
    row[ISY] = row[ISY] * fac;
    double gone[NC];
    const int v = c.nodep[L.node].local;
    if (es.out_sum) {
        double sum = es.out_sum[v];
        if (D != 0.0) {
            sum = damped(sum, es.out_min_sum ? es.out_min_sum[v] : 0.0, D);
        }
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            gone[i] = row[i] * sum;
        }
    }
    else {
        const size_t off = (size_t(v) * G + L.age) * NC;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            double sum = es.out_vsum[off + i];
            if (D != 0.0) {
                sum = damped(sum, es.out_vmin_sum ? es.out_vmin_sum[off + i] : 0.0, D);
            }
            gone[i] = row[i] * sum;
        }
    }
    if (nd != 1.0) {
        // test_commuters on the source: detected commuters stay home as confirmed cases
        y[INS] -= gone[INS] * (1 - nd);
        y[INSC] += gone[INS] * (1 - nd);
        y[ISY] -= gone[ISY] * (1 - nd);
        y[ISYC] += gone[ISY] * (1 - nd);
        gone[ISY] *= nd;
        gone[INS] *= nd;
        row[ISY] *= nd;
        row[INS] *= nd;
    }
    bool odd = !(D >= 0.0 && D <= 1.0);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        y[i] -= gone[i];
        odd = odd || !(row[i] >= 0.0);
    }
    store_planes(c.dep, size_t(c.num_nodes) * G, lane, row);
    if (odd) {
        I.fx_neg = 1; // negative travelers: the returns of this departure walk their edges (every writer stores 1)
    }
}

// ------------------------------------------------------------------------------- dynamic NPIs
// The check at the start of one piece of osecir::Simulation::advance (models/ode_secir/model.h:301-349) for
// the lane's node at time t with state y, and the length of the piece (model.h:351-357: at most one day,
// ending at the active NPI's end). Every lane of the node reaches the same decision; the first lane of the
// group implements the NPI on the node's damping list and cache (mgo_npi.h). Returns true in `changed`
// when the contact matrix changed.
template <int G, int M>
__device__ double npi_piece(Seg& c, Lane<G, M>& L, InstDev& I, const double (&y)[NC], double t, double tmax,
                            bool& changed)
{
    NpiNode* nn         = c.npi + L.node;
    const double sum    = group_sum<G>(y[ISY], L.base); // InfectedSymptoms summed over the groups in order
    const double begin  = nn->begin, end = nn->end;
    double t_end        = nn->t_end;
    changed             = false;
    // floating_point_greater_equal(a, b, 1e-10) (math/floating_point.h:96-100)
    auto ge = [](double a, double b) {
        return !(a - b < -(1e-10 + DBL_MIN * fmax(fabs(a), fabs(b))));
    };
    if (ge(t, begin) && t < end) {
        const double inf_rel = sum / nn->total * nn->base;
        int k                = 0;
        while (k < nn->thr_count && !(inf_rel > c.npi_thr[nn->thr_first + k])) {
            ++k;
        }
        const bool expired = ge(t, t_end);
        if (k < nn->thr_count) {
            const double thr   = c.npi_thr[nn->thr_first + k];
            const double value = nn->value;
            if (thr > value || expired) {
                const bool renewal = expired && !(thr > value);
                const double delay = renewal ? 0.0 : (t > 0 ? nn->delay : 0.0);
                if (t + delay < end) {
                    const double t_start = t + delay;
                    const double te      = (t_start + nn->duration < end) ? t_start + nn->duration : end;
                    const double tsd     = (!renewal && t_start > 0.0) ? t_start + 1.0 : t_start;
                    t_end                = te;
                    changed              = true;
                    if (L.age == 0) {
                        nn->value = thr;
                        nn->t_end = te;
                        const int gi = nn->thr_first + k;
                        const int d0 = c.npi_thr_damp[gi], d1 = c.npi_thr_damp[gi + 1];
                        int count    = nn->list_count;
                        bool ok      = npi_implement(nn->list, count, nn->list_cap, G, true,
                                                     c.npi_damp + d0 * (3 + G), d1 - d0, tsd, te + 1.0, nn->work);
                        const int m  = ok ? npi_build_cache(nn->list, count, G * G, nn->list_cap, nn->cache_t,
                                                            nn->cache_m, nn->work)
                                          : -1;
                        if (m < 0) {
                            I.status = MGO_ERR_OUT_OF_RANGE; // damping list or level capacity exceeded
                        }
                        else {
                            nn->list_count  = count;
                            nn->cache_count = m;
                            const_cast<NodeP*>(c.nodep)[L.node].damp_cnt = m;
                        }
                    }
                }
            }
        }
    }
    if (changed) {
        __threadfence(); // the group's other lanes read the new cache written by its first lane
        L.damp_cnt = __shfl(*static_cast<volatile int32_t*>(&nn->cache_count), L.base);
        L.row_lo   = INFINITY; // the kept contact row is of the old cache
        L.row_hi   = -INFINITY;
    }
    double dt_eff = (tmax - t < 1.0) ? tmax - t : 1.0;
    if (t < t_end) {
        dt_eff = (t_end - t < dt_eff) ? t_end - t : dt_eff;
    }
    return dt_eff;
}

// Out-edge dampings of the lane's node at the cycle's edge action (MobilityEdge::apply_mobility at t = c_t1,
// metapopulation_mobility_instant.h:549-566): the edge NPI check on the node's last state (no delay, no
// directive; begin t, end t + duration, per-group mobility dampings), then on a departure the damping factor
// D of the lane's age group at t (Dampings::get_matrix_at, damping.h:381-396) for the edge kernels.
template <int G, int M>
__device__ double out_damping(Seg& c, Lane<G, M>& L, InstDev& I, const double (&y)[NC])
{
    NpiNode* od    = c.out_npi + L.node;
    const double t = I.c_t1;
    if (od->thr_count > 0) {
        const double sum     = group_sum<G>(y[ISY], L.base);
        const double inf_rel = sum / od->total * od->base;
        int k                = 0;
        while (k < od->thr_count && !(inf_rel > c.out_thr[od->thr_first + k])) {
            ++k;
        }
        const double te    = od->t_end;
        const bool expired = !(t - te < -(1e-10 + DBL_MIN * fmax(fabs(t), fabs(te))));
        bool changed       = false;
        if (k < od->thr_count) {
            const double thr = c.out_thr[od->thr_first + k];
            if (thr > od->value || expired) {
                changed = true;
                if (L.age == 0) {
                    const double t_end = t + od->duration;
                    od->value          = thr;
                    od->t_end          = t_end;
                    const int gi       = od->thr_first + k;
                    const int d0 = c.out_thr_damp[gi], d1 = c.out_thr_damp[gi + 1];
                    int count    = od->list_count;
                    const bool ok = npi_implement(od->list, count, od->list_cap, G, false, c.out_damp + d0 * (3 + G),
                                                  d1 - d0, t, t_end, od->work);
                    const int m   = ok ? npi_build_cache(od->list, count, G, od->list_cap, od->cache_t, od->cache_m,
                                                         od->work)
                                       : -1;
                    if (m < 0) {
                        I.status = MGO_ERR_OUT_OF_RANGE; // damping list or level capacity exceeded
                    }
                    else {
                        od->list_count  = count;
                        od->cache_count = m;
                    }
                }
            }
        }
        if (changed) {
            __threadfence(); // the group's other lanes read the cache written by its first lane
        }
    }
    if (I.c_action == 1) {
        const int cnt    = *static_cast<volatile int32_t*>(&od->cache_count);
        const double* tk = od->cache_t;
        int k            = 1;
        while (k < cnt - 1 && !(tk[k] > t)) {
            ++k;
        }
        const double xr = tk[k], xl = xr - 1.0;
        const double Dl = od->cache_m[(k - 1) * G + L.age], Dr = od->cache_m[k * G + L.age];
        double d;
        if (t <= xl) {
            d = Dl;
        }
        else if (t >= xr) {
            d = Dr;
        }
        else {
            d = fma(0.5 * (Dl - Dr), cospi((t - xl) / (xr - xl)), 0.5 * (Dl + Dr));
        }
        c.out_d[size_t(L.node) * G + L.age] = d;
        return d;
    }
    return 0.0;
}

// ------------------------------------------------------------------------------- node phase
// SystemIntegrator::advance (integrator.h:184-249) of every node to the cycle's end time with the
// integrator core K: odeint Cash-Karp controller (stepper_wrapper.h:112-163), RKIntegratorCore
// (adapt_rk.h:217-298), fixed Cash-Karp (stepper_wrapper.h:240-255) or Euler (euler.h:54-62).
// Loop is flattened to one try_step attempt per iteration so that a rejected node stays in step with its
// neighbours in the wavefront.
//
// Bound by the FP64 issue rate and, with few wavefronts, by the chain of dependent operations of one attempt (six
// right-hand sides with an LDS exchange each). The plain instantiation fits 256 registers, two wavefronts per SIMD (12 B
// of scratch for Cash-Karp and G = 8, 20 B in the mixed Cash-Karp and RKF45 kernels, none else): eight compartments, no
// feature code (the arguments of sin, cos and pow alone took a third of 107 KB of code, above the 64 KB instruction
// cache; 15 KB now), the scalars of a step in LDS (Cold). 512 runs x 400 nodes x 6 groups at 1e-10: 580 us per half-day
// against 1030 us for ten compartments at one wavefront per SIMD; a single 400-node graph 39 us against 50 us. Two
// wavefronts with the cold scalars in registers spilled 25 values per attempt: 768 us and 51 us.
constexpr uint32_t kMaxAttemptsPerPhase = 1u << 20;

template <int G, int K, int M>
__device__ __forceinline__ void node_body(const LaunchDev& ld, InstDev* __restrict__ inst, double* wx)
{
    using X         = Comps<M>;
    constexpr int N = X::N;
    Lane<G, M> L;
    Seg* cp = load_lane(ld, L, wx);
    if (!cp) {
        return;
    }
    Seg& c     = *cp;
    InstDev& I = inst[L.inst];
    if (!I.c_active) {
        return;
    }
    double* yp = c.y + (size_t(L.node) * G + L.age) * NC;
    double y[N];
    {
        const double2* y2 = reinterpret_cast<const double2*>(yp);
#pragma unroll
        for (int q = 0; q < NC / 2; ++q) {
            const double2 v = y2[q];
            if (X::of(2 * q) >= 0) {
                y[X::of(2 * q)] = v.x;
            }
            if (X::of(2 * q + 1) >= 0) {
                y[X::of(2 * q + 1)] = v.y;
            }
        }
    }
    double t            = c.tnode[L.node];
    double dt           = c.dtnode[L.node];
    const double t_phase = I.c_t1;
    // Without dynamic NPIs the phase is one SystemIntegrator::advance to c_t1; with them it is the pieces of
    // osecir::Simulation::advance (at most a day each, ending at NPI ends), each starting with the NPI check
    const bool npi      = M == NPIS && (L.flags & NF_NPI) != 0;
    double t_loop       = t; // osecir::Simulation::advance's loop time (model.h:301)
    auto cold           = [&](Cold k) -> double& {
        return L.cold[k * BLOCK];
    };
    auto cold_int = [&](Cold k) {
        return reinterpret_cast<int32_t*>(&L.cold[k * BLOCK]);
    };
    cold(COLD_ABS)        = I.abs_tol;
    cold(COLD_REL)        = I.rel_tol;
    cold(COLD_DT_MAX)     = I.dt_max;
    cold(COLD_DT_MIN)     = I.dt_min;
    cold(COLD_DT_RESTORE) = 0.0;
    cold(COLD_TMAX)       = t_phase;
    // season of the next k1: an accepted step ends at t + h, where its fifth stage (c5 = 1 in both tableaus)
    // evaluated the season already
    cold(COLD_SEASON) = season_at(L, t);
    // output days strictly inside this phase are interpolated here; a day at the phase end is written
    // after the edge action
    // (the first is the day after the node's own time: a fixed-step node can end a phase just below the day
    // the phase ended on, and then its first step here encloses that day)
    cold_int(COLD_DAYS)[0]   = max(0, int(floor(t)) + 1 - I.day0);
    cold_int(COLD_DAYS)[1]   = I.ndays;
    cold_int(COLD_COUNTS)[0] = 0;
    cold_int(COLD_COUNTS)[1] = 0;
    const double eps = 1e-12;

    bool active = false;
    bool fresh  = true; // the next attempt begins a step
    bool valid = true, first = true, stalled = false;
    double k1[N];
    for (;;) { // pieces of the node advance (one without dynamic NPIs)
        bool changed = false;
        if constexpr (M == NPIS) {
            if (npi) {
                cold(COLD_TMAX) = t_loop + npi_piece(c, L, I, y, t_loop, t_phase, changed);
            }
        }
        if (I.c_action == 2 && (first || changed)) {
            // return coefficients of this node as a destination: its state after the departures, at the
            // departure time (the `pop` of calculate_mobility_returns, metapopulation_mobility_instant.h:460-471),
            // with the contact matrix as it is after the node's NPI checks of this phase
            if constexpr (M == NPIS) {
                double pop[N];
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    pop[i] = first ? y[i] : c.npi[L.node].y0[L.age * NC + i];
                    if (first && npi) {
                        c.npi[L.node].y0[L.age * NC + i] = y[i];
                    }
                }
                return_coefficients(c, L, I, pop);
            }
            else {
                return_coefficients(c, L, I, y);
            }
        }
        first           = false;
        cold(COLD_SPAN) = cold(COLD_TMAX) - t;
        active          = fabs((cold(COLD_TMAX) - t) / cold(COLD_SPAN)) > eps;
        fresh           = true;
        rhs(c, L, y, t, cold(COLD_SEASON), k1);
        while (active) {
            int32_t* counts = cold_int(COLD_COUNTS);
            if (uint32_t(counts[1]) >= kMaxAttemptsPerPhase) {
                // a step size driven below any progress (dt_min ~ DBL_MIN with a persistent error): stop this
                // node and report instead of spinning; the reference would not terminate here
                if (L.age == 0) {
                    I.status = MGO_ERR_OUT_OF_RANGE;
                }
                stalled = true;
                break;
            }
            if (fresh) {
                const double left = cold(COLD_TMAX) - t;
                if (dt > left) {
                    cold(COLD_DT_RESTORE) = dt;
                    dt                    = left;
                    cold(COLD_DT_MIN)     = fmin(left, cold(COLD_DT_MIN));
                }
                fresh = false;
                valid = true;
                if (K == MGO_INTEGRATOR_RKF45) {
                    dt = fmin(dt, cold(COLD_DT_MAX));
                }
            }
            double yo[N], er[N];
            bool done       = true;
            const double ta = t;
            // scale of the next step size is factor (clamped below by factor_min), or 1
            double base = 1.0, power = 0.0, factor_min = 0.0;
            bool scale = false;
            ++counts[1];
            if (K == MGO_INTEGRATOR_CASH_KARP54) {
                if (dt < cold(COLD_DT_MIN)) {
                    valid = false;
                    dt    = cold(COLD_DT_MIN);
                }
                if (!(dt - cold(COLD_DT_MAX) <= DBL_EPSILON)) {
                    dt = cold(COLD_DT_MAX); // check_step_size_limit: rejected without a step
                    continue;
                }
                cash_karp_stages(c, L, y, k1, t, dt, yo, er, true);
                // max_i |err_i| / (abs + rel (|y_i| + dt |k1_i|)) (odeint default_error_checker): the index of
                // the largest quotient by cross-multiplied comparison, then one division
                double en = 0.0, ed = 1.0;
                const double abs_tol = cold(COLD_ABS), rel_tol = cold(COLD_REL);
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const double n = fabs(er[i]);
                    const double d = fma(rel_tol, fma(dt, fabs(k1[i]), fabs(y[i])), abs_tol);
                    if (n * ed > en * d) {
                        en = n;
                        ed = d;
                    }
                }
                double e = en / ed;
                // maximum over the node's lanes through the wavefront's slots (the same fmax order)
                L.wx[threadIdx.x % WAVE] = e;
                wave_sync();
                e = L.wx[L.base];
#pragma unroll
                for (int j = 1; j < G; ++j) {
                    e = fmax(e, L.wx[L.base + j]);
                }
                wave_sync();
                // rejected: dt *= max(0.9 e^(-1/3), 0.2); accepted below 0.5: dt *= 0.9 max(5^-5, e)^(-1/5)
                const bool rejected = e > 1.0;
                base                = rejected ? e : fmax(1.0 / 3125.0, e);
                power               = rejected ? -1.0 / 3.0 : -0.2;
                factor_min          = rejected ? 0.2 : 0.0;
                scale               = rejected || e < 0.5;
                done                = !(rejected && valid);
                if (!rejected) {
                    t += dt;
                    cold(COLD_SEASON) = stage_season<3>(L);
                }
                else if (done) {
                    t += cold(COLD_DT_MIN);
                    cold(COLD_SEASON) = season_at(L, t);
                }
            }
            else if (K == MGO_INTEGRATOR_RKF45) {
                if (dt < cold(COLD_DT_MIN)) {
                    valid = false;
                    dt    = cold(COLD_DT_MIN);
                }
                rkf45_stages(c, L, y, k1, t, dt, yo, er);
                const double abs_tol = cold(COLD_ABS), rel_tol = cold(COLD_REL);
                bool conv = true;
                double q  = INFINITY;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const double ep = fma(fabs(yo[i]), rel_tol, abs_tol);
                    conv            = conv && (er[i] <= ep);
                    q               = fmin(q, ep / er[i]);
                }
                conv  = group_all<G>(conv, L.base);
                base  = group_min<G>(q, L.base);
                power = 1.0 / 5.0;
                scale = true;
                done  = conv || !valid;
                if (done) {
                    t += dt;
                    cold(COLD_SEASON) = stage_season<3>(L);
                }
            }
            else if (K == MGO_INTEGRATOR_CASH_KARP54_FIXED) {
                cash_karp_stages(c, L, y, k1, t, dt, yo, er, false);
                t += dt;
                cold(COLD_SEASON) = stage_season<3>(L);
            }
            else { // Euler
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    yo[i] = fma(dt, k1[i], y[i]);
                }
                t += dt;
                cold(COLD_SEASON) = season_at(L, t);
            }
            // k1 of the next attempt, before its step size is known: independent of the power below, whose chain of
            // dependent operations it overlaps (after a rejection it is the same k1 again)
            double yn[N];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                yn[i] = done ? yo[i] : y[i];
            }
            rhs(c, L, yn, t, cold(COLD_SEASON), k1);
            if (K == MGO_INTEGRATOR_CASH_KARP54 || K == MGO_INTEGRATOR_RKF45) {
                const double factor = 0.9 * step_pow(base, power);
                const double scaled = fmin(dt * fmax(factor, factor_min), cold(COLD_DT_MAX));
                dt                  = scale ? scaled : dt;
                if (done) {
                    dt = fmax(dt, cold(COLD_DT_MIN));
                }
            }
            if (done) {
                ++counts[0];
                // interpolate_simulation_result (analyze_result.h:235-252): days in (ta, t] strictly inside
                // the phase
                int32_t* days = cold_int(COLD_DAYS);
                while (days[0] < days[1]) {
                    const double dd = double(days[0] + I.day0);
                    if (!(dd <= t && dd < I.c_t1 - 1e-10)) {
                        break;
                    }
                    if (dd > ta) {
                        const double w = (dd - ta) / (t - ta);
                        gdouble* op    = out_ptr(I, c.nodep[L.node].local, L.age, G, days[0]);
#pragma unroll
                        for (int i = 0; i < NC; ++i) {
                            const int x = X::of(i);
                            op[i]       = x < 0 ? 0.0 : lerp_ref(y[x < 0 ? 0 : x], yo[x < 0 ? 0 : x], w);
                        }
                    }
                    ++days[0];
                }
                active = fabs((cold(COLD_TMAX) - t) / cold(COLD_SPAN)) > eps;
                if (!active && I.c_out_day >= 0) {
                    // the last step of the phase (so far): the phase-end day is interpolated from it after the
                    // edge action (write_phase_end_day)
                    const double dd = double(I.c_out_day + I.day0);
                    double* pr      = c.yint + (size_t(L.node) * G + L.age) * YINT_STRIDE;
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        pr[i] = X::of(i) < 0 ? 0.0 : y[X::of(i) < 0 ? 0 : X::of(i)];
                    }
                    pr[YINT_W] = (t >= dd) ? (dd - ta) / (t - ta) : -1.0;
                }
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    y[i] = yo[i];
                }
                fresh = true;
            }
        }
        if (!npi || stalled) {
            break;
        }
        // end of a piece: SystemIntegrator::advance's exit (integrator.h:244-248), then the next piece
        dt                    = fmax(dt, cold(COLD_DT_RESTORE));
        cold(COLD_DT_RESTORE) = 0.0;
        cold(COLD_DT_MIN)     = I.dt_min;
        t_loop                = cold(COLD_TMAX);
        if (!(t_loop < t_phase)) {
            break;
        }
    }
    dt = fmax(dt, cold(COLD_DT_RESTORE));
    if (L.age == 0) {
        c.tnode[L.node]  = t;
        c.dtnode[L.node] = dt;
        c.steps[L.node] += uint32_t(cold_int(COLD_COUNTS)[0]);
        c.attempts[L.node] += uint32_t(cold_int(COLD_COUNTS)[1]);
    }
    double ye[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        ye[i] = X::of(i) < 0 ? 0.0 : y[X::of(i) < 0 ? 0 : X::of(i)];
    }
    double D = 0.0;
    if constexpr (M == NPIS) {
        if ((L.flags & NF_OUT_DAMP) && I.c_action != 0) {
            D = out_damping(c, L, I, ye);
        }
    }
    if (I.c_action == 2) {
        store_planes(c.ypre, size_t(c.num_nodes) * G, size_t(L.node) * G + L.age, ye);
        return; // the return phase writes the state and the day
    }
    if (I.c_action == 1) {
        // the departure phase adds the arrivals and writes the day
        const double nd = (M != PLAIN && (L.flags & NF_DETECTION)) ? detect_nondetection(c.nodep[L.node], t_phase) : 1.0;
        leave(c, L, I, mobility_factor(L, ye[INS]), nd, D, ye);
    }
    else if (I.c_out_day >= 0) {
        write_phase_end_day<G>(c, I, size_t(L.node) * G + L.age, c.nodep[L.node].local, L.age, ye);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        yp[i] = ye[i];
    }
}

// ------------------------------------------------------------------------------- edge phase
// Lane -> (segment, node, age group) without loading the lane's coefficients (edge kernels need none).
template <int G>
__device__ __forceinline__ Seg* lane_map(const LaunchDev& ld, int& node, int& age, int& base)
{
    constexpr int NPW = WAVE / G;
    const int lb      = xcd_block();
    if (lb >= ld.num_blocks) {
        return nullptr;
    }
    const int seg = ld.block_seg[lb];
    if (seg < 0) {
        return nullptr;
    }
    Seg* c = segment(ld, seg);
    const int wave  = (lb - ld.block_first[seg]) * (BLOCK / WAVE) + int(threadIdx.x) / WAVE;
    const int lane  = int(threadIdx.x) % WAVE;
    const int grp   = lane / G;
    age             = lane - grp * G;
    node            = wave * NPW + grp;
    base            = grp * G;
    if (grp >= NPW || node >= c->num_nodes) {
        return nullptr;
    }
    return c;
}

// coefficient of entry k of the in- or out-entries for compartments i of age group `age`, at the departure time
struct EdgeCoef {
    double c;          // uniform coefficient
    const double* vec; // else the coefficients of the lane's age group, and their minima (or NULL)
    const double* vmin;
    double D;
};

__device__ __forceinline__ EdgeCoef edge_coef(Est& es, const EdgeEnt& e, const double* mn, int k,
                                              double D, int G, int age)
{
    EdgeCoef r{e.cval, nullptr, nullptr, D};
    if (e.cidx < 0) {
        if (D != 0.0) {
            r.c = damped(e.cval, mn ? mn[k] : 0.0, D);
        }
    }
    else {
        const size_t off = size_t(e.cidx) * G * NC + size_t(age) * NC;
        r.vec            = es.cvec + off;
        r.vmin           = es.cvec_min ? es.cvec_min + off : nullptr;
    }
    return r;
}

__device__ __forceinline__ double coef_of(const EdgeCoef& e, int i)
{
    if (!e.vec) {
        return e.c;
    }
    return e.D != 0.0 ? damped(e.vec[i], e.vmin ? e.vmin[i] : 0.0, e.D) : e.vec[i];
}

// rates of one lane's Euler step of returning travelers (calculate_mobility_returns,
// metapopulation_mobility_instant.h:460-471; euler.h:54-62), one per flow with the flow's source compartment;
// f[0] = the force of infection
constexpr int NFLOW = 15;
__device__ __forceinline__ constexpr int flow_src(int f)
{
    constexpr int src[NFLOW] = {S, E, INS, INS, INSC, INSC, ISY, ISY, ISYC, ISYC, ISEV, ISEV, ISEV, ICR, ICR};
    return src[f];
}
// the flow's rate in the lane coefficients (f >= 1)
__device__ __forceinline__ constexpr int flow_rate(int f)
{
    constexpr int rate[NFLOW] = {-1,          LC_E,      LC_INS_ISY, LC_INS_R,    LC_INS_ISY,
                                 LC_INS_R,    LC_ISY_ISEV, LC_ISY_R, LC_ISY_ISEV, LC_ISY_R,
                                 LC_ISEV_ICR, LC_ISEV_R, LC_ISEV_D,  LC_ICR_D,    LC_ICR_R};
    return rate[f];
}

__device__ __forceinline__ void lane_rates(Seg& c, bool icu, size_t lane, double (&w)[NFLOW])
{
    static_assert(LC_ICR_R == 9 && NUM_LC % 2 == 0, "the flow rates are the first ten lane coefficients");
    double lc[10];
    const double2* p = reinterpret_cast<const double2*>(c.lcoef + lane * NUM_LC);
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        const double2 v = p[q];
        lc[2 * q]       = v.x;
        lc[2 * q + 1]   = v.y;
    }
    w[0] = c.kap[lane];
#pragma unroll
    for (int f = 1; f < NFLOW; ++f) {
        w[f] = lc[flow_rate(f)];
    }
    if (icu) {
        const double2 k = c.kicu[lane];
        w[10]           = k.x;
        w[12]           = k.y;
    }
}

// change of the travelers m over one Euler step h with rates w; `dm` in the Flows order of get_derivatives
__device__ __forceinline__ void euler_change(const double (&m)[NC], const double (&w)[NFLOW], double h,
                                             double (&dm)[NC])
{
#pragma clang fp contract(off)
    double f[NFLOW];
#pragma unroll
    for (int k = 0; k < NFLOW; ++k) {
        f[k] = w[k] * m[flow_src(k)];
    }
    dm[S]    = h * (-f[0]);
    dm[E]    = h * (f[0] - f[1]);
    dm[INS]  = h * ((f[1] - f[2]) - f[3]);
    dm[INSC] = h * (-f[4] - f[5]);
    dm[ISY]  = h * ((f[2] - f[6]) - f[7]);
    dm[ISYC] = h * ((f[4] - f[8]) - f[9]);
    dm[ISEV] = h * ((((f[6] + f[8]) - f[10]) - f[11]) - f[12]);
    dm[ICR]  = h * ((f[10] - f[13]) - f[14]);
    dm[R]    = h * (((((f[3] + f[5]) + f[7]) + f[9]) + f[11]) + f[14]);
    dm[D]    = h * (f[12] + f[13]);
}

template <int G>
__device__ __forceinline__ bool group_any(bool v, int base)
{
    return ((__ballot(v) >> base) & ((1ull << G) - 1)) != 0;
}

// MobilityEdge::apply_mobility return branch fix-up (metapopulation_mobility_instant.h:576-596): every
// compartment of the age group that would go negative at the destination is taken from the group's
// largest remaining compartment instead (remaining computed once, first maximum wins).
__device__ __forceinline__ bool fixup_negative(const double (&y)[NC], double (&m)[NC])
{
    double rem[NC];
    bool neg = false;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        rem[i] = y[i] - m[i];
        neg    = neg || (rem[i] < 0);
    }
    if (neg) {
        int mx = 0;
#pragma unroll
        for (int q = 1; q < NC; ++q) {
            if (rem[q] > rem[mx]) {
                mx = q;
            }
        }
        for (int j = 0; j < NC; ++j) {
            if (rem[j] < 0) {
                m[mx] -= rem[j];
                m[j] += rem[j];
            }
        }
    }
    return neg;
}

constexpr int EDGE_WAVES   = 3; // wavefronts per SIMD of the edge kernel (20 B of scratch, 28 B in the mixed one)
constexpr int DEPART_ROWS  = 4; // departure rows in flight per lane
constexpr int RETURN_EDGES = 8; // forces of infection in flight per lane

// Arrivals at c_t1 (metapopulation_mobility_instant.h:605-621): every edge (s, d) adds its source's departure
// row times its coefficient to d. The lane sums its age group over the node's in-edges, in the reference's
// order; the sum is kept for the returns (come_home).
//
// Bound by the gathered rows: 80 B per lane and edge, 4.9 GB per launch for 512 runs of a 400-node, 20k-edge
// graph with 6 groups. The rows lie in planes of compartment pairs: a wavefront that holds one graph node of
// several runs reads one contiguous kilobyte per pair, where rows of 96 B touched every line of the rows five
// times. Measured there: 300 us (16 TB/s from the L2 caches) against 470 us for the walk over rows and out-edges; one
// run alone, bound by the gathers' latency: 25 us with the entries a batch ahead, 33 us without (6 or 8 rows in
// flight are no faster).
template <int G>
__device__ __forceinline__ void arrive(Seg& c, InstDev& I, int node, int age)
{
    Est& es = edge_struct(c, I.estruct);
    const int v             = c.nodep[node].local;
    const int in_b = es.in_ptr[v], in_e = es.in_ptr[v + 1];
    const size_t lane     = size_t(node) * G + age;
    const size_t src_base = size_t(I.node_base) * G + age;   // lane of local node 0
    const size_t src_step = size_t(I.node_stride) * G;       // lanes between local nodes
    const size_t np       = size_t(c.num_nodes) * G;         // lanes of a plane
    const double2* dep    = c.dep;
    double M[NC] = {};
    if (es.out_sum) {
        const double* mn = es.in_min;
        constexpr int U  = DEPART_ROWS;
        // U edges: their sources and coefficients (loaded a batch ahead), the rows, the sums in edge order
        int32_t src[U];
        double w[U];
        auto entries = [&](int k) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int ku = min(k + u, in_e - 1);
                src[u]       = es.in_src[ku];
                w[u]         = es.in_c[ku];
            }
        };
        auto batch = [&](int k, auto full) {
            double2 r[U][NC / 2];
            double wk[U];
            size_t sl[U];
#pragma unroll
            for (int u = 0; u < U; ++u) { // no branch between the loads
                sl[u] = src_base + size_t(src[u]) * src_step;
                wk[u] = w[u];
#pragma unroll
                for (int q = 0; q < NC / 2; ++q) {
                    r[u][q] = dep[size_t(q) * np + sl[u]];
                }
            }
            if (c.out_d) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const double D = c.out_d[sl[u]];
                    if (D != 0.0) {
                        wk[u] = damped(wk[u], mn ? mn[min(k + u, in_e - 1)] : 0.0, D);
                    }
                }
            }
            if (decltype(full)::value) {
                entries(k + U);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (!decltype(full)::value && k + u >= in_e) {
                    continue;
                }
#pragma unroll
                for (int q = 0; q < NC / 2; ++q) {
                    M[2 * q]     = fma(wk[u], r[u][q].x, M[2 * q]);
                    M[2 * q + 1] = fma(wk[u], r[u][q].y, M[2 * q + 1]);
                }
            }
        };
        if (in_b < in_e) {
            entries(in_b);
            int k = in_b;
            for (; k + U <= in_e; k += U) {
                batch(k, std::true_type{});
            }
            if (k < in_e) {
                batch(k, std::false_type{});
            }
        }
    }
    else {
        for (int k = in_b; k < in_e; ++k) {
            const EdgeEnt e   = es.in_ent[k];
            const size_t sl   = src_base + size_t(e.nbr) * src_step;
            const EdgeCoef ec = edge_coef(es, e, es.in_min, k, c.out_d ? c.out_d[sl] : 0.0, G, age);
            double r[NC];
            load_planes(dep, np, sl, r);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                M[i] = fma(coef_of(ec, i), r[i], M[i]);
            }
        }
    }
    store_planes(c.arr, np, lane, M);
    double* yp = c.y + lane * NC;
    double y[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        y[i]  = yp[i] + M[i];
        yp[i] = y[i];
    }
    if (I.c_out_day >= 0) {
        write_phase_end_day<G>(c, I, lane, v, age, y);
    }
}

// Constant part of the returns of a node as a source (once per batch): per flow, the sum over its out-edges of
// the coefficient times the destination's rate, in planes; wmin: the same with the minimum coefficients.
template <int G>
__device__ __forceinline__ void weights_body(const LaunchDev& ld, InstDev* __restrict__ inst, int inst_offset)
{
    int node, age, base;
    Seg* cp = lane_map<G>(ld, node, age, base);
    if (!cp) {
        return;
    }
    Seg& c  = *cp;
    const InstDev& I = inst[c.nodep[node].inst - inst_offset];
    if (I.estruct < 0) {
        return;
    }
    Est& es = edge_struct(c, I.estruct);
    const int v             = c.nodep[node].local;
    const size_t lane       = size_t(node) * G + age;
    const size_t src_base   = size_t(I.node_base) * G + age;
    const size_t src_step   = size_t(I.node_stride) * G;
    const size_t np         = size_t(c.num_nodes) * G;
    double w[NFLOW] = {}, wm[NFLOW] = {};
    for (int k = es.out_ptr[v]; k < es.out_ptr[v + 1]; ++k) {
        const EdgeEnt e  = es.out_ent[k];
        const double* lc = c.lcoef + (src_base + size_t(e.nbr) * src_step) * NUM_LC;
        const size_t off = size_t(e.cidx < 0 ? 0 : e.cidx) * G * NC + size_t(age) * NC;
#pragma unroll
        for (int f = 1; f < NFLOW; ++f) {
            const int i       = flow_src(f);
            const double rate = lc[flow_rate(f)];
            w[f]              = fma(e.cidx < 0 ? e.cval : es.cvec[off + i], rate, w[f]);
            if (c.wmin) {
                const double mn = e.cidx < 0 ? (es.out_min ? es.out_min[k] : 0.0)
                                             : (es.cvec_min ? es.cvec_min[off + i] : 0.0);
                wm[f]           = fma(mn, rate, wm[f]);
            }
        }
    }
    auto put = [&](double2* p, const double (&x)[NFLOW]) {
        if (c.wplanes == 7) {
#pragma unroll
            for (int q = 0; q < 7; ++q) {
                p[size_t(q) * np + lane] = double2{x[1 + 2 * q], x[2 + 2 * q]};
            }
        }
        else { // one coefficient per edge: the confirmed flows have the weights of the unconfirmed ones
            p[0 * np + lane] = double2{x[1], x[2]};
            p[1 * np + lane] = double2{x[3], x[6]};
            p[2 * np + lane] = double2{x[7], x[10]};
            p[3 * np + lane] = double2{x[11], x[12]};
            p[4 * np + lane] = double2{x[13], x[14]};
        }
    };
    put(c.wst, w);
    if (c.wmin) {
        put(c.wmin, wm);
    }
}

__device__ __forceinline__ void load_weights(Seg& c, const double2* p, size_t np, size_t lane,
                                             double (&x)[NFLOW])
{
    if (c.wplanes == 7) {
#pragma unroll
        for (int q = 0; q < 7; ++q) {
            const double2 t = p[size_t(q) * np + lane];
            x[1 + 2 * q]    = t.x;
            x[2 + 2 * q]    = t.y;
        }
        return;
    }
    const double2 a = p[0 * np + lane], b = p[1 * np + lane], d = p[2 * np + lane], e = p[3 * np + lane],
                  g = p[4 * np + lane];
    x[1]  = a.x;
    x[2]  = x[4] = a.y;
    x[3]  = x[5] = b.x;
    x[6]  = x[8] = b.y;
    x[7]  = x[9] = d.x;
    x[10] = d.y;
    x[11] = e.x;
    x[12] = e.y;
    x[13] = g.x;
    x[14] = g.y;
}

// Whether a compartment may fall below zero while a node's in-edges are taken off one by one, where some rate exceeds
// 1 / h. An edge's travelers after the step are what stays of them (negative if the rate is steep) and what flows in,
// both linear in nonnegative numbers with the node's own rates: no sum over some of the edges exceeds the inflow of
// all and, unless the rate is steep, what stays of all. y: state before the returns; m: all arrivals, dm: their
// change, w: the node's rates; home: the homecomings, added at once between two in-edges.
__device__ __forceinline__ bool falls_short(const double (&y)[NC], const double (&m)[NC], const double (&dm)[NC],
                                            const double (&w)[NFLOW], double h, const double (&home)[NC])
{
    double out[NC] = {};
#pragma unroll
    for (int f = 0; f < NFLOW; ++f) {
        out[flow_src(f)] += w[f];
    }
    bool low = false;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const double most = h * out[i] > 1.0 ? fma(h * out[i], m[i], dm[i]) : m[i] + dm[i];
        low               = low || !((y[i] - most) + fmin(home[i], 0.0) >= 0.0);
    }
    return low;
}

// All travelers that come home to a lane's node, each after its destination's Euler step: the lane's departure
// row stepped with the sums over the out-edges of coefficient times rate. k0: the sum of the forces of infection;
// k10, k12: those of the ICU-adjusted rates (used with ICU limits, else the kept constants).
template <int G>
__device__ __forceinline__ void homecoming(Seg& c, const InstDev& I, Est& es, int v,
                                           size_t lane, int age, double D_v, double k0, double k10, double k12,
                                           double (&home)[NC])
{
#pragma clang fp contract(off)
    const size_t np = size_t(c.num_nodes) * G;
    double m[NC], dm[NC], w[NFLOW];
    load_planes(c.dep, np, lane, m);
    load_weights(c, c.wst, np, lane, w);
    if (D_v != 0.0) {
        double wm[NFLOW];
        load_weights(c, c.wmin, np, lane, wm);
#pragma unroll
        for (int f = 1; f < NFLOW; ++f) {
            w[f] = damped(w[f], wm[f], D_v);
        }
    }
    w[0] = k0;
    if (I.icu) {
        w[10] = k10;
        w[12] = k12;
    }
    euler_change(m, w, I.c_step, dm);
    if (es.out_sum) {
        double sum = es.out_sum[v];
        if (D_v != 0.0) {
            sum = damped(sum, es.out_min_sum ? es.out_min_sum[v] : 0.0, D_v);
        }
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            home[i] = sum * m[i] + dm[i];
        }
    }
    else {
        const size_t off = (size_t(v) * G + age) * NC;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            double sum = es.out_vsum[off + i];
            if (D_v != 0.0) {
                sum = damped(sum, es.out_vmin_sum ? es.out_vmin_sum[off + i] : 0.0, D_v);
            }
            home[i] = sum * m[i] + dm[i];
        }
    }
}

// travelers of one edge after the Euler step at their destination: the source's departure row m in, the
// returning travelers out
__device__ __forceinline__ void edge_return(const EdgeCoef& ec, const double (&rates)[NFLOW], double h, double (&m)[NC])
{
#pragma clang fp contract(off)
    double dm[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        m[i] = m[i] * coef_of(ec, i);
    }
    euler_change(m, rates, h, dm);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        m[i] = m[i] + dm[i];
    }
}

// Returns at c_t1 of the travelers that left at c_tdep (metapopulation_mobility_instant.h:568-603) in closed
// form. The Euler step of the travelers is linear in them and, per flow, in the destination's rate. So all
// travelers that a node sends home are one Euler step of its arrivals (the sum that the departure phase kept)
// with its own rates, and all that come home to it are its departure row stepped with the sums over its
// out-edges of coefficient times rate: those of the constant rates are kept per lane (weights_body), the
// force of infection (and, with ICU limits, two more) is summed here, 8 B per lane and edge instead of the
// 2 x 96 B per lane and edge that a walk over all edges gathers. Measured (512 runs, 400 nodes, 20k edges, 6
// groups): 304 us per launch against 1315 us for the walk (350 us, and 30 instead of 17 us for one run, with a
// branch on the ICU limits between the loads, which then waited for each other).
//
// The fix-up acts where a compartment of a destination falls below zero while its in-edges are taken off one
// by one. With nonnegative returning travelers every partial difference is at least the full one, ypre - arrivals
// (homecomings only add), so a node whose full difference is nonnegative has none. The others are marked and
// walk their edges one by one (walk_node, settle_body). The step's factor of a compartment, 1 - h * (sum of its
// outgoing rates), keeps travelers nonnegative if it is: coefficients and constant rates are checked on the host
// (InstDev::general), the departure rows as they are written (InstDev::fx_neg). Only S, whose rate is the force
// of infection, may step below zero in earnest (more than 1 / h infections per day at a peak). It has no inflow,
// so all in-edges of a node change it in one direction and its extremes are at the ends of the sequence and at
// the homecomings: ypre, ypre - arrivals and both with the homecomings added. Runs in which another rate exceeds
// 1 / h (STEEP) take the bound of falls_short instead.
template <int G, bool ANY_STEEP>
__device__ __forceinline__ void come_home(Seg& c, InstDev& I, int node, int age, int base)
{
    Est& es = edge_struct(c, I.estruct);
    const int v             = c.nodep[node].local;
    const size_t lane       = size_t(node) * G + age;
    const size_t src_base   = size_t(I.node_base) * G + age;
    const size_t src_step   = size_t(I.node_stride) * G;
    const size_t np         = size_t(c.num_nodes) * G;
    const double h          = I.c_step;
    const bool icu          = I.icu != 0;
    const double D_v        = c.out_d ? c.out_d[lane] : 0.0;
    // sums over the out-edges: force of infection of the destinations, and their ICU-adjusted rates
    double w[NFLOW];
    double k0 = 0.0, k10 = 0.0, k12 = 0.0, k_min = 0.0;
    const int out_b = es.out_ptr[v], out_e = es.out_ptr[v + 1];
    if (es.out_sum) {
        // U edges at a time, their loads in flight together; the sums in edge order
        constexpr int U = RETURN_EDGES;
        for (int k = out_b; k < out_e; k += U) {
            double cf[U], kd[U];
            size_t dl[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int ku = min(k + u, out_e - 1);
                dl[u]        = src_base + size_t(es.out_dst[ku]) * src_step;
                cf[u]        = es.out_c[ku];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                kd[u] = c.kap[dl[u]];
            }
            if (D_v != 0.0) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    cf[u] = damped(cf[u], es.out_min ? es.out_min[min(k + u, out_e - 1)] : 0.0, D_v);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool in = k + u < out_e;
                k0            = in ? fma(cf[u], kd[u], k0) : k0;
                k_min         = fmin(k_min, kd[u]); // the last edge again past the end
            }
            if (icu) {
                double2 ri[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    ri[u] = c.kicu[dl[u]];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool in = k + u < out_e;
                    k10           = in ? fma(cf[u], ri[u].x, k10) : k10;
                    k12           = in ? fma(cf[u], ri[u].y, k12) : k12;
                }
            }
        }
    }
    else {
        for (int k = out_b; k < out_e; ++k) {
            const EdgeEnt e   = es.out_ent[k];
            const size_t dl   = src_base + size_t(e.nbr) * src_step;
            const EdgeCoef ec = edge_coef(es, e, es.out_min, k, D_v, G, age);
            const double kd   = c.kap[dl];
            k0                = fma(coef_of(ec, S), kd, k0);
            k_min             = fmin(k_min, kd);
            if (icu) {
                const double2 r = c.kicu[dl];
                k10             = fma(coef_of(ec, ISEV), r.x, k10);
                k12             = fma(coef_of(ec, ISEV), r.y, k12);
            }
        }
    }
    // travelers sent home
    double y[NC], m[NC], dm[NC];
    load_planes(c.ypre, np, lane, y);
    load_planes(c.arr, np, lane, m);
    lane_rates(c, icu, lane, w);
    euler_change(m, w, h, dm);
    bool mark        = I.fx_neg != 0 || !(w[0] >= 0.0) || !(k_min >= 0.0);
    const double y_s = y[S];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        y[i] = y[i] - (m[i] + dm[i]);
        mark = mark || !(y[i] >= 0.0);
    }
    // travelers coming home
    double home[NC];
    homecoming<G>(c, I, es, v, lane, age, D_v, k0, k10, k12, home);
    if (ANY_STEEP && I.general == STEEP) {
        double ypre[NC];
        load_planes(c.ypre, np, lane, ypre);
        load_planes(c.arr, np, lane, m);
        lane_rates(c, icu, lane, w);
        euler_change(m, w, h, dm);
        mark = mark || falls_short(ypre, m, dm, w, h, home);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        y[i] = y[i] + home[i];
    }
    mark = mark || !(y_s >= 0.0) || !(y_s + home[S] >= 0.0) || !(y[S] >= 0.0);
    if (group_any<G>(mark, base) && age == 0 && out_e - out_b + (es.in_ptr[v + 1] - es.in_ptr[v]) > 0) {
        c.fx_dirty[node] = I.fx_epoch; // walks its edges in pass 1
        if (__hip_atomic_load(&I.fx_changed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <= SETTLE_BLOCK / WAVE) {
            atomicAdd(&I.fx_changed, 1); // it only matters whether there are more than that
        }
    }
    double* yp = c.y + lane * NC;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        yp[i] = y[i];
    }
    if (I.c_out_day >= 0) {
        write_phase_end_day<G>(c, I, lane, v, age, y);
    }
}

// Edge action of the cycle: arrivals or returns, one launch for both (a cycle has one or the other, or some runs
// each; an idle launch costs about 4.5 us). ANY_STEEP: instantiation for launches with steep rates (in all launches,
// the code for them had 68 instead of 20 B of registers spilled).
template <int G, bool ANY_STEEP>
__device__ __forceinline__ void edge_body(const LaunchDev& ld, InstDev* __restrict__ inst)
{
    int node, age, base;
    Seg* cp = lane_map<G>(ld, node, age, base);
    if (!cp) {
        return;
    }
    Seg& c     = *cp;
    InstDev& I = inst[c.nodep[node].inst];
    if (!I.c_active) {
        return;
    }
    if (I.c_action == 1) {
        arrive<G>(c, I, node, age);
    }
    else if (I.c_action == 2 && I.general != GENERAL) {
        come_home<G, ANY_STEEP>(c, I, node, age, base);
    }
}

// newest fix-up record version of an in-edge written in [lo, hi] (slot, -1 = unfixed or none)
__device__ __forceinline__ int32_t record_slot(const FxRec* r, int32_t lo, int32_t hi)
{
    const FxRec a = r[0];
    const FxRec b = r[1];
    const bool va = a.tag >= lo && a.tag <= hi;
    const bool vb = b.tag >= lo && b.tag <= hi;
    if (va && (!vb || a.tag > b.tag)) {
        return a.slot;
    }
    return vb ? b.slot : -1;
}

// Return walk of one node by one wavefront (returns at c_t1 of the travelers that left at c_tdep,
// metapopulation_mobility_instant.h:568-603) from the pre-return state, the node's edges in the reference's
// global (start, end) order: in-edges of lower sources, homecomings, the other in-edges.
//
// The fix-up of edge (s, d) depends on d's state at that point of the sequence, which includes d's
// earlier out-edges (d, x) with their own fix-ups decided at x. Pass p applies the fix-ups of the node's
// in-edges locally and takes the out-edge vectors from the records as of pass p-1 (pass 0: unfixed). The
// dependencies follow the global edge order (a DAG), so the records reach the reference's sequential
// values after at most (longest dependency chain + 1) passes; a pass in which no record changes
// reproduces the sequential result exactly. A node whose out-edge records did not change in pass p-1
// would repeat its walk of pass p-1 unchanged, so pass p only re-walks the nodes marked dirty then.
//
// A walk is a chain over the in-edges, and only the subtractions and the sign checks depend on the previous
// edge: the lanes load and step the travelers of 64 / G in-edges at a time (all lanes busy, one gather latency
// per 64 / G edges), then every group of lanes runs the chain over them from LDS (buf, 64 x 10 doubles per
// wavefront). With one group of lanes per node and an edge at a time, a pass over nodes of 50 in- and 50
// out-edges took 120 us and more.
//
// Returns (in every lane) WALK_CHANGED if some record changed, WALK_FULL if the record pool is full and
// WALK_CONFIRMED if the node ends with confirmed cases: a fix-up moves a shortfall to the group's largest
// remaining compartment, which is INSC where all others are negative.
constexpr int WALK_CHANGED   = 1;
constexpr int WALK_FULL      = 2;
constexpr int WALK_CONFIRMED = 4;

__device__ __forceinline__ bool confirmed_cases(const double (&y)[NC])
{
    return y[INSC] != 0.0 || y[ISYC] != 0.0;
}

template <int G>
__device__ __forceinline__ int walk_node(Seg& c, InstDev& I, int node, int pass, double* buf)
{
    constexpr int NPW = WAVE / G;
    const int lane    = int(threadIdx.x) % WAVE;
    const int grp     = lane / G;
    const int age     = lane - grp * G;
    const bool act    = grp < NPW;
    const int32_t tag = I.fx_epoch + pass;
    // marks of pass p-1 are in plane (p-1)&1; this pass writes plane p&1
    int32_t* dirty_out      = c.fx_dirty + size_t(pass & 1) * c.num_nodes;
    Est& es = edge_struct(c, I.estruct);
    const int v             = c.nodep[node].local;
    const int in_b = es.in_ptr[v], in_e = es.in_ptr[v + 1];
    const int in_s  = in_b + es.split[v];
    const int out_b = es.out_ptr[v], out_e = es.out_ptr[v + 1];
    const size_t own      = size_t(node) * G + age;
    const size_t src_base = size_t(I.node_base) * G + age;   // lane of local node 0
    const size_t src_step = size_t(I.node_stride) * G;       // lanes between local nodes
    const size_t np       = size_t(c.num_nodes) * G;
    FxRec* recs           = c.fx_rec + 2 * I.fx_base;
    double* pool          = c.fx_pool + I.fx_pool_base;
    const int32_t lo      = I.fx_epoch;
    const double h        = I.c_step;
    const bool icu        = I.icu != 0;
    const double D_v      = c.out_d ? c.out_d[own] : 0.0;
    double rates[NFLOW], y[NC], home[NC];
    // homecomings: sums over the out-edges, in 64 / G parts
    double k0 = 0.0, k10 = 0.0, k12 = 0.0, k_min = 0.0;
    if (act) {
        for (int k = out_b + grp; k < out_e; k += NPW) {
            const EdgeEnt e   = es.out_ent[k];
            const size_t dl   = src_base + size_t(e.nbr) * src_step;
            const EdgeCoef ec = edge_coef(es, e, es.out_min, k, D_v, G, age);
            const double kd   = c.kap[dl];
            k0                = fma(coef_of(ec, S), kd, k0);
            k_min             = fmin(k_min, kd);
            if (icu) {
                const double2 r = c.kicu[dl];
                k10             = fma(coef_of(ec, ISEV), r.x, k10);
                k12             = fma(coef_of(ec, ISEV), r.y, k12);
            }
        }
    }
    auto total = [&](double x) {
        buf[lane] = x;
        wave_sync();
        double t = 0.0;
        for (int j = 0; j < NPW; ++j) {
            t += buf[j * G + age];
        }
        wave_sync();
        return t;
    };
    k0 = total(k0);
    if (icu) {
        k10 = total(k10);
        k12 = total(k12);
    }
    homecoming<G>(c, I, es, v, own, age, D_v, k0, k10, k12, home);
    if (pass > 0) {
        // out-edges whose travelers a destination changed: their record instead of the unfixed vector
        for (int kb = out_b; kb < out_e; kb += WAVE) {
            const int k      = kb + lane;
            const int32_t ps = k < out_e ? record_slot(recs + 2 * es.out_ent[k].peer, lo, tag - 1) : -1;
            for (unsigned long long left = __ballot(ps >= 0); left; left &= left - 1) {
                const int b       = __ffsll(left) - 1;
                const int slot    = __shfl(ps, b);
                const EdgeEnt e   = es.out_ent[kb + b];
                const EdgeCoef ec = edge_coef(es, e, es.out_min, kb + b, D_v, G, age);
                double m[NC];
                load_planes(c.dep, np, own, m);
                lane_rates(c, icu, src_base + size_t(e.nbr) * src_step, rates);
                edge_return(ec, rates, h, m);
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    home[i] += pool[(size_t(slot) * G + age) * NC + i] - m[i];
                }
            }
        }
    }
    lane_rates(c, icu, own, rates);
    load_planes(c.ypre, np, own, y);
    auto finish = [&]() {
        if (grp == 0) {
            double* yp = c.y + own * NC;
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                yp[i] = y[i];
            }
            if (I.c_out_day >= 0) {
                write_phase_end_day<G>(c, I, own, v, age, y);
            }
        }
    };
    if (I.general != GENERAL) {
        // A node that walks because a homecoming changed (its travelers were fixed up elsewhere) is mostly done with
        // the closed form of come_home and the new sum, if no fix-up of its own can act and none did so far.
        double m[NC], dm[NC], y1[NC];
        load_planes(c.arr, np, own, m);
        euler_change(m, rates, h, dm);
        bool full = I.fx_neg != 0 || !(rates[0] >= 0.0) || !(k_min >= 0.0);
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            y1[i]            = y[i] - (m[i] + dm[i]);
            const double low = fmin(home[i], 0.0);
            full             = full || !(y1[i] >= 0.0) || !(y1[i] + low >= 0.0) || !(y[i] + low >= 0.0);
        }
        if (I.general == STEEP) {
            full = full || falls_short(y, m, dm, rates, h, home);
        }
        if (pass > 1) {
            for (int k = in_b + lane; k < in_e; k += WAVE) {
                full = full || record_slot(recs + 2 * k, lo, tag - 1) >= 0;
            }
        }
        if (!__any(full)) {
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                y[i] = y1[i] + home[i];
            }
            finish();
            return __any(confirmed_cases(y)) ? WALK_CONFIRMED : 0;
        }
    }
    int result    = 0;
    auto in_edges = [&](int first, int last) {
        for (int kb = first; kb < last; kb += NPW) {
            const int k = kb + grp;
            int32_t ps  = -1;
            bool slow   = false; // negative travelers or a record among these edges
            if (act && k < last) {
                const EdgeEnt e   = es.in_ent[k];
                const size_t sl   = src_base + size_t(e.nbr) * src_step;
                const EdgeCoef ec = edge_coef(es, e, es.in_min, k, c.out_d ? c.out_d[sl] : 0.0, G, age);
                double m[NC];
                load_planes(c.dep, np, sl, m);
                edge_return(ec, rates, h, m);
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    buf[i * WAVE + lane] = m[i];
                    slow                 = slow || !(m[i] >= 0.0);
                }
                if (pass > 0) {
                    ps   = record_slot(recs + 2 * k, lo, tag - 1);
                    slow = slow || ps >= 0;
                }
            }
            wave_sync();
            const int n = min(NPW, last - kb);
            // all of them at once, in order: with nonnegative travelers no compartment fell below zero on the way if
            // none is below zero after them
            double z[NC];
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                z[i] = y[i];
            }
            for (int j = 0; j < n; ++j) {
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    z[i] -= buf[i * WAVE + j * G + age];
                }
            }
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                slow = slow || !(z[i] >= 0.0);
            }
            if (!__any(slow)) {
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    y[i] = z[i];
                }
                wave_sync();
                continue;
            }
            for (int j = 0; j < n; ++j) {
                double m[NC];
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    m[i] = buf[i * WAVE + j * G + age];
                }
                const bool any    = __any(act && fixup_negative(y, m));
                const int32_t psj = __shfl(ps, j * G);
                bool diff         = (psj >= 0) != any;
                if (any && !diff) {
                    bool d = false;
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        d = d || (pool[(size_t(psj) * G + age) * NC + i] != m[i]);
                    }
                    diff = __any(act && d);
                }
                if (diff) {
                    int32_t slot = -1;
                    if (any) {
                        if (lane == 0) {
                            slot = atomicAdd(&I.fx_count, 1);
                        }
                        slot = __shfl(slot, 0);
                        if (slot < FX_SLOTS) {
                            if (grp == 0) {
#pragma unroll
                                for (int i = 0; i < NC; ++i) {
                                    pool[(size_t(slot) * G + age) * NC + i] = m[i];
                                }
                            }
                        }
                        else {
                            slot = -1;
                            result |= WALK_FULL; // the sequential replay resolves this phase
                        }
                    }
                    if (lane == 0) {
                        FxRec* r        = recs + 2 * (kb + j);
                        const int older = (r[0].tag <= r[1].tag) ? 0 : 1;
                        r[older]        = FxRec{tag, slot};
                        dirty_out[seg_node(I, es.in_ent[kb + j].nbr)] = tag; // the source re-walks in the next pass
                    }
                    result |= WALK_CHANGED;
                }
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    y[i] -= m[i];
                }
            }
            wave_sync();
        }
    };
    in_edges(in_b, in_s);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        y[i] += home[i];
    }
    in_edges(in_s, in_e);
    finish();
    return result | (__any(confirmed_cases(y)) ? WALK_CONFIRMED : 0);
}

// Pass 0 of the instances whose returns walk their edges (InstDev::general): every node, one wavefront each. Row y of
// the grid has the nodes y, y + gridDim.y, ... of each wavefront's 64 / G: as many rows as fill the chip (400 nodes of
// 1 group: 160 us per half-day in 16 rows and more, 507 us in one; 102400 nodes of 3 groups, 1219 blocks: 1093 us in
// one row, 1185 us in 21).
constexpr int WALK_BLOCKS = 2048; // blocks of the walk, in whole rows

inline dim3 walk_grid(int num_blocks, int groups)
{
    return dim3(unsigned(num_blocks), unsigned(std::clamp(WALK_BLOCKS / std::max(num_blocks, 1), 1, WAVE / groups)));
}

template <int G>
__device__ __forceinline__ void walk_body(const LaunchDev& ld, InstDev* __restrict__ inst, double* buf)
{
    const int lb = xcd_block();
    if (lb >= ld.num_blocks || ld.block_seg[lb] < 0) {
        return;
    }
    const int seg   = ld.block_seg[lb];
    Seg& c = *segment(ld, seg);
    constexpr int NPW = WAVE / G;
    const int wave    = (lb - ld.block_first[seg]) * (BLOCK / WAVE) + int(threadIdx.x) / WAVE;
    for (int node = wave * NPW + int(blockIdx.y); node < min(c.num_nodes, (wave + 1) * NPW); node += int(gridDim.y)) {
        InstDev& I = inst[c.nodep[node].inst];
        if (I.c_active && I.c_action == 2 && I.general == GENERAL) {
            const int r = walk_node<G>(c, I, node, 0, buf + (threadIdx.x / WAVE) * (WAVE * NC));
            if (r != 0 && threadIdx.x % WAVE == 0) {
                // every writer of a field stores the same value
                if (r & (WALK_CHANGED | WALK_FULL)) {
                    I.fx_changed = FX_MANY;
                }
                if (r & WALK_FULL) {
                    I.fx_state = 2;
                }
                if ((r & WALK_CONFIRMED) && I.plain) {
                    I.plain = PLAIN_LOST;
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------- settling the fix-ups
// Sequential return pass of one instance in the reference's edge order with the negative-value fix-up
// (metapopulation_mobility_instant.h:568-603), for the return phases whose fix-up records did not settle within
// FX_MAX_PASSES passes or overflowed the record pool. The edges are sorted by source and the edges of one source go to
// different nodes, so their fix-ups do not depend on each other: one wavefront takes 64 / G of them at a time (an edge
// from a node to itself alone) and adds what comes home in order. Edge by edge, on G lanes, a graph of 400 nodes and
// 20k edges whose returns all replay took 12.5 ms per half-day; 2.8 ms so.
template <int G>
__device__ __forceinline__ void replay(Seg& c, InstDev& I, double* buf)
{
    constexpr int NPW = WAVE / G;
    const size_t np   = size_t(c.num_nodes) * G;
    // restore the pre-return state of every node
    for (int k = int(threadIdx.x); k < I.num_nodes * G; k += int(blockDim.x)) {
        const size_t lane = seg_node(I, k / G) * G + size_t(k % G);
        double y[NC];
        load_planes(c.ypre, np, lane, y);
        for (int i = 0; i < NC; ++i) {
            c.y[lane * NC + i] = y[i];
        }
    }
    __syncthreads();
    Est& es = edge_struct(c, I.estruct);
    if (threadIdx.x < WAVE) {
        const int lane  = int(threadIdx.x);
        const int grp   = lane / G;
        const int age   = lane - grp * G;
        const double h  = I.c_step;
        const bool icu  = I.icu != 0;
        bool confirmed  = false;
        for (int v = 0; v < I.num_nodes; ++v) {
            const int out_e   = es.out_ptr[v + 1];
            int k             = es.out_ptr[v];
            const size_t soff = seg_node(I, v) * G + age;
            const double D    = c.out_d ? c.out_d[soff] : 0.0;
            if (k == out_e) {
                continue;
            }
            double row[NC], ys[NC];
            load_planes(c.dep, np, soff, row);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                ys[i] = c.y[soff * NC + i];
            }
            while (k < out_e) {
                const int mine   = min(k + grp, out_e - 1);
                const EdgeEnt e  = es.out_ent[mine];
                const bool in    = grp < NPW && k + grp < out_e;
                const auto selfs = __ballot(in && e.nbr == v);
                const int ahead  = selfs ? (__ffsll(selfs) - 1) / G : NPW; // edges before one to the node itself
                const int n      = min(max(ahead, 1), out_e - k);
                if (in && grp < n) {
                    const size_t doff = seg_node(I, e.nbr) * G + age;
                    const EdgeCoef ec = edge_coef(es, e, es.out_min, mine, D, G, age);
                    double rates[NFLOW], m[NC], y[NC];
                    lane_rates(c, icu, doff, rates);
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        m[i] = row[i];
                        y[i] = ahead == 0 ? ys[i] : c.y[doff * NC + i];
                    }
                    edge_return(ec, rates, h, m);
                    fixup_negative(y, m);
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        buf[i * WAVE + lane] = m[i];
                    }
                    if (ahead != 0) {
#pragma unroll
                        for (int i = 0; i < NC; ++i) {
                            c.y[doff * NC + i] = y[i] - m[i];
                        }
                    }
                    confirmed = confirmed || confirmed_cases(m); // no others without a node that has some
                }
                wave_sync();
                for (int j = 0; j < n; ++j) {
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        ys[i] += buf[i * WAVE + j * G + age];
                    }
                }
                if (ahead == 0) {
#pragma unroll
                    for (int i = 0; i < NC; ++i) {
                        ys[i] -= buf[i * WAVE + age];
                    }
                }
                wave_sync(); // also before the next edges read the states written here
                k += n;
            }
            if (grp == 0) {
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    c.y[soff * NC + i] = ys[i];
                }
            }
            wave_sync();
        }
        confirmed = __any(confirmed);
        if (lane == 0) {
            I.replays += 1;
            if (confirmed && I.plain) {
                I.plain = PLAIN_LOST;
            }
        }
    }
    __syncthreads();
    if (I.c_out_day >= 0) {
        for (int k = int(threadIdx.x); k < I.num_nodes * G; k += int(blockDim.x)) {
            const int v       = k / G;
            const size_t lane = seg_node(I, v) * G + size_t(k % G);
            double y[NC];
            for (int i = 0; i < NC; ++i) {
                y[i] = c.y[lane * NC + i];
            }
            write_phase_end_day<G>(c, I, lane, v, k % G, y);
        }
    }
}

// Blocks among which the first pass is shared out: one where its wavefronts have a node each at most. (Then the block
// does without the fences and the arrivals: 100 days of a graph of 400 nodes 18.3 against 19.0 ms.)
__device__ __forceinline__ int settle_blocks(const LaunchDev& ld, const InstDev& I)
{
    return I.fx_changed <= SETTLE_BLOCK / WAVE && I.num_nodes <= SETTLE_LIST ? 1 : ld.slices;
}

// The passes of walk_node over the marked nodes until no record changes. In the first one an instance's marked nodes
// are shared out to its ld.slices blocks; the last block to arrive goes on with the further passes, which have about a
// tenth of the nodes, alone: they end at a barrier instead of a kernel boundary. Graphs too large for that have their
// first passes in launches of their own (last = false) before. Returns whether the block has the instance's last word
// (what the others did is visible to it).
template <int G>
__device__ __forceinline__ bool settle_body(const LaunchDev& ld, InstDev& I, int slice, bool last, int32_t* list,
                                            double* buf)
{
    constexpr int CAP  = SETTLE_LIST;      // marked nodes a block holds at a time
    constexpr int SCAN = 4 * SETTLE_BLOCK; // nodes looked at at a time
    static_assert(CAP >= SCAN);
    Seg& c             = *segment(ld, I.seg);
    const int wave     = int(threadIdx.x) / WAVE;
    // list[CAP]: number of marked nodes, list[CAP + 1]: results of the pass's walks, list[CAP + 2]: arrivals
    bool sequential = I.fx_sequential != 0 || I.fx_state == 2;
    int step        = settle_blocks(ld, I);
    int pass        = I.fx_pass + 1;
    int walked      = 0; // passes
    int results     = 0; // of all passes
    bool more       = false;
    for (;; ++pass) {
        __syncthreads();
        if (threadIdx.x == 0) {
            list[CAP]     = 0;
            list[CAP + 1] = 0;
        }
        __syncthreads();
        if (!sequential) {
            const int32_t* marks = c.fx_dirty + size_t((pass - 1) & 1) * c.num_nodes;
            const int32_t tag    = I.fx_epoch + pass - 1;
            const int share      = (I.num_nodes - slice + step - 1) / step; // nodes slice, slice + step, ...
            for (int first = 0; first < share; first += SCAN) {
                int32_t node[SCAN / SETTLE_BLOCK], mark[SCAN / SETTLE_BLOCK];
#pragma unroll
                for (int q = 0; q < SCAN / SETTLE_BLOCK; ++q) {
                    const int k = first + q * SETTLE_BLOCK + int(threadIdx.x);
                    node[q]     = int(seg_node(I, slice + min(k, share - 1) * step));
                    mark[q]     = k < share ? marks[node[q]] : -1;
                }
#pragma unroll
                for (int q = 0; q < SCAN / SETTLE_BLOCK; ++q) {
                    if (mark[q] == tag) {
                        list[atomicAdd(&list[CAP], 1)] = node[q];
                    }
                }
                __syncthreads();
                const int n = list[CAP];
                __syncthreads(); // everyone has read it before the next nodes are added
                if (n > CAP - SCAN || first + SCAN >= share) {
                    for (int k = wave; k < n; k += SETTLE_BLOCK / WAVE) {
                        const int r = walk_node<G>(c, I, list[k], pass, buf + wave * (WAVE * NC));
                        if (r != 0 && threadIdx.x % WAVE == 0) {
                            atomicOr(&list[CAP + 1], r);
                        }
                    }
                    __syncthreads();
                    if (threadIdx.x == 0) {
                        list[CAP] = 0;
                    }
                    __syncthreads();
                }
            }
            walked += 1;
        }
        int r = list[CAP + 1];
        if (step > 1) {
            // marks, records and record vectors of this pass are read by another block in the next one
            __threadfence();
            __syncthreads();
            if (threadIdx.x == 0) {
                const uint32_t mine = 1u | (r & WALK_CHANGED ? 1u << 8 : 0u) | (r & WALK_FULL ? 1u << 16 : 0u) |
                                      (r & WALK_CONFIRMED ? 1u << 24 : 0u);
                list[CAP + 2] = int32_t(atomicAdd(&I.fx_arrived, mine) + mine);
            }
            __syncthreads();
            const uint32_t all = uint32_t(list[CAP + 2]);
            if ((all & 255u) != uint32_t(step)) {
                return false;
            }
            __threadfence();
            r = (all >> 8 & 255u ? WALK_CHANGED : 0) | (all >> 16 & 255u ? WALK_FULL : 0) |
                (all >> 24 ? WALK_CONFIRMED : 0);
            slice = 0;
            step  = 1;
        }
        results |= r;
        more = (r & WALK_CHANGED) != 0;
        if (more) {
            sequential = sequential || (r & WALK_FULL) || pass + 1 >= FX_MAX_PASSES;
        }
        if (!more || sequential || !last) {
            break;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        I.fx_arrived = 0;
        I.fx_passes += walked + (sequential && last ? 1 : 0);
        if ((results & WALK_CONFIRMED) && I.plain) {
            I.plain = PLAIN_LOST;
        }
        if (!last) {
            I.fx_pass    = pass;
            I.fx_changed = (more || sequential) ? FX_MANY : 0;
            I.fx_state   = sequential ? 2 : 0;
        }
    }
    if (sequential && last) {
        __syncthreads();
        replay<G>(c, I, buf);
    }
    return true;
}

// ------------------------------------------------------------------------------- kernels
// One kernel per (G, integrator) for launches over segments of one G; the *_mixed kernels serve launch
// tables whose segments have different G (LaunchDev::G == 0): each block reads its segment's G and runs
// the body specialised for it (blocks never span segments).
__device__ __forceinline__ int block_groups(const LaunchDev& ld)
{
    const int lb = xcd_block();
    if (lb >= ld.num_blocks) {
        return 0;
    }
    const int seg = ld.block_seg[lb];
    return seg < 0 ? 0 : ld.segs[seg].G;
}

#define MGO_DISPATCH_G(G_EXPR, CALL)                                                                           \
    switch (G_EXPR) {                                                                                          \
    case 1: { constexpr int GG = 1; CALL; } break;                                                             \
    case 2: { constexpr int GG = 2; CALL; } break;                                                             \
    case 3: { constexpr int GG = 3; CALL; } break;                                                             \
    case 4: { constexpr int GG = 4; CALL; } break;                                                             \
    case 5: { constexpr int GG = 5; CALL; } break;                                                             \
    case 6: { constexpr int GG = 6; CALL; } break;                                                             \
    case 7: { constexpr int GG = 7; CALL; } break;                                                             \
    case 8: { constexpr int GG = 8; CALL; } break;                                                             \
    default: break;                                                                                            \
    }

// the plain kernel's registers are allocated for two wavefronts per SIMD
template <int G, int K, int M>
__global__ void __launch_bounds__(BLOCK, M == PLAIN ? 2 : 1) node_phase(LaunchDev ld, InstDev* __restrict__ inst)
{
    __shared__ double wx[node_lds<G>()];
    node_body<G, K, M>(ld, inst, wx);
}

template <int K, int M>
__global__ void __launch_bounds__(BLOCK, M == PLAIN ? 2 : 1) node_phase_mixed(LaunchDev ld, InstDev* __restrict__ inst)
{
    __shared__ double wx[node_lds<1>()]; // G = 1 has the most stage-season planes
    MGO_DISPATCH_G(block_groups(ld), (node_body<GG, K, M>(ld, inst, wx)))
}

template <int G, bool ANY_STEEP>
__global__ void __launch_bounds__(BLOCK, EDGE_WAVES) edge_phase(LaunchDev ld, InstDev* __restrict__ inst)
{
    edge_body<G, ANY_STEEP>(ld, inst);
}

template <int G>
__global__ void __launch_bounds__(BLOCK) weights_phase(LaunchDev ld, InstDev* __restrict__ inst, int inst_offset)
{
    weights_body<G>(ld, inst, inst_offset);
}

template <int G>
__global__ void __launch_bounds__(BLOCK) walk_phase(LaunchDev ld, InstDev* __restrict__ inst)
{
    __shared__ double buf[BLOCK * NC];
    walk_body<G>(ld, inst, buf);
}

// Last kernel of a cycle: settles the fix-ups and, with clock, begins the run's next cycle: by the block that settled
// them or, where there was nothing to settle, the first of the run's blocks (the others look at fx_changed alone, which
// the clock leaves zero).
__device__ __forceinline__ void next_cycle(InstDev& I, bool clock)
{
    __syncthreads(); // every thread is done with the cycle's record
    if (clock && threadIdx.x == 0) {
        clock_one(I);
    }
}

template <int G>
__global__ void __launch_bounds__(SETTLE_BLOCK) settle_phase(LaunchDev ld, InstDev* __restrict__ inst, bool last,
                                                             bool clock)
{
    __shared__ int32_t list[SETTLE_LIST + 3];
    __shared__ double buf[SETTLE_BLOCK * NC];
    InstDev& I      = inst[ld.inst_ids[int(blockIdx.x) / ld.slices]];
    const int slice = int(blockIdx.x) % ld.slices;
    if (I.fx_changed && slice < settle_blocks(ld, I) ? settle_body<G>(ld, I, slice, last, list, buf) : slice == 0) {
        next_cycle(I, last && clock);
    }
}

#if MGO_SHARD == 13
template <bool ANY_STEEP>
__global__ void __launch_bounds__(BLOCK, EDGE_WAVES) edge_phase_mixed(LaunchDev ld, InstDev* __restrict__ inst)
{
    MGO_DISPATCH_G(block_groups(ld), (edge_body<GG, ANY_STEEP>(ld, inst)))
}

__global__ void __launch_bounds__(BLOCK) walk_phase_mixed(LaunchDev ld, InstDev* __restrict__ inst)
{
    __shared__ double buf[BLOCK * NC];
    MGO_DISPATCH_G(block_groups(ld), (walk_body<GG>(ld, inst, buf)))
}

__global__ void __launch_bounds__(SETTLE_BLOCK) settle_phase_mixed(LaunchDev ld, InstDev* __restrict__ inst, bool last,
                                                                   bool clock)
{
    __shared__ int32_t list[SETTLE_LIST + 3];
    __shared__ double buf[SETTLE_BLOCK * NC];
    InstDev& I      = inst[ld.inst_ids[int(blockIdx.x) / ld.slices]];
    const int slice = int(blockIdx.x) % ld.slices;
    bool done       = slice == 0;
    if (I.fx_changed && slice < settle_blocks(ld, I)) {
        MGO_DISPATCH_G(ld.segs[I.seg].G, (done = settle_body<GG>(ld, I, slice, last, list, buf)))
    }
    if (done) {
        next_cycle(I, last && clock);
    }
}
#endif

// ------------------------------------------------------------------------------- launchers

template <int G>
hipError_t launch_node_g(const LaunchDev& c, InstDev* inst, hipStream_t s)
{
    const int nb = c.num_blocks;
#define MGO_NODE_LAUNCH(KIND)                                                                                  \
    if (c.mode == PLAIN) {                                                                                     \
        hipLaunchKernelGGL((node_phase<G, KIND, PLAIN>), dim3(nb), dim3(BLOCK), 0, s, c, inst);                \
    }                                                                                                          \
    else if (c.mode == FEATURES) {                                                                             \
        hipLaunchKernelGGL((node_phase<G, KIND, FEATURES>), dim3(nb), dim3(BLOCK), 0, s, c, inst);             \
    }                                                                                                          \
    else {                                                                                                     \
        hipLaunchKernelGGL((node_phase<G, KIND, NPIS>), dim3(nb), dim3(BLOCK), 0, s, c, inst);                 \
    }
    switch (c.kind) {
    case MGO_INTEGRATOR_CASH_KARP54:
        MGO_NODE_LAUNCH(MGO_INTEGRATOR_CASH_KARP54)
        break;
    case MGO_INTEGRATOR_RKF45:
        MGO_NODE_LAUNCH(MGO_INTEGRATOR_RKF45)
        break;
    case MGO_INTEGRATOR_CASH_KARP54_FIXED:
        MGO_NODE_LAUNCH(MGO_INTEGRATOR_CASH_KARP54_FIXED)
        break;
    default:
        MGO_NODE_LAUNCH(MGO_INTEGRATOR_EULER)
        break;
    }
#undef MGO_NODE_LAUNCH
    return hipGetLastError();
}

// Edge phase and settling of one cycle; with clock, the runs' next cycle begins.
template <int G>
hipError_t launch_edge_g(const LaunchDev& c, InstDev* inst, bool clock, hipStream_t s)
{
    if (c.edges) {
        if (c.steep) {
            hipLaunchKernelGGL((edge_phase<G, true>), dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst);
        }
        else {
            hipLaunchKernelGGL((edge_phase<G, false>), dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst);
        }
        if (c.general) {
            hipLaunchKernelGGL((walk_phase<G>), walk_grid(c.num_blocks, G), dim3(BLOCK), 0, s, c, inst);
        }
    }
    if (c.num_inst > 0 && (c.edges || clock)) {
        for (int p = c.edges ? c.wide : 0; p >= 0; --p) {
            hipLaunchKernelGGL((settle_phase<G>), dim3(c.num_inst * c.slices), dim3(SETTLE_BLOCK), 0, s, c, inst, p == 0,
                               clock);
        }
    }
    return hipGetLastError();
}

template <int G>
hipError_t launch_weights_g(const LaunchDev& c, InstDev* inst, int inst_offset, hipStream_t s)
{
    hipLaunchKernelGGL((weights_phase<G>), dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst, inst_offset);
    return hipGetLastError();
}

template <int K>
hipError_t launch_node_mixed(const LaunchDev& c, InstDev* inst, hipStream_t s)
{
    if (c.mode == PLAIN) {
        hipLaunchKernelGGL((node_phase_mixed<K, PLAIN>), dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst);
    }
    else {
        hipLaunchKernelGGL((node_phase_mixed<K, FEATURES>), dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst);
    }
    return hipGetLastError();
}


// ------------------------------------------------------------------------------- ensemble percentiles
// ensemble_percentile (analyze_result.h:316-343): the value at index floor(num_runs * p) of the sorted
// run values of each position.
//
// Up to 4096 runs: a position's values are sorted in the registers of LP lanes, K values each (K = 64; fewer with
// LP = 1 where the runs fit): every lane sorts its values with an odd-even merge network, then the lanes merge
// theirs pairwise, quads with quads and so on. All lists ascend: a merge first compares mirrored elements, then
// halves the distance; between lanes a value is fetched with a DPP move (distances within 16 lanes) or a
// permute. Comparisons within a lane are a minimum and a maximum; the more values a lane holds, the fewer of the
// costlier comparisons between lanes, and 64 doubles leave two wavefronts per SIMD (with 36 to 64 B of scratch from
// two lanes on; three spill more and are no faster). Values are read once; bound by the comparisons. 1000 runs x 33333 positions: 163 us, 512 runs x 744000
// positions: 1.20 ms (2.5 TB/s), against 1720 us and 15.3 ms for the bitonic sort in LDS below, which was bound by
// its LDS passes and barriers and remains for more than 4096 runs (two wavefronts per position).
//
// NaN sorts last. The sign of a zero is that of some zero of the position.
template <int K>
__device__ __forceinline__ void cmp_swap(double (&r)[K], int i, int j)
{
    const double a = r[i], b = r[j];
    r[i] = fmin(a, b);
    r[j] = fmax(a, b);
}

// one step of the odd-even merge sort (Batcher): lists of P, distance Q
template <int K, int P, int Q>
__device__ __forceinline__ void lane_sort_step(double (&r)[K])
{
#pragma unroll
    for (int x = Q % P; x + Q < K; ++x) {
        if ((x - Q % P) % (2 * Q) < Q && x / (2 * P) == (x + Q) / (2 * P)) {
            cmp_swap(r, x, x + Q);
        }
    }
    if constexpr (Q > 1) {
        lane_sort_step<K, P, Q / 2>(r);
    }
    else if constexpr (2 * P < K) {
        lane_sort_step<K, 2 * P, 2 * P>(r);
    }
}

// the value of lane (l ^ MASK)
template <int MASK>
__device__ __forceinline__ double lane_xor(double v)
{
    constexpr int dpp = MASK == 1 ? 0xB1 : MASK == 2 ? 0x4E : MASK == 3 ? 0x1B : MASK == 7 ? 0x141 : MASK == 8 ? 0x128
                        : MASK == 15 ? 0x140 : -1; // quad_perm, half mirror, rotation by 8, mirror
    if constexpr (dpp >= 0) {
        const int lo = __double2loint(v), hi = __double2hiint(v);
        return __hiloint2double(__builtin_amdgcn_mov_dpp(hi, dpp, 0xf, 0xf, true),
                                __builtin_amdgcn_mov_dpp(lo, dpp, 0xf, 0xf, true));
    }
    else {
        return __shfl_xor(v, MASK);
    }
}

// keeps the smaller (lower lane of the pair) or the larger value. Zeros of different sign are equal: both lanes may end
// with the same one (keeping them apart needs a second comparison: 218 instead of 164 us for 1000 runs x 33333
// positions).
__device__ __forceinline__ double keep(double a, double x, bool upper)
{
    return ((x < a) != upper) ? x : a;
}

// keeps the scheduler from overlapping more than N elements' fetches (it would spill for it)
template <int N>
__device__ __forceinline__ void sched_every(int i)
{
    if (i % N == N - 1) {
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <int K, int D>
__device__ __forceinline__ void merge_lanes(double (&r)[K], int l)
{
    if constexpr (D >= 1) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
            r[i] = keep(r[i], lane_xor<D>(r[i]), (l & D) != 0);
            asm volatile("" : "+v"(r[i])); // one value after the other: overlapped, they need a second copy of r
        }
        merge_lanes<K, D / 2>(r, l);
    }
}

template <int K, int D>
__device__ __forceinline__ void merge_lane(double (&r)[K])
{
#pragma unroll
    for (int i = 0; i < K; ++i) {
        if (!(i & D)) {
            cmp_swap(r, i, i + D);
        }
    }
    if constexpr (D > 1) {
        merge_lane<K, D / 2>(r);
    }
}

// merges the sorted lists of N / 2 lanes each into lists of N lanes, up to LP
template <int K, int LP, int N>
__device__ __forceinline__ void merge_levels(double (&r)[K], int l)
{
    if constexpr (N <= LP) {
        const bool upper = (l & (N / 2)) != 0;
#pragma unroll
        for (int i = 0; i < K / 2; ++i) {
            const double a = r[i], b = r[K - 1 - i];
            const double xb = lane_xor<N - 1>(b), xa = lane_xor<N - 1>(a);
            r[i]         = keep(a, xb, upper);
            r[K - 1 - i] = keep(b, xa, upper);
            sched_every<4>(i);
        }
        merge_lanes<K, N / 4>(r, l);
        merge_lane<K, K / 2>(r);
        merge_levels<K, LP, 2 * N>(r, l);
    }
}

// r[i] for a wavefront-uniform i in [LO, HI)
template <int K, int LO, int HI>
__device__ __forceinline__ double pick(const double (&r)[K], int i)
{
    if constexpr (HI - LO == 1) {
        double v = r[LO];
        asm volatile("" : "+v"(v)); // keeps the leaves apart: merged, they index the values in scratch memory
        return v;
    }
    else {
        constexpr int MID = (LO + HI) / 2;
        return i < MID ? pick<K, LO, MID>(r, i) : pick<K, MID, HI>(r, i);
    }
}

template <int K, int LP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) ensemble_sort_kernel(const double* __restrict__ out,
                                                            const int64_t* __restrict__ base, int runs,
                                                            int64_t positions, const int32_t* __restrict__ ranks,
                                                            int num_ranks, double* __restrict__ sel)
{
    constexpr int PW = WAVE / LP; // positions per wavefront
    // consecutive positions stay on one XCD: neighbouring blocks share cache lines
    const int64_t blk  = int64_t(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8; // the grid is a multiple of 8
    const int lane     = int(threadIdx.x) % WAVE;
    const int l        = lane % LP; // lane within the position's group
    const int64_t p    = (blk * 4 + int(threadIdx.x) / WAVE) * PW + lane / LP;
    const bool in      = p < positions;
    const double* src  = out + (in ? p : positions - 1);
    double r[K];
    int nans = 0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        // every load is in bounds and unconditional, so that many are in flight
        const int run  = i * LP + l;
        const double v = src[base[min(run, runs - 1)]];
        const bool nan = v != v;
        r[i]           = (nan || run >= runs) ? INFINITY : v;
        nans += (nan && run < runs) ? 1 : 0;
        sched_every<16>(i);
    }
#pragma unroll
    for (int d = 1; d < LP; d <<= 1) {
        nans += __shfl_xor(nans, d);
    }
    lane_sort_step<K, 1, 1>(r);
    merge_levels<K, LP, 2>(r, l);
    for (int q = 0; q < num_ranks; ++q) {
        const int rank = __builtin_amdgcn_readfirstlane(ranks[q]);
        const double v = pick<K, 0, K>(r, rank % K);
        if (in && l == rank / K) {
            sel[int64_t(q) * positions + p] = rank < runs - nans ? v : NAN;
        }
    }
}

template <int K, int LP>
hipError_t launch_sort(const double* out, const int64_t* base, int runs, int64_t positions, const int32_t* ranks,
                       int num_ranks, double* sel, hipStream_t s)
{
    constexpr int64_t per_block = 4 * (WAVE / LP);
    const int64_t nb            = ((positions + per_block - 1) / per_block + 7) / 8 * 8;
    hipLaunchKernelGGL((ensemble_sort_kernel<K, LP>), dim3(unsigned(nb)), dim3(256), 0, s, out, base, runs, positions,
                       ranks, num_ranks, sel);
    return hipGetLastError();
}

// runs <= MAX_SORT_RUNS: the smallest K x LP that holds them (fewer, longer lists are the cheaper ones)
hipError_t launch_ensemble_sort(const double* out, const int64_t* base, int runs, int64_t positions,
                                const int32_t* ranks, int num_ranks, double* sel, hipStream_t s);

#if MGO_SHARD == 14
hipError_t launch_ensemble_sort(const double* out, const int64_t* base, int runs, int64_t positions,
                                const int32_t* ranks, int num_ranks, double* sel, hipStream_t s)
{
#define MGO_SORT(K, LP)                                                                                        \
    if (runs <= K * LP) {                                                                                      \
        return launch_sort<K, LP>(out, base, runs, positions, ranks, num_ranks, sel, s);                       \
    }
    MGO_SORT(8, 1)
    MGO_SORT(16, 1)
    MGO_SORT(32, 1)
    MGO_SORT(64, 1)
    MGO_SORT(64, 2)
    MGO_SORT(64, 4)
    MGO_SORT(64, 8)
    MGO_SORT(64, 16)
    MGO_SORT(64, 32)
    MGO_SORT(64, 64)
#undef MGO_SORT
    return hipErrorInvalidValue;
}
#endif

hipError_t launch_edge_mixed(const LaunchDev& c, InstDev* inst, bool clock, hipStream_t s);

#if MGO_SHARD >= 1 && MGO_SHARD <= 8
template hipError_t launch_node_g<MGO_SHARD>(const LaunchDev&, InstDev*, hipStream_t);
template hipError_t launch_edge_g<MGO_SHARD>(const LaunchDev&, InstDev*, bool, hipStream_t);
template hipError_t launch_weights_g<MGO_SHARD>(const LaunchDev&, InstDev*, int, hipStream_t);
#elif MGO_SHARD >= 9 && MGO_SHARD <= 12
template hipError_t launch_node_mixed<MGO_SHARD - 9>(const LaunchDev&, InstDev*, hipStream_t);
#elif MGO_SHARD == 13
hipError_t launch_edge_mixed(const LaunchDev& c, InstDev* inst, bool clock, hipStream_t s)
{
    if (c.edges) {
        if (c.steep) {
            hipLaunchKernelGGL(edge_phase_mixed<true>, dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst);
        }
        else {
            hipLaunchKernelGGL(edge_phase_mixed<false>, dim3(c.num_blocks), dim3(BLOCK), 0, s, c, inst);
        }
        if (c.general) {
            hipLaunchKernelGGL(walk_phase_mixed, walk_grid(c.num_blocks, 1), dim3(BLOCK), 0, s, c, inst);
        }
    }
    if (c.num_inst > 0 && (c.edges || clock)) {
        for (int p = c.edges ? c.wide : 0; p >= 0; --p) {
            hipLaunchKernelGGL(settle_phase_mixed, dim3(c.num_inst * c.slices), dim3(SETTLE_BLOCK), 0, s, c, inst, p == 0,
                               clock);
        }
    }
    return hipGetLastError();
}

#elif MGO_SHARD == 0
#define MGO_EXTERN_G(GG)                                                                                       \
    extern template hipError_t launch_node_g<GG>(const LaunchDev&, InstDev*, hipStream_t);                     \
    extern template hipError_t launch_edge_g<GG>(const LaunchDev&, InstDev*, bool, hipStream_t);               \
    extern template hipError_t launch_weights_g<GG>(const LaunchDev&, InstDev*, int, hipStream_t);
MGO_EXTERN_G(1)
MGO_EXTERN_G(2)
MGO_EXTERN_G(3)
MGO_EXTERN_G(4)
MGO_EXTERN_G(5)
MGO_EXTERN_G(6)
MGO_EXTERN_G(7)
MGO_EXTERN_G(8)
#undef MGO_EXTERN_G
extern template hipError_t launch_node_mixed<MGO_INTEGRATOR_CASH_KARP54>(const LaunchDev&, InstDev*, hipStream_t);
extern template hipError_t launch_node_mixed<MGO_INTEGRATOR_RKF45>(const LaunchDev&, InstDev*, hipStream_t);
extern template hipError_t launch_node_mixed<MGO_INTEGRATOR_CASH_KARP54_FIXED>(const LaunchDev&, InstDev*, hipStream_t);
extern template hipError_t launch_node_mixed<MGO_INTEGRATOR_EULER>(const LaunchDev&, InstDev*, hipStream_t);

hipError_t launch_clock(InstDev* inst, int n, hipStream_t s)
{
    hipLaunchKernelGGL(clock_kernel, dim3(unsigned(n + 255) / 256), dim3(256), 0, s, inst, n);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------- instance slots
// Serving keeps every resident request's instance record in one table of slots. Admission and retirement
// write whole records (table[ids[k]] = src[k]), class rebuilds renumber the segments (table[ids[k]].seg = k);
// one launch each per loop iteration instead of one copy per request.
static __global__ void scatter_slots_kernel(InstDev* __restrict__ table, const InstDev* __restrict__ src,
                                     const int32_t* __restrict__ ids, int n)
{
    constexpr int W = int(sizeof(InstDev) / 8);
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= int64_t(n) * W) {
        return;
    }
    const int k = int(i / W), w = int(i % W);
    reinterpret_cast<uint64_t*>(table + ids[k])[w] = reinterpret_cast<const uint64_t*>(src + k)[w];
}

static __global__ void set_segments_kernel(InstDev* __restrict__ table, const int32_t* __restrict__ ids, int n)
{
    const int k = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (k < n) {
        table[ids[k]].seg = k;
    }
}

hipError_t launch_scatter_slots(InstDev* table, const InstDev* src, const int32_t* ids, int n, hipStream_t s)
{
    if (n <= 0) {
        return hipSuccess;
    }
    const int64_t words = int64_t(n) * int64_t(sizeof(InstDev) / 8);
    hipLaunchKernelGGL(scatter_slots_kernel, dim3(unsigned((words + 255) / 256)), dim3(256), 0, s, table, src, ids, n);
    return hipGetLastError();
}

hipError_t launch_set_segments(InstDev* table, const int32_t* ids, int n, hipStream_t s)
{
    if (n <= 0) {
        return hipSuccess;
    }
    hipLaunchKernelGGL(set_segments_kernel, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, table, ids, n);
    return hipGetLastError();
}

hipError_t launch_node(const LaunchDev& c, InstDev* inst, hipStream_t s)
{
    switch (c.G) {
    case 0:
        switch (c.kind) {
        case MGO_INTEGRATOR_CASH_KARP54:
            return launch_node_mixed<MGO_INTEGRATOR_CASH_KARP54>(c, inst, s);
        case MGO_INTEGRATOR_RKF45:
            return launch_node_mixed<MGO_INTEGRATOR_RKF45>(c, inst, s);
        case MGO_INTEGRATOR_CASH_KARP54_FIXED:
            return launch_node_mixed<MGO_INTEGRATOR_CASH_KARP54_FIXED>(c, inst, s);
        default:
            return launch_node_mixed<MGO_INTEGRATOR_EULER>(c, inst, s);
        }
    case 1:
        return launch_node_g<1>(c, inst, s);
    case 2:
        return launch_node_g<2>(c, inst, s);
    case 3:
        return launch_node_g<3>(c, inst, s);
    case 4:
        return launch_node_g<4>(c, inst, s);
    case 5:
        return launch_node_g<5>(c, inst, s);
    case 6:
        return launch_node_g<6>(c, inst, s);
    case 7:
        return launch_node_g<7>(c, inst, s);
    case 8:
        return launch_node_g<8>(c, inst, s);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_edge(const LaunchDev& c, InstDev* inst, bool clock, hipStream_t s)
{
    switch (c.G) {
    case 0:
        return launch_edge_mixed(c, inst, clock, s);
    case 1:
        return launch_edge_g<1>(c, inst, clock, s);
    case 2:
        return launch_edge_g<2>(c, inst, clock, s);
    case 3:
        return launch_edge_g<3>(c, inst, clock, s);
    case 4:
        return launch_edge_g<4>(c, inst, clock, s);
    case 5:
        return launch_edge_g<5>(c, inst, clock, s);
    case 6:
        return launch_edge_g<6>(c, inst, clock, s);
    case 7:
        return launch_edge_g<7>(c, inst, clock, s);
    case 8:
        return launch_edge_g<8>(c, inst, clock, s);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_weights(const LaunchDev& c, InstDev* inst, int inst_offset, hipStream_t s)
{
    switch (c.G) {
    case 1:
        return launch_weights_g<1>(c, inst, inst_offset, s);
    case 2:
        return launch_weights_g<2>(c, inst, inst_offset, s);
    case 3:
        return launch_weights_g<3>(c, inst, inst_offset, s);
    case 4:
        return launch_weights_g<4>(c, inst, inst_offset, s);
    case 5:
        return launch_weights_g<5>(c, inst, inst_offset, s);
    case 6:
        return launch_weights_g<6>(c, inst, inst_offset, s);
    case 7:
        return launch_weights_g<7>(c, inst, inst_offset, s);
    case 8:
        return launch_weights_g<8>(c, inst, inst_offset, s);
    default:
        return hipErrorInvalidValue;
    }
}

// ------------------------------------------------------------------------------- ensemble analysis
// Post-processing of the daily outputs of several runs of the same shape (cpp/memilio/data/
// analyze_result.h:267-343). A "position" is one (day, node, compartment) value of a run's output; run r's
// output starts at base[r] (doubles). Every kernel reproduces the reference's arithmetic order.

// ensemble_mean (analyze_result.h:289-315): mean = sum over runs, in run order, of value / num_runs
__global__ void ensemble_mean_kernel(const double* __restrict__ out, const int64_t* __restrict__ base, int runs,
                                     int64_t positions, double* __restrict__ mean)
{
    const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= positions) {
        return;
    }
    const double n = double(runs);
    double acc     = 0.0;
    for (int r = 0; r < runs; ++r) {
        acc += out[base[r] + p] / n;
    }
    mean[p] = acc;
}

// sum_nodes (analyze_result.h:267-287): per run and day, the node values summed in node order
__global__ void sum_nodes_kernel(const double* __restrict__ out, const int64_t* __restrict__ base, int runs,
                                 int days, int nodes, int width, double* __restrict__ sums)
{
    const int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; // (run, day, element)
    if (q >= int64_t(runs) * days * width) {
        return;
    }
    const int e   = int(q % width);
    const int64_t rd = q / width;
    const int d   = int(rd % days);
    const int r   = int(rd / days);
    const double* src = out + base[r] + (int64_t(d) * nodes) * width + e;
    double acc        = 0.0;
    for (int v = 0; v < nodes; ++v) {
        acc += src[int64_t(v) * width];
    }
    sums[q] = acc;
}

// The same for any number of runs: a block sorts the values of `ppb` consecutive positions in LDS (bitonic
// sort over a power-of-two length padded with +inf) and writes the requested order statistics.
__global__ void __launch_bounds__(256) ensemble_select_kernel(const double* __restrict__ out,
                                                               const int64_t* __restrict__ base, int runs, int npad,
                                                               int ppb, int64_t positions,
                                                               const int32_t* __restrict__ ranks, int num_ranks,
                                                               double* __restrict__ sel)
{
    extern __shared__ double lds[];
    const int64_t p0 = int64_t(blockIdx.x) * ppb;
    const int total  = ppb * npad;
    for (int i = int(threadIdx.x); i < total; i += int(blockDim.x)) {
        const int j      = i % ppb; // position within the block (fastest: adjacent addresses)
        const int r      = i / ppb;
        const int64_t p  = p0 + j;
        double v         = INFINITY;
        if (r < runs && p < positions) {
            v = out[base[r] + p];
        }
        lds[j * npad + r] = v;
    }
    __syncthreads();
    const int half = total / 2;
    for (int k = 2; k <= npad; k <<= 1) {
        for (int s = k >> 1; s > 0; s >>= 1) {
            for (int i = int(threadIdx.x); i < half; i += int(blockDim.x)) {
                const int j   = i / (npad / 2);            // segment
                const int t   = i % (npad / 2);            // pair index within the segment
                const int lo  = 2 * s * (t / s) + (t % s); // first element of the pair
                const int hi  = lo + s;
                const bool up = ((lo & k) == 0);
                double* seg   = lds + j * npad;
                const double a = seg[lo], b = seg[hi];
                if ((a > b) == up) {
                    seg[lo] = b;
                    seg[hi] = a;
                }
            }
            __syncthreads();
        }
    }
    for (int i = int(threadIdx.x); i < ppb * num_ranks; i += int(blockDim.x)) {
        const int j     = i % ppb;
        const int q     = i / ppb;
        const int64_t p = p0 + j;
        if (p < positions) {
            sel[int64_t(q) * positions + p] = lds[j * npad + ranks[q]];
        }
    }
}

hipError_t launch_ensemble_mean(const double* out, const int64_t* base, int runs, int64_t positions, double* mean,
                                hipStream_t s)
{
    const int64_t nb = (positions + 255) / 256;
    hipLaunchKernelGGL(ensemble_mean_kernel, dim3(unsigned(nb)), dim3(256), 0, s, out, base, runs, positions, mean);
    return hipGetLastError();
}

hipError_t launch_sum_nodes(const double* out, const int64_t* base, int runs, int days, int nodes, int width,
                            double* sums, hipStream_t s)
{
    const int64_t n  = int64_t(runs) * days * width;
    const int64_t nb = (n + 255) / 256;
    hipLaunchKernelGGL(sum_nodes_kernel, dim3(unsigned(nb)), dim3(256), 0, s, out, base, runs, days, nodes, width,
                       sums);
    return hipGetLastError();
}

hipError_t launch_ensemble_select(const double* out, const int64_t* base, int runs, int64_t positions,
                                  const int32_t* ranks, int num_ranks, double* sel, hipStream_t s)
{
    if (runs <= MAX_SORT_RUNS) {
        return launch_ensemble_sort(out, base, runs, positions, ranks, num_ranks, sel, s);
    }
    int npad = 2;
    while (npad < runs) {
        npad <<= 1;
    }
    const int ppb = std::max(1, 8192 / npad); // 64 KiB of LDS per block
    const size_t lds = size_t(ppb) * npad * sizeof(double);
    const int64_t nb = (positions + ppb - 1) / ppb;
    hipLaunchKernelGGL(ensemble_select_kernel, dim3(unsigned(nb)), dim3(256), lds, s, out, base, runs, npad, ppb,
                       positions, ranks, num_ranks, sel);
    return hipGetLastError();
}

#endif // MGO_SHARD

} // namespace mgo
