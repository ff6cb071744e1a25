// Compact (polynomial) symmetry functions, types 20-25: SymGrpCompRad
// (SymGrpCompRad.cpp:128-214), SymGrpCompAngn (SymGrpCompAngn.cpp:148-388),
// SymGrpCompAngw and the weighted SymGrpComp*Weighted groups.
//
// These run as their own FP64 pass beside the exponential families: the SF
// pass writes the compact groups' G after the main SF kernel, the force pass
// adds the compact groups' per-slot contributions dE/dG . dG/dr to cslot
// (and their negative sum to cself) after the main backward kernel, before
// the gather, and the training pass forms their part of the force-loss
// tangent.  One kernel, three modes (CompMode).
//
// Each member s of a group has an open radial interval (rl, rc) and, for the
// angular types, an open angle interval (al, ar); its radial function is
// the compact function cr(r) = core(|r - center| / width) (asymmetric cores:
// core((2 - y) y), CoreFunction.h:178-191) and its angular function
// ca(theta) alike with theta = acos(cos theta_ijk).
//
// What is shared.  The members of a group come in runs of one radial
// function (CompRun) and use few distinct angle functions (CompAng), so
//   * cr of every staged neighbour is tabulated once per run (LDS), instead
//     of twice per member and pair;
//   * a pair evaluates each distinct angle function once (a lane's column of
//     LDS);
//   * a run forms its radial products once; a member costs one or two reads
//     and multiply-adds.
// Neighbours are staged partitioned by element and only the pairs of the
// group's blocks are walked, passing ones compacted through an LDS queue as
// in the exponential kernels.  Four waves share an atom (pairs dealt in
// batches of 64, member sums and slot sums combined in wave order), because
// a structure of a thousand atoms otherwise leaves one wave per SIMD.
// The form before walked every pair of the list for each group with one
// wave, a lane idle unless its pair was of the group's elements, and
// evaluated every member's three functions per pair: value 4.27 and force
// 5.62 ms on 1,000 B/C/N atoms (three elements, 6 groups of 18 members
// each), now 0.267 and 0.255 ms.
//
// The reference's reuse of cr(r_jk) (calculateComp, SymGrpCompAngn.cpp:
// 98-112): a narrow member whose (rl, rc) equal the previous member's takes
// the previous member's cr(r_jk) unless that member was skipped for this
// pair.  Within a run that is the run's own function.  Only where a run's
// (rl, rc) equal the previous run's with another core (CompRun::carry) is the
// value another one; those runs follow the members one by one.
#include "device_common.h"
#include "kernel_args.h"
#include "kernels.h"

#include <algorithm>

namespace hdnnp {

namespace {

enum CompMode
{
    CM_VALUE = 0,     // G
    CM_FORCE = 1,     // cslot += dE/dG . dG/dr, cself -= their sum
    CM_TANGENT = 2    // u = cF sum_i d_i . dG/dr_i, d = F - Fref
};

// Member sums held in registers (24 doubles: with 32 the compiler runs out of
// registers for two waves per SIMD).
constexpr int kCompChunk = 24;

template <int V> struct IntC { static constexpr int value = V; };

struct CompArgs
{
    ModelTables T;
    int n;
    const int* off;
    const int* cnt;
    const double4* geo;
    const int* nbrJ;
    const int* elem;
    int ldG;
    int cap;              // LDS neighbour capacity
    int wcap;             // radial functions tabulated at once
    int acap;             // angle functions tabulated per pair
    double* G;            // CM_VALUE
    int raw;
    const double* dEdG;   // CM_FORCE
    double* cslot;
    double* cself;
    const double* F;      // CM_TANGENT
    const double* Fref;
    double* U;
    double cF;
};

// The polynomial cores p1-p4 (CoreFunction.h:214-318) as
//   f = 1 + y^(k+1) (c0 + c1 y + ...),  f' = y^k (d0 + d1 y + ...),
// read with wave-uniform loads instead of a branch per core whose constants
// would all be kept in registers through the pair loop.
struct CorePoly
{
    double c[5], d[5];
};

__constant__ CorePoly kCore[4] = {
    {{-3.0, 2.0, 0.0, 0.0, 0.0}, {-6.0, 6.0, 0.0, 0.0, 0.0}},
    {{-10.0, 15.0, -6.0, 0.0, 0.0}, {-30.0, 60.0, -30.0, 0.0, 0.0}},
    {{-35.0, 84.0, -70.0, 20.0, 0.0}, {-140.0, 420.0, -420.0, 140.0, 0.0}},
    {{-126.0, 420.0, -540.0, 315.0, -70.0},
     {-630.0, 2520.0, -3780.0, 2520.0, -630.0}}};

// The exponential core, f = e^(1 - 1/(1 - y^2)).  Its own function: inlined,
// the constants of exp would be kept in registers beside the polynomials'.
__device__ __noinline__ double2 core_exp(double y)
{
    double const e = 2.718281828459045090795598298427648842334747314453125;
    double const t = 1.0 / (y * y - 1.0);
    double const ex = exp(t);
    return make_double2(e * ex, -2.0 * e * y * t * t * ex);
}

__device__ __forceinline__ void core_fdf(int core, double y, double& f,
                                         double& df)
{
    if (core == CT_EXP)
    {
        double2 const v = core_exp(y);
        f = v.x;
        df = v.y;
        return;
    }
    int const k = core - CT_POLY1 + 1;
    CorePoly const& p = kCore[k - 1];
    double const y2 = y * y;
    double yk = k <= 2 ? y : y2;
    if (k == 2) yk = y2;
    else if (k == 3) yk = y2 * y;
    else if (k == 4) yk = y2 * y2;
    double c = p.c[4], d = p.d[4];
#pragma unroll
    for (int q = 3; q >= 0; --q)
    {
        c = fma(c, y, p.c[q]);
        d = fma(d, y, p.d[q]);
    }
    f = fma(yk * y, c, 1.0);
    df = yk * d;
}

// CompactFunction::fdf (CompactFunction.h:153-160) for x inside the open
// interval: a = (x - center) scale, f = core(|a|), f' = core'(|a|)
// copysign(scale, a).
__device__ __forceinline__ void compact_fdf(int core, int asym, double center,
                                            double scale, double x, double& f,
                                            double& df)
{
    double const a = (x - center) * scale;
    double const y = fabs(a);
    core_fdf(core, asym ? (2.0 - y) * y : y, f, df);
    if (asym) df *= 2.0 - 2.0 * y;
    df *= copysign(scale, a);
}

// A run's radial function and an angle function, zero outside their open
// intervals.
__device__ __forceinline__ void run_fdf(CompRun const& u, double r, double& f,
                                        double& df)
{
    f = df = 0.0;
    if (r > u.rl && r < u.rc)
        compact_fdf(u.core, u.asym, u.rcenter, u.rscale, r, f, df);
}

__device__ __forceinline__ void ang_fdf(CompAng const& g, double th, double& f,
                                        double& df)
{
    f = df = 0.0;
    if (th > g.al && th < g.ar)
        compact_fdf(g.core, 0, g.acenter, g.ascale, th, f, df);
}

// Whether the reference skips a member of run u with angle function g for
// this pair (SymGrpCompAngn.cpp:246-262).
__device__ __forceinline__ bool member_skipped(CompRun const& u,
                                               CompAng const& g, double radij,
                                               double rik, double rjk,
                                               double th)
{
    return radij == 0.0 || rik <= u.rl || rik >= u.rc || rjk <= u.rl
        || rjk >= u.rc || th <= g.al || th >= g.ar;
}

// cr(r_jk) and its derivative that the first member of carry run r finds,
// and whether the member before it was skipped (then it takes its own).
// Follows the chain of runs of equal (rl, rc) member by member.
__device__ __forceinline__ bool carried_radjk(CompRun const* run, int r,
                                           CompMember const* mem,
                                           CompAng const* ang, double rij,
                                           double rik, double rjk, double th,
                                           double& f, double& df)
{
    int s = r;
    while (run[s].carry) --s;
    bool skipped = true;
    f = df = 0.0;
    for (int q = s; q < r; ++q)
    {
        CompRun const u = run[q];
        double own, down, radij, d;
        run_fdf(u, rjk, own, down);
        run_fdf(u, rij, radij, d);
        for (int m = u.m0; m < u.mend; ++m)
        {
            if (member_skipped(u, ang[mem[m].ang], radij, rik, rjk, th))
            {
                skipped = true;
                continue;
            }
            if (q == s || skipped)
            {
                f = own;
                df = down;
            }
            skipped = false;
        }
    }
    return skipped;
}

__device__ __forceinline__ void lds_add_d(double* p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int MODE>
__global__ __launch_bounds__(256) void k_compact(CompArgs a)
{
    constexpr bool DERIV = MODE != CM_VALUE;
    constexpr int ND = DERIV ? 2 : 1;
    extern __shared__ __align__(16) double sm[];
    __shared__ int sStart[kMaxElements], sCnt[kMaxElements];
    __shared__ double RED[4 * kCompChunk];
    ModelTables const& T = a.T;
    int const i = blockIdx.x;
    ElemDesc const& ed = T.elem[a.elem[i]];
    if (ed.ncg == 0) return;
    int const tid = threadIdx.x, nthr = blockDim.x;
    int const lane = tid & 63, w = uniform(tid >> 6), nw = nthr >> 6;
    int const cap = a.cap, wcap = a.wcap, acap = a.acap, ne = T.ne;
    // LDS: staged neighbours, 1/r; the waves' slot sums (force) or the
    // residuals (tangent); radial tables; the lanes' angle functions;
    // member weights (force); the waves' queues.
    double4* const P = (double4*)sm;
    double* const INV = (double*)(P + cap);
    double* p = INV + cap;
    int* const SLOT = (int*)p;      // place in the list (carry runs)
    p += (cap + 1) / 2;
    double* const ACC = p;
    double* const E = p;
    if (MODE == CM_FORCE) p += (size_t)nw * 3 * cap;
    if (MODE == CM_TANGENT) p += 4 * (size_t)cap;
    double* const RAD = p;
    p += (size_t)ND * wcap * cap;
    double* const ANG = p + w * (ND * acap * 64) + lane;
    p += nw * ND * acap * 64;
    double* const W = p;
    if (MODE == CM_FORCE) p += T.maxCompMembers;
    int* const Q = (int*)p + w * kQueue;
    int const s0 = a.off[i], n = a.cnt[i];
    double da[3] = {0.0, 0.0, 0.0};
    if (MODE == CM_TANGENT)
        for (int k = 0; k < 3; ++k)
            da[k] = a.F[3 * (size_t)i + k] - a.Fref[3 * (size_t)i + k];

    // Stage by element (stable): every wave counts all entries and places
    // those of its own batches.
    {
        int start[kMaxElements];
#pragma unroll
        for (int q = 0; q < kMaxElements; ++q) start[q] = 0;
        for (int base = 0; base < n; base += 64)
        {
            int const s = base + lane;
            int const e = s < n ? a.elem[a.nbrJ[s0 + s]] : -1;
#pragma unroll
            for (int q = 0; q < kMaxElements; ++q)
                if (q < ne) start[q] += __popcll(__ballot(e == q));
        }
        int acc = 0;
#pragma unroll
        for (int q = 0; q < kMaxElements; ++q)
        {
            int const c = q < ne ? start[q] : 0;
            if (tid == 0)
            {
                sStart[q] = acc;
                sCnt[q] = c;
            }
            start[q] = acc;
            acc += c;
        }
        int turn = 0;
        for (int base = 0; base < n; base += 64, turn = turn + 1 == nw ? 0 : turn + 1)
        {
            int const s = base + lane;
            int j = 0, e = -1;
            if (s < n)
            {
                j = a.nbrJ[s0 + s];
                e = a.elem[j];
            }
            int pos = 0;
#pragma unroll
            for (int q = 0; q < kMaxElements; ++q)
                if (q < ne)
                {
                    uint64_t const mask = __ballot(e == q);
                    if (e == q) pos = start[q] + lanes_below(mask);
                    start[q] += __popcll(mask);
                }
            if (turn == w && s < n)
            {
                double4 const g = a.geo[s0 + s];
                P[pos] = g;
                INV[pos] = 1.0 / g.w;
                SLOT[pos] = s;
                if (MODE == CM_FORCE)
                    for (int q = 0; q < nw; ++q)
                        for (int k = 0; k < 3; ++k)
                            ACC[(size_t)(3 * q + k) * cap + pos] = 0.0;
                if (MODE == CM_TANGENT)
                {
                    double ej[3];
                    for (int k = 0; k < 3; ++k)
                    {
                        ej[k] = da[k] - (a.F[3 * (size_t)j + k]
                                         - a.Fref[3 * (size_t)j + k]);
                        E[k * cap + pos] = ej[k];
                    }
                    E[3 * cap + pos] = g.x * ej[0] + g.y * ej[1]
                                     + g.z * ej[2];
                }
            }
        }
    }
    for (int cg = ed.cg0; cg < ed.cg0 + ed.ncg; ++cg)
    {
        CompGroup const g = T.cgroup[cg];
        CompMember const* __restrict__ mem = T.cmember + g.mem0;
        bool const weighted = sf_weighted(g.type);
        __syncthreads();   // staging, or the previous group, is done
        if (MODE == CM_FORCE)
        {
            for (int l = tid; l < g.nmem; l += nthr)
                W[l] = a.dEdG[(size_t)i * a.ldG + mem[l].sf] * mem[l].sfac;
            __syncthreads();
        }
        if (sf_radial(g.type))
        {
            int const a0 = weighted ? 0 : sStart[g.e1];
            int const na = weighted ? n : sCnt[g.e1];
            if (MODE == CM_FORCE)
            {
                // SymGrpCompRad.cpp:176-200: p = drad sfac / r (times Z_j for
                // the weighted type); slot j receives -p dr_ij.
                for (int t = a0 + tid; t < a0 + na; t += nthr)
                {
                    double4 const pj = P[t];
                    if (!(pj.w < g.rmax && pj.w > 0.0)) continue;
                    double S = 0.0;
                    for (int l = 0; l < g.nmem; ++l)
                    {
                        CompMember const& m = mem[l];
                        if (pj.w <= m.rl || pj.w >= m.rc) continue;
                        double f, df;
                        compact_fdf(m.core, m.asym, m.rcenter, m.rscale, pj.w,
                                    f, df);
                        S += W[l] * df;
                    }
                    S *= INV[t];
                    if (weighted) S *= staged_weight(T, sStart, sCnt, t);
                    ACC[t] -= S * pj.x;
                    ACC[cap + t] -= S * pj.y;
                    ACC[2 * cap + t] -= S * pj.z;
                }
                continue;
            }
            // Members dealt to the waves, lanes over the neighbours.
            for (int l = w; l < g.nmem; l += nw)
            {
                CompMember const& m = mem[l];
                double S = 0.0;
                for (int t = a0 + lane; t < a0 + na; t += 64)
                {
                    double const r = P[t].w;
                    if (!(r > 0.0) || r <= m.rl || r >= m.rc) continue;
                    double f, df;
                    compact_fdf(m.core, m.asym, m.rcenter, m.rscale, r, f, df);
                    double v = MODE == CM_VALUE
                             ? f : df * m.sfac * INV[t] * E[3 * cap + t];
                    if (weighted) v *= staged_weight(T, sStart, sCnt, t);
                    S += v;
                }
                S = wave_sum(S);
                if (lane == 0)
                {
                    if (MODE == CM_VALUE)
                        a.G[(size_t)i * a.ldG + m.sf] = a.raw ? S
                            : scale_sf(T.scale[ed.sf0 + m.sf], S);
                    else a.U[(size_t)i * a.ldG + m.sf] = a.cF * S;
                }
            }
            continue;
        }
        bool const wide = g.type == 22 || g.type == 25;
        CompRun const* __restrict__ run = T.crun + g.run0;
        CompAng const* __restrict__ ang = T.cang + g.ang0;
        // Angle functions shared by the members, or (more than the columns
        // hold) one column per member of a chunk.
        bool const shared = g.nang <= acap;
        int const b1 = weighted ? 0 : sStart[g.e1];
        int const n1 = weighted ? n : sCnt[g.e1];
        int const b2 = weighted || g.e1 == g.e2 ? 0 : sStart[g.e2];
        int const n2 = weighted || g.e1 == g.e2 ? 0 : sCnt[g.e2];
        DiagPairs dp = weighted
            ? DiagPairs(true, 0, n, 0, n)
            : DiagPairs(g.e1 == g.e2, sStart[g.e1], sCnt[g.e1],
                        sStart[g.e2], sCnt[g.e2]);
        // A lane's next pair is nthr pairs on.
        dp.q64 = dp.d > 0 ? nthr / dp.d : 0;
        dp.r64 = nthr - dp.q64 * dp.d;
        // Chunks of members: as many runs as the tables hold, at most
        // kCompChunk members where sums are held per member and acap where
        // each has its own angle column.
        int most = kMaxCompMembers;
        if (MODE != CM_FORCE)   // equal parts
            most = (g.nmem + kCompChunk - 1) / kCompChunk;
        if (MODE != CM_FORCE) most = (g.nmem + most - 1) / most;
        if (!shared) most = min(most, acap);
        int r0 = 0;
        for (int m0 = 0; m0 < g.nmem;)
        {
            while (run[r0].mend <= m0) ++r0;
            int r1 = min(r0 + wcap, g.nrun);
            int const mend = min(run[r1 - 1].mend, m0 + most);
            while (run[r1 - 1].m0 >= mend) --r1;
            // Radial functions of the runs at the blocks' neighbours.
            {
                int const nb = n1 + n2;
                for (int idx = tid; idx < (r1 - r0) * nb; idx += nthr)
                {
                    int const q = idx / nb, x = idx - q * nb;
                    int const t = x < n1 ? b1 + x : b2 + x - n1;
                    double f, df;
                    run_fdf(run[r0 + q], P[t].w, f, df);
                    RAD[q * cap + t] = f;
                    if (DERIV) RAD[(size_t)(wcap + q) * cap + t] = df;
                }
            }
            __syncthreads();
            double acc[MODE == CM_FORCE ? 1 : kCompChunk];
            int code[MODE == CM_FORCE ? 1 : kCompChunk];   // angle columns
            if constexpr (MODE != CM_FORCE)
            {
#pragma unroll
                for (int m = 0; m < kCompChunk; ++m)
                {
                    acc[m] = 0.0;
                    code[m] = !shared ? m : m0 + m < mend
                            ? uniform(mem[m0 + m].ang) : 0;
                }
            }
            int const na = shared ? g.nang : mend - m0;
            auto evaluate = [&](int j, int k) {
                double4 const pj = P[j], pk = P[k];
                double const invj = INV[j], invk = INV[k];
                double const dx = pk.x - pj.x, dy = pk.y - pj.y,
                             dz = pk.z - pj.z;
                double rjk = 0.0, invjk = 0.0;
                if (!wide)
                {
                    rjk = sqrt(dx * dx + dy * dy + dz * dz);
                    if (DERIV) invjk = 1.0 / rjk;
                }
                double const rinv = invj * invk;
                double const cost = (pj.x * pk.x + pj.y * pk.y + pj.z * pk.z)
                                  * rinv;
                // Outside (-1, 1) the pair is left out
                // (SymGrpCompAngn.cpp:233): weight 0.
                bool const ok = cost > -1.0 && cost < 1.0;
                double const cs = ok ? cost : 0.5;
                double const th = acos(cs);
                double z = weighted ? staged_weight(T, sStart, sCnt, j)
                                      * staged_weight(T, sStart, sCnt, k)
                                    : 1.0;
                if (!ok) z = 0.0;
                double phij = 0.0, phik = 0.0, dac = 0.0;
                if (DERIV)
                {
                    phij = invj * (invk - invj * cs);
                    phik = invk * (invj - invk * cs);
                    dac = -1.0 / sqrt(1.0 - cs * cs);
                }
                for (int q = 0; q < na; ++q)
                {
                    double f, df;
                    ang_fdf(ang[shared ? q : mem[m0 + q].ang], th, f, df);
                    ANG[q * 64] = f;
                    if (DERIV) ANG[(acap + q) * 64] = df * dac;
                }
                double P1 = 0.0, P2 = 0.0, P3 = 0.0;    // force
                double t1 = 0.0, t2 = 0.0, t3 = 0.0;    // tangent
                if (MODE == CM_TANGENT)
                {
                    t1 = z * E[3 * cap + j];
                    t2 = z * E[3 * cap + k];
                    t3 = z * (dx * (E[j] - E[k])
                              + dy * (E[cap + j] - E[cap + k])
                              + dz * (E[2 * cap + j] - E[2 * cap + k]));
                }
                for (int r = r0; r < r1; ++r)
                {
                    CompRun const& u = run[r];
                    int const ma = max(u.m0, m0), me = min(u.mend, mend);
                    // Radial functions at j, k and (narrow) jk.
                    int const q = (r - r0) * cap;
                    double const fj = RAD[q + j], fk = RAD[q + k];
                    double dfj = 0.0, dfk = 0.0, own = 1.0, down = 0.0;
                    if (DERIV)
                    {
                        dfj = RAD[wcap * cap + q + j];
                        dfk = RAD[wcap * cap + q + k];
                    }
                    if (!wide) run_fdf(u, rjk, own, down);
                    // Radial products with cr(r_jk) = f3: the value, and the
                    // slopes along r_ij, r_ik and r_jk over their distances.
                    double R, Cj, Ck, C3;
                    auto products = [&](double f3, double df3) {
                        double const fjk = fj * fk;
                        R = fjk * f3;
                        if (DERIV)
                        {
                            Cj = invj * dfj * fk * f3;
                            Ck = invk * fj * dfk * f3;
                            C3 = -invjk * fjk * df3;
                        }
                    };
                    // Carry runs: the members' functions one by one.
                    double used = own, dused = down;
                    bool useOwn = true;
                    double f1 = fj, r2 = pk.w;
                    if (u.carry)
                    {
                        // The reference's j is the earlier of the two in the
                        // list, and only its function is tested for zero.
                        double r1 = pj.w;
                        if (SLOT[j] > SLOT[k])
                        {
                            f1 = fk;
                            r1 = pk.w;
                            r2 = pj.w;
                        }
                        useOwn = carried_radjk(run, r, mem, ang, r1, r2, rjk,
                                               th, used, dused);
                        for (int m = u.m0; m < ma; ++m)
                            useOwn = useOwn
                                || member_skipped(u, ang[mem[m].ang], f1, r2,
                                                  rjk, th);
                    }
                    if constexpr (MODE == CM_FORCE)
                    {
                        double A = 0.0, D = 0.0;
                        auto flush = [&]() {
                            double const DR = D * R;
                            P1 += DR * phij + A * Cj;
                            P2 += DR * phik + A * Ck;
                            P3 += DR * rinv + A * C3;
                        };
                        products(own, down);
                        for (int m = ma; m < me; ++m)
                        {
                            int const c = shared ? mem[m].ang : m - m0;
                            A += W[m] * ANG[c * 64];
                            D += W[m] * ANG[(acap + c) * 64];
                            if (u.carry)
                            {
                                products(useOwn ? own : used,
                                         useOwn ? down : dused);
                                flush();
                                A = D = 0.0;
                                useOwn = useOwn
                                    || member_skipped(u, ang[mem[m].ang], f1,
                                                      r2, rjk, th);
                            }
                        }
                        if (!u.carry) flush();
                    }
                    else
                    {
                        // Value: Y = R; tangent: Y and X multiply the angle
                        // function and its slope.
                        double X = 0.0, Y = 0.0, Xu = 0.0, Yu = 0.0;
                        auto set = [&](double f3, double df3, double& x,
                                       double& y) {
                            products(f3, df3);
                            if (MODE == CM_VALUE) y = z * R;
                            else
                            {
                                x = R * (phij * t1 + phik * t2 + rinv * t3);
                                y = Cj * t1 + Ck * t2 + C3 * t3;
                            }
                        };
                        uint32_t ownBits = ~0u;
                        if (u.carry)
                        {
                            ownBits = 0;
                            set(used, dused, Xu, Yu);
                            for (int m = ma; m < me; ++m)
                            {
                                ownBits |= (useOwn ? 1u : 0u) << (m - m0);
                                useOwn = useOwn
                                    || member_skipped(u, ang[mem[m].ang], f1,
                                                      r2, rjk, th);
                            }
                        }
                        set(own, down, X, Y);
#pragma unroll
                        for (int b = 0; b < kCompChunk; b += 8)
                            if (ma < m0 + b + 8 && me > m0 + b)
                            {
#pragma unroll
                                for (int m = b; m < b + 8; ++m)
                                    if (m0 + m >= ma && m0 + m < me)
                                    {
                                        double x = X, y = Y;
                                        if (u.carry && !(ownBits >> m & 1))
                                        {
                                            x = Xu;
                                            y = Yu;
                                        }
                                        acc[m] += y * ANG[code[m] * 64];
                                        if (DERIV)
                                            acc[m] += x * ANG[(acap + code[m])
                                                              * 64];
                                    }
                            }
                    }
                }
                if (MODE == CM_FORCE)
                {
                    P1 *= z;
                    P2 *= z;
                    P3 *= z;
                    double* const S = ACC + (size_t)(3 * w) * cap;
                    lds_add_d(S + j, -(P1 * pj.x + P3 * dx));
                    lds_add_d(S + cap + j, -(P1 * pj.y + P3 * dy));
                    lds_add_d(S + 2 * cap + j, -(P1 * pj.z + P3 * dz));
                    lds_add_d(S + k, P3 * dx - P2 * pk.x);
                    lds_add_d(S + cap + k, P3 * dy - P2 * pk.y);
                    lds_add_d(S + 2 * cap + k, P3 * dz - P2 * pk.z);
                }
            };
            int qn = 0, pc = 0, pr = 0;
            dp.start(tid, pc, pr);
            double const rmax2 = g.rmax * g.rmax;
            // A wave evaluates whenever 64 pairs are queued, and what is left
            // once its batches are through.
            for (int base = 0; base < dp.npairs || qn > 0; base += nthr)
            {
                if (base < dp.npairs)
                {
                    bool const valid = base + tid < dp.npairs;
                    int j, k;
                    dp.pair(pc, pr, j, k);
                    if (!valid) j = k = dp.s0;
                    dp.advance(pc, pr);
                    double4 const pj = P[j], pk = P[k];
                    double const dx = pk.x - pj.x, dy = pk.y - pj.y,
                                 dz = pk.z - pj.z;
                    double const d2 = dx * dx + dy * dy + dz * dz;
                    // Group range (rmin = 0, SymGrpBaseComp.cpp:26 with
                    // SymGrpCompRad.cpp:82-84).
                    bool const pass = valid & (pj.w < g.rmax) & (pj.w > 0.0)
                                    & (pk.w < g.rmax) & (pk.w > 0.0)
                                    & (wide | ((d2 < rmax2) & (d2 > 0.0)));
                    uint64_t const mask = __ballot(pass);
                    if (pass) Q[qn + lanes_below(mask)] = j | (k << 16);
                    qn += __popcll(mask);
                    wave_lds_fence();
                }
                if (qn >= 64 || base + nthr >= dp.npairs)
                {
                    int const q0 = max(qn - 64, 0);
                    if (q0 + lane < qn)
                    {
                        int const e = Q[q0 + lane];
                        evaluate(e & 0xffff, e >> 16);
                    }
                    qn = q0;
                    wave_lds_fence();
                }
            }
            if constexpr (MODE != CM_FORCE)
            {
                // Member totals: each wave by the transposing butterfly in
                // blocks of 16 and 4, then over the waves in order.
                auto part = [&](auto width, int first) {
                    constexpr int M = decltype(width)::value;
                    if (m0 + first >= mend) return;
                    double v[M];
#pragma unroll
                    for (int q = 0; q < M; ++q) v[q] = acc[first + q];
                    double const s = wave_sum_transposed<M>(v);
                    constexpr int sh = M == 16 ? 2 : 4;   // 6 - log2 M
                    if ((lane & ((1 << sh) - 1)) == 0)
                        RED[w * kCompChunk + first + (lane >> sh)] = s;
                };
                part(IntC<16>(), 0);
                part(IntC<4>(), 16);
                part(IntC<4>(), 20);
                __syncthreads();
                if (tid < mend - m0)
                {
                    double v = 0.0;
                    for (int q = 0; q < nw; ++q)
                        v += RED[q * kCompChunk + tid];
                    CompMember const& m = mem[m0 + tid];
                    if (MODE == CM_VALUE)
                        a.G[(size_t)i * a.ldG + m.sf] = a.raw ? v
                            : scale_sf(T.scale[ed.sf0 + m.sf], v);
                    else a.U[(size_t)i * a.ldG + m.sf] = a.cF * m.sfac * v;
                }
            }
            m0 = mend;
            if (m0 < g.nmem) __syncthreads();   // the tables are refilled
        }
    }
    if (MODE != CM_FORCE) return;
    __syncthreads();
    // Slot sums over the waves, then cself = -(their sum) by wave 0, and the
    // entries of cslot in slot order.
    for (int t = tid; t < 3 * cap; t += nthr)
    {
        if (t % cap >= n) continue;
        double v = ACC[t];
        for (int q = 1; q < nw; ++q) v += ACC[(size_t)3 * q * cap + t];
        ACC[t] = v;
    }
    __syncthreads();
    if (w == 0)
    {
        double sx = 0.0, sy = 0.0, sz = 0.0;
        for (int t = lane; t < n; t += 64)
        {
            sx += ACC[t];
            sy += ACC[cap + t];
            sz += ACC[2 * cap + t];
        }
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        sz = wave_sum(sz);
        if (lane == 0)
        {
            a.cself[3 * (size_t)i] -= sx;
            a.cself[3 * (size_t)i + 1] -= sy;
            a.cself[3 * (size_t)i + 2] -= sz;
        }
    }
    int start[kMaxElements];
#pragma unroll
    for (int q = 0; q < kMaxElements; ++q) start[q] = sStart[q];
    int turn = 0;
    for (int base = 0; base < n; base += 64, turn = turn + 1 == nw ? 0 : turn + 1)
    {
        int const s = base + lane;
        int const e = s < n ? a.elem[a.nbrJ[s0 + s]] : -1;
        int pos = 0;
#pragma unroll
        for (int q = 0; q < kMaxElements; ++q)
            if (q < ne)
            {
                uint64_t const mask = __ballot(e == q);
                if (e == q) pos = start[q] + lanes_below(mask);
                start[q] += __popcll(mask);
            }
        if (turn == w && s < n)
        {
            size_t const q = 3 * (size_t)(s0 + s);
            a.cslot[q] += ACC[pos];
            a.cslot[q + 1] += ACC[cap + pos];
            a.cslot[q + 2] += ACC[2 * cap + pos];
        }
    }
}

// Doubles of LDS without the radial tables.
template <int MODE>
size_t comp_fixed(ModelTables const& T, int cap, int nw, int acap)
{
    size_t const nd = MODE == CM_VALUE ? 1 : 2;
    size_t d = 5 * (size_t)cap + ((size_t)cap + 1) / 2
             + (size_t)nw * nd * acap * 64
             + (size_t)nw * kQueue / 2;
    if (MODE == CM_FORCE)
        d += (size_t)nw * 3 * cap + (size_t)T.maxCompMembers;
    if (MODE == CM_TANGENT) d += 4 * (size_t)cap;
    return d;
}

// Four waves per atom with all functions of the largest group tabulated if
// that fits 64 KiB of LDS (the 1,000-atom case above needs 16 to 38 KiB),
// else two or one; with one wave at most 8 angle columns, and as many radial
// functions as fit, at least one.  Only then, for the longest accepted
// lists, 64 KiB are exceeded (a workgroup may use 160 KiB).
template <int MODE>
hipError_t launch_compact(CompArgs& a, hipStream_t s)
{
    size_t const per = (size_t)(MODE == CM_VALUE ? 1 : 2) * a.cap;
    size_t const most = 65536 / sizeof(double);
    int nw = 4;
    a.acap = a.T.maxCompAngs;
    while (nw > 1 && comp_fixed<MODE>(a.T, a.cap, nw, a.acap)
                     + a.T.maxCompRuns * per > most)
        nw /= 2;
    if (nw == 1 && comp_fixed<MODE>(a.T, a.cap, nw, a.acap)
                   + a.T.maxCompRuns * per > most)
        a.acap = std::min(a.acap, 8);
    size_t const fixed = comp_fixed<MODE>(a.T, a.cap, nw, a.acap);
    size_t const fits = fixed < most ? (most - fixed) / per : 0;
    a.wcap = (int)std::max<size_t>(1, std::min<size_t>(a.T.maxCompRuns, fits));
    size_t const bytes = (fixed + a.wcap * per) * sizeof(double);
    k_compact<MODE><<<a.n, 64 * nw, bytes, s>>>(a);
    return hipGetLastError();
}

template <class A>
CompArgs comp_args(A const& b, int cap)
{
    CompArgs a{};
    a.T = b.T;
    a.n = b.n;
    a.off = b.off;
    a.cnt = b.cnt;
    a.geo = b.geo;
    a.nbrJ = b.nbrJ;
    a.elem = b.elem;
    a.ldG = b.ldG;
    a.cap = cap;
    return a;
}

}  // namespace

// The list lengths the compact pass accepts, as the LDS of one wave per atom
// with a row of member sums per lane (value, tangent) or one set of slot sums
// (force): at most 64 KiB.
size_t sf_compact_lds_bytes(ModelTables const& T, int cap)
{
    return (size_t)((64 * T.maxCompMembers + 3) & ~3) * sizeof(double)
         + (size_t)cap * (sizeof(double4) + sizeof(int));
}

size_t force_compact_lds_bytes(ModelTables const& T, int cap)
{
    return (size_t)((T.maxCompMembers + 3) & ~3) * sizeof(double)
         + (size_t)((3 * cap + 3) & ~3) * sizeof(double)
         + (size_t)cap * (sizeof(double4) + sizeof(int));
}

size_t train_u_compact_lds_bytes(ModelTables const& T, int cap)
{
    return sf_compact_lds_bytes(T, cap)
         + (size_t)cap * 3 * sizeof(double);
}

hipError_t launch_sf_compact(SFArgs const& b, hipStream_t s)
{
    if (b.n <= 0 || b.T.ncgroup == 0) return hipSuccess;
    CompArgs a = comp_args(b, b.cap);
    a.G = b.G;
    a.raw = b.raw;
    return launch_compact<CM_VALUE>(a, s);
}

hipError_t launch_force_compact(ForceArgs const& b, hipStream_t s)
{
    if (b.n <= 0 || b.T.ncgroup == 0) return hipSuccess;
    CompArgs a = comp_args(b, b.cap);
    a.dEdG = b.dEdG;
    a.cslot = b.cslot;
    a.cself = b.cself;
    return launch_compact<CM_FORCE>(a, s);
}

hipError_t launch_train_u_compact(TrainArgs const& b, int cap, hipStream_t s)
{
    if (b.n <= 0 || b.T.ncgroup == 0) return hipSuccess;
    CompArgs a = comp_args(b, cap);
    a.F = b.F;
    a.Fref = b.Fref;
    a.U = b.U;
    a.cF = b.cF;
    return launch_compact<CM_TANGENT>(a, s);
}

}  // namespace hdnnp
