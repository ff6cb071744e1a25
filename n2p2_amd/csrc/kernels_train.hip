// Training kernels (the distilled surrogate of the multiple-time-step
// integrator, and 2G models with radial and angular SFs): the gradient of
//
//   L = wE ((E - Eref) / N)^2 + wF / (3N) sum_i |F_i - Fref_i|^2
//
// with respect to every network weight, and an Adam step.
//
// With F_i = -sum_a sum_s (dE_a/dG_as)(dG_as/dr_i) the force term's
// gradient is sum_a d/dw [ sum_s u_as dE_a/dG_as ], where
//
//   u_as = -(2 wF / 3N) sum_i (F_i - Fref_i) . dG_as/dr_i,
//
// the derivative of E_a along the direction u_a: a forward-mode tangent
// through the atom's network, then reverse mode through that tangent.
// For a radial G2 member g(r) = exp(-eta (r - rs)^2) fc(r) of neighbour
// element e1 (SymGrpExpRad.cpp:144-239):
//
//   sum_i d_i . dG_as/dr_i = sfac_s sum_j g'(r_aj) (dr_aj . (d_a - d_j)) / r_aj
//
// with dr_aj = r_a - r_j and sfac_s the SF's scaling slope.  The energy
// term is ordinary backpropagation of kappa = 2 wE (E - Eref) / N^2.
// Everything is FP64 and summed in a fixed order.
//
// No counterpart in the reference's 2G prediction path; the reference
// trains with libnnptrain (Training.cpp, NeuralNetwork::calculateDEdc /
// calculateDFdc, NeuralNetwork.cpp:444-719), which this does not mirror.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "device_common.h"
#include "kernels.h"

namespace hdnnp {

namespace {

// Value, first and second derivative of the activations training supports.
__device__ __forceinline__ void activate2(int a, double x, double& v,
                                          double& d, double& dd)
{
    switch (a)
    {
    case AF_IDENTITY: v = x; d = 1.0; dd = 0.0; return;
    case AF_TANH:
    {
        double const t = tanh(x);
        v = t; d = 1.0 - t * t; dd = -2.0 * t * d;
        return;
    }
    case AF_LOGISTIC:
    case AF_SOFTPLUS:
    {
        double s1;
        activate(a, x, v, s1);
        if (x > 35.0 || x < -35.0) { d = s1; dd = 0.0; return; }
        double const s = 1.0 / (1.0 + exp(-x));
        d = s1;
        dd = a == AF_SOFTPLUS ? s * (1.0 - s) : s1 * (1.0 - 2.0 * s);
        return;
    }
    default: v = 0.0; d = 0.0; dd = 0.0; return;
    }
}

__device__ __forceinline__ double scale_slope(ScaleDesc const& s)
{
    return (s.type == ST_SCALE || s.type == ST_SCALECENTER
            || s.type == ST_SCALESIGMA) ? s.sfac : 1.0;
}

// u_as for every SF of atom a, and |F_a - Fref_a|^2.
//
// One wave per atom, organised as the SF kernel (sf_core.h): neighbours
// staged in LDS partitioned by element, unordered pairs of a group's blocks
// in diagonal order, passing pairs compacted through an LDS queue so that
// every lane evaluates one triplet.  Staged per neighbour j, besides the
// geometry and the cutoff values: e_j = d_a - d_j and t_j = dr_aj . e_j with
// the residuals d = F - Fref, so that a triplet needs three scalars
//   t_j, t_k, t_jk = dr_jk . (d_k - d_j) = (dr_ak - dr_aj) . (e_j - e_k).
// With p1, p2, p3 of SymFncExpAngn.cpp:79-225 / SymFncExpAngw.cpp:79-208 (and
// SymFncExpAngnWeighted.cpp:79-228) the members' terms contract to
//   p1 t_j + p2 t_k + p3 t_jk = fg (zeta lambda A + plambda (B - 2 eta C)),
//   A = pfc ((t_j + t_k + t_jk) / (rij rik) - cos (t_j / rij^2 + t_k / rik^2)),
//   B = f'c(rij)/rij fc(rik) fc(rjk) t_j + fc(rij) f'c(rik)/rik fc(rjk) t_k
//     - fc(rij) fc(rik) f'c(rjk)/rjk t_jk               (last term narrow only)
//   C = pfc ((rij - rs)/rij t_j + (rik - rs)/rik t_k - (rjk - rs)/rjk t_jk),
// so a member costs its power and three operations, one exponential serves an
// (eta, rs) run and one power chain a lambda run.
//
// Bound by FP64 VALU issue like the SF kernel.  The form before walked the
// pairs row by row over the whole list (every element pair tested for every
// group, idle lanes kept) and evaluated exp, pow, square roots and divisions
// per member: 4.33 ms on a 1,536-atom water box and 3.27 ms on 192 atoms,
// against 0.131 and 0.103 ms here.
template <int MAXM, int CT, bool GENPOW>
__global__ __launch_bounds__(64) void k_train_u(TrainArgs A)
{
    extern __shared__ __align__(16) double sm[];
    __shared__ int sStart[kMaxElements], sCnt[kMaxElements];
    __shared__ MParam<double> MP[kMaxMembers];
    int const cap = A.cap;
    double4* const P = (double4*)sm;        // x, y, z, r
    double4* const Q = P + cap;             // f_c, 1/r, f_c'/r, t
    double* const E = (double*)(Q + cap);   // d_a - d_j, x, y, z planes
    int* const QUEUE = (int*)(E + 3 * cap);
    int const a = blockIdx.x;
    int const lane = threadIdx.x;
    ModelTables const& T = A.T;
    int const ne = T.ne;
    ElemDesc const& ed = T.elem[A.elem[a]];
    double da[3];
    for (int k = 0; k < 3; ++k)
        da[k] = A.F[3 * (size_t)a + k] - A.Fref[3 * (size_t)a + k];
    if (lane == 0) A.d2[a] = da[0] * da[0] + da[1] * da[1] + da[2] * da[2];
    double* __restrict__ U = A.U + (size_t)a * A.ldG;
    int const s0 = A.off[a], n = A.cnt[a];
    {
        int start[kMaxElements];
#pragma unroll
        for (int q = 0; q < kMaxElements; ++q) start[q] = 0;
        for (int base = 0; base < n; base += 64)
        {
            int const s = base + lane;
            int const e = s < n ? A.elem[A.nbrJ[s0 + s]] : -1;
#pragma unroll
            for (int q = 0; q < kMaxElements; ++q)
                if (q < ne) start[q] += __popcll(__ballot(e == q));
        }
        int acc = 0;
#pragma unroll
        for (int q = 0; q < kMaxElements; ++q)
        {
            int const c = q < ne ? start[q] : 0;
            if (lane == 0)
            {
                sStart[q] = acc;
                sCnt[q] = c;
            }
            start[q] = acc;
            acc += c;
        }
        for (int base = 0; base < n; base += 64)
        {
            int const s = base + lane;
            int e = -1, j = 0;
            double4 g = make_double4(0, 0, 0, 1);
            if (s < n)
            {
                j = A.nbrJ[s0 + s];
                e = A.elem[j];
                g = A.geo[s0 + s];
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
            if (s < n)
            {
                double ej[3];
                for (int k = 0; k < 3; ++k)
                    ej[k] = da[k] - (A.F[3 * (size_t)j + k]
                                     - A.Fref[3 * (size_t)j + k]);
                P[pos] = g;
                Q[pos] = make_double4(0.0, 1.0 / g.w, 0.0,
                                      g.x * ej[0] + g.y * ej[1] + g.z * ej[2]);
                E[pos] = ej[0];
                E[cap + pos] = ej[1];
                E[2 * cap + pos] = ej[2];
            }
        }
    }
    __syncthreads();
    int keyCached = -1;
    for (int gi = ed.g0; gi < ed.g0 + ed.ng; ++gi)
    {
        GroupDesc const g = T.group[gi];
        int const cfg = ed.cfg0 + g.cfg;
        CutCfg const cc = T.cfg[cfg];
        MemberDesc const* __restrict__ mem = T.member + g.mem0;
        int const nmem = g.nmem;
        bool const weighted = sf_weighted(g.type);
        int const key = 2 * cfg + (weighted ? 1 : 0);
        if (lane < nmem) MP[lane] = make_mparam<double>(mem[lane], 0.0);
        if (key != keyCached)
        {
            // Weighted types: both values times Z_j, so radial terms carry
            // Z_j and triplet products Z_j Z_k
            // (SymGrpExpAngnWeighted.cpp:263-270).
            for (int t = lane; t < n; t += 64)
            {
                double f, df;
                cutoff_fdf_t<CT>(cc, P[t].w, f, df);
                if (weighted)
                {
                    double const z = staged_weight(T, sStart, sCnt, t);
                    f *= z;
                    df *= z;
                }
                Q[t].x = f;
                Q[t].z = df * Q[t].y;
            }
            keyCached = key;
        }
        __syncthreads();
        double acc[MAXM];
#pragma unroll
        for (int m = 0; m < MAXM; ++m) acc[m] = 0.0;
        if (sf_radial(g.type))
        {
            int const a0 = weighted ? 0 : sStart[g.e1];
            int const na = weighted ? n : sCnt[g.e1];
            for (int t = lane; t < na; t += 64)
            {
                double const r = P[a0 + t].w;
                if (!(r < g.rc)) continue;
                double4 const q = Q[a0 + t];
                double const df = q.z * q.w, f2 = 2.0 * q.x * (q.y * q.w);
#pragma unroll
                for (int m = 0; m < MAXM; ++m)
                    if (m < nmem)
                    {
                        double const eta = MP[m].eta, x = r - MP[m].rs;
                        acc[m] += (df - eta * x * f2) * exp(-eta * x * x);
                    }
            }
        }
        else
        {
            bool const wide = g.type == 9;
            DiagPairs const dp = weighted
                ? DiagPairs(true, 0, n, 0, n)
                : DiagPairs(g.e1 == g.e2, sStart[g.e1], sCnt[g.e1],
                            sStart[g.e2], sCnt[g.e2]);
            double lam[MAXM], zl[MAXM];
            int code[MAXM];
#pragma unroll
            for (int m = 0; m < MAXM; ++m)
            {
                MParam<double> const& p = MP[m < nmem ? m : 0];
                lam[m] = uniform_r(p.lambda);
                zl[m] = uniform_r(p.zl);
                code[m] = uniform(p.flags);
            }
            auto triplet = [&](int j, int k) {
                double4 const pj = P[j], pk = P[k], qj = Q[j], qk = Q[k];
                double const dx = pk.x - pj.x, dy = pk.y - pj.y,
                             dz = pk.z - pj.z;
                double const tjk = dx * (E[j] - E[k])
                                 + dy * (E[cap + j] - E[cap + k])
                                 + dz * (E[2 * cap + j] - E[2 * cap + k]);
                double const rinv = qj.y * qk.y;
                double const cost = (pj.x * pk.x + pj.y * pk.y + pj.z * pk.z)
                                  * rinv;
                double const fij_ik = qj.x * qk.x;
                double pfc = fij_ik, r2sum = pj.w * pj.w + pk.w * pk.w;
                double B = qk.x * qj.z * qj.w + qj.x * qk.z * qk.w;
                double C = qj.w + qk.w, rjk = 0.0, injk = 0.0;
                if (!wide)
                {
                    double const rjk2 = dx * dx + dy * dy + dz * dz;
                    injk = rsqrt_nr(rjk2);
                    rjk = rjk2 * injk;
                    double fcjk, dfcjk;
                    cutoff_inside<CT>(cc, rjk, fcjk, dfcjk);
                    pfc *= fcjk;
                    r2sum += rjk2;
                    B = B * fcjk - fij_ik * (dfcjk * injk) * tjk;
                    C -= tjk;
                }
                double const Av = pfc * (rinv * (qj.w + qk.w + tjk)
                                         - cost * (qj.w * (qj.y * qj.y)
                                                   + qk.w * (qk.y * qk.y)));
                double ex = 0.0, BC = 0.0, pl = 0.0;
                PowChain<double> chain;
                chain.reset(0.0);
#pragma unroll
                for (int m = 0; m < MAXM; ++m)
                    if (m < nmem)
                    {
                        int const fl = code[m];
                        if (fl & MF_NEWEXP)
                        {
                            double const eta = MP[m].eta, rs = MP[m].rs;
                            double s = r2sum, c = C;
                            if (rs != 0.0)
                            {
                                double const x = pj.w - rs, y = pk.w - rs;
                                s = x * x + y * y;
                                c = x * qj.y * qj.w + y * qk.y * qk.w;
                                if (!wide)
                                {
                                    double const w = rjk - rs;
                                    s += w * w;
                                    c -= w * injk * tjk;
                                }
                            }
                            ex = exp(-eta * s);
                            BC = B - 2.0 * eta * pfc * c;
                        }
                        if (fl & MF_NEWLAM)
                        {
                            pl = 1.0 + lam[m] * cost;
                            chain.reset(pl);
                        }
                        double pw;
                        if (fl & MF_PREFIX) pw = chain.at((fl >> 8) & 15);
                        else if (!GENPOW || (fl & MF_INTPOW))
                            pw = pow_int(pl, MP[m].zint - 1);
                        else pw = pow(pl, MP[m].zeta - 1.0);
                        acc[m] += pl > 0.0 ? ex * pw * (zl[m] * Av + pl * BC)
                                           : 0.0;
                    }
            };
            int qn = 0, pc = 0, pr = 0;
            dp.start(lane, pc, pr);
            for (int base = 0; base < dp.npairs; base += 64)
            {
                bool const valid = base + lane < dp.npairs;
                int j, k;
                dp.pair(pc, pr, j, k);
                if (!valid) j = k = dp.s0;
                dp.advance(pc, pr);
                bool const pass = valid
                    & pair_in_range<double>(P[j], P[k], wide, g.rc, g.rc2);
                uint64_t const mask = __ballot(pass);
                if (pass) QUEUE[qn + lanes_below(mask)] = j | (k << 16);
                qn += __popcll(mask);
                wave_lds_fence();
                if (qn >= 64)
                {
                    int const e = QUEUE[qn - 64 + lane];
                    triplet(e & 0xffff, e >> 16);
                    qn -= 64;
                    wave_lds_fence();
                }
            }
            if (lane < qn)
            {
                int const e = QUEUE[lane];
                triplet(e & 0xffff, e >> 16);
            }
        }
        // Member m's total ends in the lanes (m << kSh) + t.
        double const v = wave_sum_transposed<MAXM>(acc);
        constexpr int kSh = MAXM == 8 ? 3 : 2;   // 6 - log2 MAXM
        int const m = lane >> kSh;
        if ((lane & ((1 << kSh) - 1)) == 0 && m < nmem)
        {
            MemberDesc const& md = mem[m];
            U[md.sf] = A.cF * v * (sf_radial(g.type)
                                   ? scale_slope(T.scale[ed.sf0 + md.sf])
                                   : md.fnorm);
        }
        __syncthreads();
    }
}

// The static LDS of k_train_u, rounded up.
constexpr size_t kTrainStatic = 2048;
static_assert(kMaxMembers * sizeof(MParam<double>)
                  + 2 * kMaxElements * sizeof(int) <= kTrainStatic,
              "static LDS of k_train_u");

template <int MAXM>
void launch_train_u_m(TrainArgs const& A, hipStream_t s)
{
    size_t const shm = train_u_lds_bytes(A.cap) - kTrainStatic;
    if (A.T.genpow)
        HDNNP_CUTOFF_DISPATCH(A.T.cutType,
            (k_train_u<MAXM, kCT, true><<<A.n, 64, shm, s>>>(A)));
    else
        HDNNP_CUTOFF_DISPATCH(A.T.cutType,
            (k_train_u<MAXM, kCT, false><<<A.n, 64, shm, s>>>(A)));
}

// Per-block gradient of sum over the block's atoms of
// kappa E_a + (derivative of E_a along u_a), apb atoms of one element per
// block.  LDS per atom: the inputs x, tangents t of every layer and the
// adjoints of z and s of every layer, plus two adjoint scratch vectors.
//
// The threads of the block share every layer: thread t takes atom t % apb and
// every (256 / apb)-th neuron, so a wave reads one or two weight rows
// (broadcast) and the atoms' LDS records at an odd stride (no bank
// conflicts).  Each neuron's sum still runs over its inputs in order.  With
// one thread per atom, as before, the serial chain of the whole network
// bounded the kernel (200 us per element whatever the size of the
// structure); the elements now also run in one launch: 404 -> 33 us for both
// elements of a 1,536-atom water box (40-25-25-1).
constexpr int kAtoms = 32;
constexpr int kGradThreads = 256;

// One launch covers all elements (blockIdx.y).
struct TrainGradTab
{
    const int* atoms[kMaxElements];
    int na[kMaxElements], nb[kMaxElements], nw[kMaxElements];
    int stride[kMaxElements], apb[kMaxElements];
    size_t off[kMaxElements];    // the element's offset in the partials
};

__global__ __launch_bounds__(kGradThreads) void k_train_grad(
    TrainArgs A, TrainGradTab G, double* __restrict__ partAll)
{
    extern __shared__ double lds[];
    int const e = blockIdx.y, b = blockIdx.x;
    if (b >= G.nb[e]) return;
    ModelTables const& T = A.T;
    ElemDesc const& ed = T.elem[e];
    int const L = ed.nlayers - 1;
    int const t = threadIdx.x;
    int const apb = G.apb[e], perAtom = G.stride[e], nw = G.nw[e];
    int const nat = min(apb, G.na[e] - b * apb);
    int const* __restrict__ atoms = G.atoms[e] + b * apb;
    const double* __restrict__ W = T.weights;
    // Thread -> (atom q, first neuron k0, neuron step).
    int const kstep = kGradThreads / apb;
    int const q = t % apb;
    int const k0 = q < nat && t / apb < kstep ? t / apb : INT_MAX / 2;
    double* const P = lds + (size_t)q * perAtom;
    // LDS layout per atom: for l = 1..L: X[l-1] (w_{l-1}), Tg[l-1]
    // (w_{l-1}), Z[l] (w_l), S[l] (w_l); then Xb, Tb (maxwidth each).
    int lo[kMaxLayers];   // offset of layer l's block within an atom
    {
        int p = 0;
        for (int l = 1; l <= L; ++l)
        {
            lo[l] = p;
            p += 2 * ed.width[l - 1] + 2 * ed.width[l];
        }
        lo[0] = p;        // adjoint scratch
    }
    double const kappa = 2.0 * A.wE * (A.energy[0] - A.Eref)
                       / ((double)A.n * (double)A.n);
    // inputs: scaled G and its tangent u
    {
        int const w0 = ed.width[0];
        for (int idx = t; idx < nat * w0; idx += kGradThreads)
        {
            int const m = idx / w0, j = idx - m * w0;
            size_t const g = (size_t)atoms[m] * A.ldG + j;
            double* X0 = lds + (size_t)m * perAtom + lo[1];
            X0[j] = A.G[g];
            X0[w0 + j] = A.U[g];
        }
    }
    __syncthreads();
    // forward with tangent
    for (int l = 1; l <= L; ++l)
    {
        int const nin = ed.width[l - 1], nout = ed.width[l];
        double const* X = P + lo[l];
        double const* Tg = X + nin;
        double* Z = P + lo[l] + 2 * nin;
        double* Xn = l < L ? P + lo[l + 1] : nullptr;
        for (int k = k0; k < nout; k += kstep)
        {
            double const* Wk = W + ed.woff[l] + (size_t)k * nin;
            double z = W[ed.boff[l] + k], s = 0.0;
#pragma unroll 4
            for (int j = 0; j < nin; ++j)
            {
                z += Wk[j] * X[j];
                s += Wk[j] * Tg[j];
            }
            Z[k] = z;
            Z[nout + k] = s;
            if (l < L)
            {
                double v, d, dd;
                activate2(ed.act[l], z, v, d, dd);
                Xn[k] = v;
                Xn[nout + k] = d * s;
            }
        }
        __syncthreads();
    }
    // reverse through value and tangent
    double* Xb = P + lo[0];
    double* Tb = Xb + ed.maxwidth;
    if (k0 == 0)
    {
        Xb[0] = kappa;
        Tb[0] = 1.0;
    }
    __syncthreads();
    for (int l = L; l >= 1; --l)
    {
        int const nin = ed.width[l - 1], nout = ed.width[l];
        double* Z = P + lo[l] + 2 * nin;
        double* S = Z + nout;
        double const* Wl = W + ed.woff[l];
        for (int k = k0; k < nout; k += kstep)
        {
            double v, d, dd;
            activate2(ed.act[l], Z[k], v, d, dd);
            double const zb = Xb[k] * d + Tb[k] * S[k] * dd;
            double const sb = Tb[k] * d;
            Z[k] = zb;       // adjoint of z replaces z
            S[k] = sb;       // adjoint of s replaces s
        }
        __syncthreads();
        if (l > 1)
        {
            for (int j = k0; j < nin; j += kstep)
            {
                double xb = 0.0, tb = 0.0;
#pragma unroll 4
                for (int k = 0; k < nout; ++k)
                {
                    xb += Wl[(size_t)k * nin + j] * Z[k];
                    tb += Wl[(size_t)k * nin + j] * S[k];
                }
                Xb[j] = xb;
                Tb[j] = tb;
            }
            __syncthreads();
        }
    }
    // dW_l[k][j] = sum_atoms zb_k x_j + sb_k t_j;  db_l[k] = sum_atoms zb_k
    double* __restrict__ part = partAll + G.off[e] + (size_t)b * nw;
    int const base = ed.woff[1];
    for (int idx = t; idx < nw; idx += kGradThreads)
    {
        int const gidx = base + idx;
        int l = 1;
        while (l < L && gidx >= ed.woff[l + 1]) ++l;
        int const nin = ed.width[l - 1], nout = ed.width[l];
        double acc = 0.0;
        if (gidx < ed.boff[l])
        {
            int const r = gidx - ed.woff[l];
            int const k = r / nin, j = r - k * nin;
            for (int m = 0; m < nat; ++m)
            {
                double const* X = lds + (size_t)m * perAtom + lo[l];
                double const* Z = X + 2 * nin;
                acc += Z[k] * X[j] + Z[nout + k] * X[nin + j];
            }
        }
        else
        {
            int const k = gidx - ed.boff[l];
            for (int m = 0; m < nat; ++m)
                acc += (lds + (size_t)m * perAtom + lo[l])[2 * nin + k];
        }
        part[idx] = acc;
    }
}

// grad[base + idx] = sum over the element's blocks of part (fixed order).
__global__ void k_train_reduce(TrainGradTab G, ModelTables T,
                               const double* __restrict__ partAll,
                               double* __restrict__ grad)
{
    int const e = blockIdx.y;
    int const idx = blockIdx.x * blockDim.x + threadIdx.x;
    int const nw = G.nw[e];
    if (idx >= nw) return;
    const double* __restrict__ part = partAll + G.off[e];
    double acc = 0.0;
#pragma unroll 8
    for (int b = 0; b < G.nb[e]; ++b) acc += part[(size_t)b * nw + idx];
    grad[T.elem[e].woff[1] + idx] = acc;
}

// Adam (Kingma & Ba 2015, Algorithm 1) on w with gradient g at step t >= 1.
__global__ void k_adam(int n, double* __restrict__ w,
                       float* __restrict__ w32,
                       const double* __restrict__ g, double* __restrict__ m,
                       double* __restrict__ v, double lr, double b1,
                       double b2, double eps, double c1, double c2)
{
    int const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double const gi = g[i];
    double const mi = b1 * m[i] + (1.0 - b1) * gi;
    double const vi = b2 * v[i] + (1.0 - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    double const wi = w[i] - lr * (mi / c1) / (sqrt(vi / c2) + eps);
    w[i] = wi;
    w32[i] = (float)wi;
}

__global__ void k_to_f32(int n, const double* __restrict__ w,
                         float* __restrict__ w32)
{
    int const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) w32[i] = (float)w[i];
}

// dE_s/dw for every structure s: per block (atoms of one element and one
// structure, at most kAtoms) the forward pass and backpropagation of each
// atom's network (NeuralNetwork::calculateDEdc, NeuralNetwork.cpp:444-490),
// then per weight the sum over the block's atoms in atom order.  LDS per
// atom: for every layer its input x and the adjoint of z, plus one adjoint
// scratch vector.  Threads share the layers as in k_train_grad (one thread
// per atom took 230 us for a 192-atom structure, now 39 us).
__global__ __launch_bounds__(kGradThreads) void k_energy_wgrad(
    ModelTables T, const double* __restrict__ G, int ldG,
    const int* __restrict__ blkAtoms, const int* __restrict__ blk0,
    const int* __restrict__ blkN, const int* __restrict__ blkElem,
    int perAtom, double* __restrict__ part, int maxP)
{
    extern __shared__ double lds[];
    int const b = blockIdx.x;
    int const t = threadIdx.x;
    int const e = blkElem[b];
    ElemDesc const& ed = T.elem[e];
    int const L = ed.nlayers - 1;
    int const nat = blkN[b];
    int const* __restrict__ atoms = blkAtoms + blk0[b];
    const double* __restrict__ W = T.weights;
    constexpr int kstep = kGradThreads / kAtoms;
    int const q = t % kAtoms;
    int const k0 = q < nat ? t / kAtoms : INT_MAX / 2;
    double* const P = lds + (size_t)q * perAtom;
    int lo[kMaxLayers];
    {
        int p = 0;
        for (int l = 1; l <= L; ++l)
        {
            lo[l] = p;
            p += ed.width[l - 1] + ed.width[l];
        }
        lo[0] = p;
    }
    {
        int const w0 = ed.width[0];
        for (int idx = t; idx < nat * w0; idx += kGradThreads)
        {
            int const m = idx / w0, j = idx - m * w0;
            (lds + (size_t)m * perAtom + lo[1])[j]
                = G[(size_t)atoms[m] * ldG + j];
        }
    }
    __syncthreads();
    for (int l = 1; l <= L; ++l)
    {
        int const nin = ed.width[l - 1], nout = ed.width[l];
        double const* X = P + lo[l];
        double* Z = P + lo[l] + nin;
        double* Xn = l < L ? P + lo[l + 1] : nullptr;
        for (int k = k0; k < nout; k += kstep)
        {
            double const* Wk = W + ed.woff[l] + (size_t)k * nin;
            double z = W[ed.boff[l] + k];
#pragma unroll 4
            for (int j = 0; j < nin; ++j) z += Wk[j] * X[j];
            Z[k] = z;
            if (l < L)
            {
                double v, d;
                activate(ed.act[l], z, v, d);
                Xn[k] = v;
            }
        }
        __syncthreads();
    }
    double* Xb = P + lo[0];
    for (int k = k0; k < ed.width[L]; k += kstep) Xb[k] = 1.0;
    __syncthreads();
    for (int l = L; l >= 1; --l)
    {
        int const nin = ed.width[l - 1], nout = ed.width[l];
        double* Z = P + lo[l] + nin;
        const double* Wl = W + ed.woff[l];
        for (int k = k0; k < nout; k += kstep)
        {
            double v, d;
            activate(ed.act[l], Z[k], v, d);
            Z[k] = Xb[k] * d;        // adjoint of z replaces z
        }
        __syncthreads();
        if (l > 1)
        {
            for (int j = k0; j < nin; j += kstep)
            {
                double xb = 0.0;
#pragma unroll 4
                for (int k = 0; k < nout; ++k)
                    xb += Wl[(size_t)k * nin + j] * Z[k];
                Xb[j] = xb;
            }
            __syncthreads();
        }
    }
    int const base = ed.woff[1];
    int nw = 0;
    for (int l = 1; l <= L; ++l) nw += ed.width[l] * ed.width[l - 1] + ed.width[l];
    for (int idx = t; idx < nw; idx += kGradThreads)
    {
        int const gidx = base + idx;
        int l = 1;
        while (l < L && gidx >= ed.woff[l + 1]) ++l;
        int const nin = ed.width[l - 1];
        double acc = 0.0;
        if (gidx < ed.boff[l])
        {
            int const r = gidx - ed.woff[l];
            int const k = r / nin, j = r - k * nin;
            for (int m = 0; m < nat; ++m)
            {
                double const* X = lds + (size_t)m * perAtom + lo[l];
                acc += X[nin + k] * X[j];
            }
        }
        else
        {
            int const k = gidx - ed.boff[l];
            for (int m = 0; m < nat; ++m)
                acc += (lds + (size_t)m * perAtom + lo[l])[nin + k];
        }
        part[(size_t)b * maxP + idx] = acc;
    }
}

// J[s][base_e + idx] = sum over the blocks of (structure s, element e), in
// block order.  One workgroup per (s, e) and 256 weights; blocks of (s, e)
// are [grp0[s*ne+e], grp0[s*ne+e+1]).
__global__ __launch_bounds__(256) void k_energy_wgrad_reduce(
    const double* __restrict__ part, int maxP, const int* __restrict__ grp0,
    const int* __restrict__ base, const int* __restrict__ nwe, int ne,
    int nwTotal, double* __restrict__ J)
{
    int const se = blockIdx.x;
    int const s = se / ne, e = se - s * ne;
    int const b0 = grp0[se], b1 = grp0[se + 1];
    int const idx = blockIdx.y * 256 + threadIdx.x;
    if (idx >= nwe[e]) return;
    double acc = 0.0;
#pragma unroll 4
    for (int b = b0; b < b1; ++b) acc += part[(size_t)b * maxP + idx];
    J[(size_t)s * nwTotal + base[e] + idx] = acc;
}

// Kalman filter, one scalar observation (KalmanFilter.cpp:126-196 with
// sizeObservation 1): X = P h, one wave per row of the symmetric P.
__global__ __launch_bounds__(64) void k_kf_gemv(int nw,
                                                const double* __restrict__ P,
                                                const double* __restrict__ h,
                                                double* __restrict__ X)
{
    int const i = blockIdx.x;
    if (i >= nw) return;
    double acc = 0.0;
    for (int j = threadIdx.x; j < nw; j += 64)
        acc += P[(size_t)i * nw + j] * h[j];
    acc = wave_sum(acc);
    if (threadIdx.x == 0) X[i] = acc;
}

// a = h . X (one workgroup, fixed order).
__global__ __launch_bounds__(256) void k_kf_dot(int nw,
                                                const double* __restrict__ h,
                                                const double* __restrict__ X,
                                                double* __restrict__ a)
{
    __shared__ double s[256];
    int const t = threadIdx.x;
    double acc = 0.0;
    for (int j = t; j < nw; j += 256) acc += h[j] * X[j];
    s[t] = acc;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1)
    {
        if (t < o) s[t] += s[t + o];
        __syncthreads();
    }
    if (t == 0) a[0] = s[0];
}

// K = X / (a + 1/eta); P -= K X^T; P += q I; w += K xi.  One workgroup
// per row of P, threads over its columns.
__global__ __launch_bounds__(256) void k_kf_update(
    int nw, double* __restrict__ P, const double* __restrict__ X,
    const double* __restrict__ a, double rinv, double q, double xi,
    double* __restrict__ w, float* __restrict__ w32)
{
    int const i = blockIdx.x;
    if (i >= nw) return;
    double const den = a[0] + rinv;
    double const Ki = X[i] / den;
    double const Xi = X[i];
    double* __restrict__ Pi = P + (size_t)i * nw;
    // (X_i X_j) / den: the same operands for (i, j) and (j, i), so P stays
    // exactly symmetric.
    for (int j = threadIdx.x; j < nw; j += 256)
    {
        double v = Pi[j] - (Xi * X[j]) / den;
        if (j == i) v += q;
        Pi[j] = v;
    }
    if (threadIdx.x == 0)
    {
        double const wi = w[i] + Ki * xi;
        w[i] = wi;
        w32[i] = (float)wi;
    }
}

__global__ void k_kf_init(int nw, double* __restrict__ P, double diag)
{
    size_t const k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (size_t)nw * nw) return;
    int const i = (int)(k / nw), j = (int)(k - (size_t)i * nw);
    P[k] = i == j ? diag : 0.0;
}

}  // namespace

hipError_t launch_kf_init(int nw, double* P, double diag, hipStream_t s)
{
    size_t const tot = (size_t)nw * nw;
    if (tot == 0) return hipSuccess;
    k_kf_init<<<(unsigned)((tot + 255) / 256), 256, 0, s>>>(nw, P, diag);
    return hipGetLastError();
}

hipError_t launch_kf_update(int nw, double* P, const double* h, double* X,
                            double* a, double rinv, double q, double xi,
                            double* w, float* w32, hipStream_t s)
{
    if (nw <= 0) return hipSuccess;
    k_kf_gemv<<<nw, 64, 0, s>>>(nw, P, h, X);
    k_kf_dot<<<1, 256, 0, s>>>(nw, h, X, a);
    k_kf_update<<<nw, 256, 0, s>>>(nw, P, X, a, rinv, q, xi, w, w32);
    return hipGetLastError();
}

hipError_t launch_energy_wgrad(ModelTables const& T, const double* G, int ldG,
                               const int* blkAtoms, const int* blk0,
                               const int* blkN, const int* blkElem, int nblk,
                               int perAtom, double* part, int maxP,
                               const int* grp0, const int* base,
                               const int* nwe, int ne, int nstruct,
                               int nwTotal, double* J, hipStream_t s)
{
    // An odd record stride where it fits (the caller checked perAtom).
    int const odd = perAtom | 1;
    int const stride = (size_t)odd * kAtoms * sizeof(double) <= 65536
                     ? odd : perAtom;
    if (nblk > 0)
        k_energy_wgrad<<<nblk, kGradThreads,
                         (size_t)stride * kAtoms * sizeof(double), s>>>(
            T, G, ldG, blkAtoms, blk0, blkN, blkElem, stride, part, maxP);
    if (nstruct * ne > 0)
        k_energy_wgrad_reduce<<<dim3(nstruct * ne, (maxP + 255) / 256), 256,
                                0, s>>>(part, maxP, grp0, base, nwe, ne,
                                        nwTotal, J);
    return hipGetLastError();
}

int train_atoms_per_block() { return kAtoms; }

namespace {

// Doubles between the atoms' LDS records of the loss-gradient kernel: odd
// unless only the exact size fits.
size_t train_lds_stride(ElemDesc const& ed)
{
    size_t const per = train_lds_per_atom(ed);
    return (per | 1) * sizeof(double) <= 65536 ? per | 1 : per;
}

}  // namespace

// Atoms per block of the loss-gradient kernel: up to kAtoms, fewer for wide
// networks so that their LDS stays within 64 KiB (0 if one atom does not
// fit).
int train_atoms_per_grad_block(ElemDesc const& ed)
{
    return (int)std::min<size_t>(kAtoms, 65536 / (train_lds_stride(ed)
                                                  * sizeof(double)));
}

size_t train_lds_per_atom(ElemDesc const& ed)
{
    size_t p = 0;
    for (int l = 1; l < ed.nlayers; ++l)
        p += 2 * ed.width[l - 1] + 2 * ed.width[l];
    return p + 2 * ed.maxwidth;
}

// 11 doubles per staged neighbour and the pair queue, as the FP64 force kernel
// before the pair search.  Also on the mixed path, whose force kernel admits
// lists by 56 bytes per neighbour, up to 1,161: 102 KB here.
size_t train_u_lds_bytes(int cap)
{
    return force_list_lds_bytes(cap, 0) + kTrainStatic;
}

hipError_t launch_train_u(TrainArgs const& A, hipStream_t s)
{
    if (A.n <= 0) return hipSuccess;
    if (A.T.maxGroupMembers <= 8) launch_train_u_m<8>(A, s);
    else launch_train_u_m<kMaxMembers>(A, s);
    return hipGetLastError();
}

size_t train_grad_partials(ElemDesc const& ed, int na)
{
    size_t const apb = std::max(train_atoms_per_grad_block(ed), 1);
    size_t nw = 0;
    for (int l = 1; l < ed.nlayers; ++l)
        nw += (size_t)ed.width[l] * ed.width[l - 1] + ed.width[l];
    return nw * ((na + apb - 1) / apb);
}

hipError_t launch_train_grad(TrainArgs const& A, ElemDesc const* eds,
                             const int* const* atoms, const int* na,
                             double* part, double* grad, hipStream_t s)
{
    TrainGradTab G{};
    size_t off = 0, shm = 0;
    int nb = 0, nw = 0;
    for (int e = 0; e < A.T.ne; ++e)
    {
        ElemDesc const& ed = eds[e];
        G.atoms[e] = atoms[e];
        G.na[e] = na[e];
        G.apb[e] = train_atoms_per_grad_block(ed);
        G.stride[e] = (int)train_lds_stride(ed);
        G.nb[e] = (na[e] + G.apb[e] - 1) / G.apb[e];
        for (int l = 1; l < ed.nlayers; ++l)
            G.nw[e] += ed.width[l] * ed.width[l - 1] + ed.width[l];
        G.off[e] = off;
        off += train_grad_partials(ed, na[e]);
        if (na[e] > 0)
            shm = std::max(shm, (size_t)G.stride[e] * G.apb[e]
                                * sizeof(double));
        nb = std::max(nb, G.nb[e]);
        nw = std::max(nw, G.nw[e]);
    }
    if (nb > 0)
        k_train_grad<<<dim3(nb, A.T.ne), kGradThreads, shm, s>>>(A, G, part);
    k_train_reduce<<<dim3((nw + 255) / 256, A.T.ne), 256, 0, s>>>(G, A.T,
                                                                 part, grad);
    return hipGetLastError();
}

hipError_t launch_adam(int n, double* w, float* w32, const double* g,
                       double* m, double* v, double lr, double b1, double b2,
                       double eps, int64_t step, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    double const c1 = 1.0 - std::pow(b1, (double)step);
    double const c2 = 1.0 - std::pow(b2, (double)step);
    k_adam<<<(n + 255) / 256, 256, 0, s>>>(n, w, w32, g, m, v, lr, b1, b2,
                                           eps, c1, c2);
    return hipGetLastError();
}

hipError_t launch_weights_to_f32(int n, const double* w, float* w32,
                                 hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    k_to_f32<<<(n + 255) / 256, 256, 0, s>>>(n, w, w32);
    return hipGetLastError();
}

}  // namespace hdnnp
