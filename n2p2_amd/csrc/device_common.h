// Device helpers shared by the HIP kernels: cutoff functions, integer
// powers, activations and 64-lane wave reductions, templated on the
// arithmetic type (double, or float on the mixed-precision path).
#ifndef HDNNP_DEVICE_COMMON_H
#define HDNNP_DEVICE_COMMON_H

#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#endif

#include "tables.h"

namespace hdnnp {

constexpr int kWave = 64;
constexpr double kPi = 3.141592653589793238462643383279502884;

// Entries of the LDS queue of passing neighbour pairs (two batches of 64).
constexpr int kQueue = 128;

// q = p / d, r = p % d for 0 <= p < 2^22 and d > 0 from inv = 1 / (float)d:
// the float quotient is off by at most one, which the correction fixes.
__device__ __forceinline__ void divmod_small(int p, int d, float inv, int& q,
                                             int& r)
{
    q = (int)((float)p * inv);
    r = p - q * d;
    if (r < 0) { --q; r += d; }
    else if (r >= d) { ++q; r -= d; }
}

// Four- and two-component vectors of the arithmetic type R (LDS records).
template <typename R> struct VecT;
template <> struct VecT<float> { typedef float4 V4; typedef float2 V2; };
template <> struct VecT<double> { typedef double4 V4; typedef double2 V2; };
template <typename R> using Vec4 = typename VecT<R>::V4;
template <typename R> using Vec2 = typename VecT<R>::V2;

// sin(pi x) and cos(pi x) for x in [0, 1].  With u = x - 1/2:
// cos(pi x) = -sin(pi u) and sin(pi x) = cos(pi u); both are evaluated from
// their Taylor series in t = u^2 (|u| <= 1/2), truncated after the first
// term below 1e-17.  The coefficients (-1)^k pi^(2k+1)/(2k+1)! and
// (-1)^k pi^(2k)/(2k)! were computed in 60-digit arithmetic and rounded to
// double.  Max abs error against libm over [0, 1]: 4.4e-16.
__device__ __forceinline__ void sincospi01(double x, double& s, double& c)
{
    double const u = x - 0.5;
    double const t = u * u;
    double sp = -1.05184717169320651e-11;
    sp = fma(sp, t, 5.39266466260812895e-10);
    sp = fma(sp, t, -2.29484289972698730e-08);
    sp = fma(sp, t, 7.95205400147551261e-07);
    sp = fma(sp, t, -2.19153534478302173e-05);
    sp = fma(sp, t, 4.66302805767612554e-04);
    sp = fma(sp, t, -7.37043094571435044e-03);
    sp = fma(sp, t, 8.21458866111282326e-02);
    sp = fma(sp, t, -5.99264529320792105e-01);
    sp = fma(sp, t, 2.55016403987734552e+00);
    sp = fma(sp, t, -5.16771278004997026e+00);
    sp = fma(sp, t, 3.14159265358979312e+00);
    double cp = 1.37686472803774139e-12;
    cp = fma(cp, t, -7.70070713060135385e-11);
    cp = fma(cp, t, 3.60473079746250112e-09);
    cp = fma(cp, t, -1.38789524622137714e-07);
    cp = fma(cp, t, 4.30306958703294729e-06);
    cp = fma(cp, t, -1.04638104924845705e-04);
    cp = fma(cp, t, 1.92957430940392314e-03);
    cp = fma(cp, t, -2.58068913900140612e-02);
    cp = fma(cp, t, 2.35330630358893206e-01);
    cp = fma(cp, t, -1.33526276885458950e+00);
    cp = fma(cp, t, 4.05871212641676848e+00);
    cp = fma(cp, t, -4.93480220054467900e+00);
    cp = fma(cp, t, 1.0);
    c = -u * sp;
    s = cp;
}

// FP32: the hardware sine and cosine (v_sin_f32 / v_cos_f32 take the
// angle in revolutions, so pi x is x / 2 revolutions).  Max abs error
// against libm over [0, 1]: 1.3e-7 (measured on gfx950 with an in-bounds
// probe over 2^20 points).
__device__ __forceinline__ void sincospi01(float x, float& s, float& c)
{
    float const rev = 0.5f * x;
    s = __builtin_amdgcn_sinf(rev);
    c = __builtin_amdgcn_cosf(rev);
}

// sin and cos of pi r iw, r iw in [0, 1] (FP32: half the scale as the
// revolutions, which rounds as r iw / 2 does).  Two neighbours at one place
// have r = 0 1/sqrt(0), NaN, for 0; FP32: the clamp, a modifier of the
// multiplication, makes it that.
__device__ __forceinline__ void sincospi_scaled(double r, double iw, double& s,
                                                double& c)
{
    sincospi01(fmax(r, 0.0) * iw, s, c);
}

__device__ __forceinline__ void sincospi_scaled(float r, float iw, float& s,
                                                float& c)
{
    float const rev = fminf(fmaxf(r * (0.5f * iw), 0.0f), 1.0f);
    s = __builtin_amdgcn_sinf(rev);
    c = __builtin_amdgcn_cosf(rev);
}

// 1/sqrt(x) for x > 0: hardware estimate refined by two Newton steps
// y <- y (3 - x y^2) / 2 (each step squares the relative error).
__device__ __forceinline__ double rsqrt_nr(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    double const hx = 0.5 * x;
    y = y * fma(-hx * y, y, 1.5);
    y = y * fma(-hx * y, y, 1.5);
    return y;
}

// FP32: the hardware estimate (1 ulp) as it is.
__device__ __forceinline__ float rsqrt_nr(float x)
{
    return __builtin_amdgcn_rsqf(x);
}

// e^x.  FP64: the library function.  FP32: the hardware 2^x of x log2(e)
// (relative error below 2e-6 for |x| < 30, the range of the SF exponents).
__device__ __forceinline__ double exp_r(double x) { return exp(x); }
__device__ __forceinline__ float exp_r(float x) { return __expf(x); }

// 1 / x.  FP64: IEEE division.  FP32: the hardware reciprocal (1 ulp).
__device__ __forceinline__ double rcp_r(double x) { return 1.0 / x; }
__device__ __forceinline__ float rcp_r(float x)
{
    return __builtin_amdgcn_rcpf(x);
}

__device__ __forceinline__ double tanh_r(double x) { return tanh(x); }
__device__ __forceinline__ float tanh_r(float x) { return tanhf(x); }

// CutoffFunction::fdf (CutoffFunction.h:210-220, CutoffFunction.cpp:128-213,
// CoreFunction.h:214-318): value and derivative, zero at and beyond rc.
// R is the arithmetic type (double, or float on the mixed-precision path).
template <typename R>
__device__ __forceinline__ void cutoff_fdf(CutCfg const& c, R r, R& fc,
                                           R& dfc)
{
    if (r >= (R)c.rc) { fc = R(0); dfc = R(0); return; }
    int const t = c.type;
    if (t == CT_TANHU || t == CT_TANH)
    {
        R const th = tanh_r(R(1) - r * (R)c.rcinv);
        R const th2 = th * th;
        // CT_TANH multiplies by tanh(1)^-3 so that f(0) = 1 (host-computed).
        R const pre = (t == CT_TANH) ? (R)c.tanhpre : R(1);
        fc = pre * th * th2;
        dfc = R(3) * pre * th2 * (th2 - R(1)) * (R)c.rcinv;
        return;
    }
    if (t == CT_HARD) { fc = R(1); dfc = R(0); return; }
    if (r < (R)c.rci) { fc = R(1); dfc = R(0); return; }
    R const iw = (R)c.iw;
    R const x = (r - (R)c.rci) * iw;
    if (t == CT_COS)
    {
        // f = (cos(pi x) + 1)/2, f' = -iw pi sin(pi x)/2; the reference
        // forms sin(pi x) as sqrt(1 - cos^2), equal on [0, 1].
        R sn, cs;
        sincospi01(x, sn, cs);
        fc = R(0.5) * (cs + R(1));
        dfc = R(-0.5) * iw * (R)kPi * sn;
        return;
    }
    R f, df;
    if (t == CT_POLY1)
    {
        f = (R(2) * x - R(3)) * x * x + R(1);
        df = x * (R(6) * x - R(6));
    }
    else if (t == CT_POLY2)
    {
        R const x2 = x * x;
        f = ((R(15) - R(6) * x) * x - R(10)) * x * x2 + R(1);
        df = x2 * ((R(60) - R(30) * x) * x - R(30));
    }
    else if (t == CT_POLY3)
    {
        R const x2 = x * x;
        f = (x * (x * (R(20) * x - R(70)) + R(84)) - R(35)) * x2 * x2 + R(1);
        df = x2 * x * (x * (x * (R(140) * x - R(420)) + R(420)) - R(140));
    }
    else if (t == CT_POLY4)
    {
        R x4 = x * x;
        x4 *= x4;
        f = (x * (x * ((R(315) - R(70) * x) * x - R(540)) + R(420)) - R(126))
          * x * x4 + R(1);
        df = x4 * (x * (x * ((R(2520) - R(630) * x) * x - R(3780))
                        + R(2520)) - R(630));
    }
    else  // CT_EXP: f(x) = e^(1 - 1/(1-x^2))
    {
        R const e = (R)2.718281828459045090795598298427648842334747314453125;
        R const tmp = R(1) / (x * x - R(1));
        R const ex = exp_r(tmp);
        f = e * ex;
        df = R(-2) * e * x * tmp * tmp * ex;
    }
    fc = f;
    dfc = df * iw;
}

// Cutoff with the type fixed at compile time (CT >= 0) or read from the
// configuration (CT < 0).  The specialised forms keep the heavy kernels
// free of the other types' code and registers.
template <int CT, typename R>
__device__ __forceinline__ void cutoff_fdf_t(CutCfg const& c, R r, R& fc,
                                             R& dfc)
{
    if (CT < 0)
    {
        cutoff_fdf(c, r, fc, dfc);
        return;
    }
    if (r >= (R)c.rc) { fc = R(0); dfc = R(0); return; }
    if (CT == CT_TANHU)
    {
        R const th = tanh_r(R(1) - r * (R)c.rcinv);
        R const th2 = th * th;
        fc = th * th2;
        dfc = R(3) * th2 * (th2 - R(1)) * (R)c.rcinv;
        return;
    }
    if (r < (R)c.rci) { fc = R(1); dfc = R(0); return; }
    R const iw = (R)c.iw;
    R const x = (r - (R)c.rci) * iw;
    if (CT == CT_COS)
    {
        R sn, cs;
        sincospi01(x, sn, cs);
        fc = R(0.5) * (cs + R(1));
        dfc = R(-0.5) * iw * (R)kPi * sn;
    }
    else   // CT_POLY2
    {
        R const x2 = x * x;
        fc = ((R(15) - R(6) * x) * x - R(10)) * x * x2 + R(1);
        dfc = x2 * ((R(60) - R(30) * x) * x - R(30)) * iw;
    }
}

// The cutoff configuration of a group: the model's one configuration as
// literals where the model-specialised build defines it.
#ifndef HDNNP_CUT
#define HDNNP_CUT(cfg) (cfg)
#endif

// Launches KERNEL<CT, ...> for the cutoff types with specialised code and
// KERNEL<-1, ...> (runtime switch) for the others.
#define HDNNP_CUTOFF_DISPATCH(ct, CALL)                                    \
    do                                                                     \
    {                                                                      \
        switch (ct)                                                        \
        {                                                                  \
        case CT_COS: { constexpr int kCT = CT_COS; CALL; } break;           \
        case CT_TANHU: { constexpr int kCT = CT_TANHU; CALL; } break;       \
        case CT_POLY2: { constexpr int kCT = CT_POLY2; CALL; } break;       \
        default: { constexpr int kCT = -1; CALL; } break;                   \
        }                                                                  \
    } while (0)

// Exponentiation by squaring (utility.cpp:292-317 semantics).
template <typename R>
__device__ __forceinline__ R pow_int(R x, int n)
{
    unsigned m;
    if (n < 0) { x = R(1) / x; m = (unsigned)(-n); }
    else m = (unsigned)n;
    R r = R(1);
    do
    {
        if (m & 1u) r *= x;
        m >>= 1;
        x *= x;
    } while (m);
    return r;
}

// x^N with the products pow_int forms for exponent N, N fixed at compile
// time: straight-line code, bit-identical to pow_int(x, N).
template <int N, typename R>
__device__ __forceinline__ R pow_fixed(R x)
{
    R r = R(1);
    bool first = true;
    int m = N;
#pragma unroll
    for (int b = 0; b < 6; ++b)
    {
        if (m & 1)
        {
            r = first ? x : r * x;
            first = false;
        }
        m >>= 1;
        if (m) x *= x;
    }
    return r;
}

// Powers of x = plambda shared by the members of an (eta, rs, lambda) run
// sorted by zeta: after l steps P = x^(2^l - 1) and X = x^(2^l), the
// running product and square of pow_int's loop, so at(l) for zeta = 2^l is
// bit-identical to pow_int(x, zeta - 1).  l is wave-uniform.
template <typename R>
struct PowChain
{
    R P, X;
    int l;
    __device__ __forceinline__ void reset(R x)
    {
        P = R(1);
        X = x;
        l = 0;
    }
    __device__ __forceinline__ R at(int level)
    {
        while (l < level)
        {
            P *= X;
            X *= X;
            ++l;
        }
        return P;
    }
};

// pow_int(x, n) for a wave-uniform n: a scalar branch to straight-line
// products for 0 <= n <= 16, the loop otherwise.
template <typename R>
__device__ __forceinline__ R pow_uniform(R x, int n)
{
    switch (n)
    {
    case 0: return R(1);
    case 1: return x;
    case 2: return pow_fixed<2>(x);
    case 3: return pow_fixed<3>(x);
    case 4: return pow_fixed<4>(x);
    case 5: return pow_fixed<5>(x);
    case 6: return pow_fixed<6>(x);
    case 7: return pow_fixed<7>(x);
    case 8: return pow_fixed<8>(x);
    case 9: return pow_fixed<9>(x);
    case 10: return pow_fixed<10>(x);
    case 11: return pow_fixed<11>(x);
    case 12: return pow_fixed<12>(x);
    case 13: return pow_fixed<13>(x);
    case 14: return pow_fixed<14>(x);
    case 15: return pow_fixed<15>(x);
    case 16: return pow_fixed<16>(x);
    default: return pow_int(x, n);
    }
}

// NeuralNetwork::propagateLayer activations (NeuralNetwork.cpp:761-896):
// value and first derivative.  Logistic and softplus clamp at |x| > 35.
__device__ __forceinline__ void activate(int a, double x, double& v, double& d)
{
    switch (a)
    {
    case AF_IDENTITY: v = x; d = 1.0; break;
    case AF_TANH:
    {
        double const t = tanh(x);
        v = t; d = 1.0 - t * t;
        break;
    }
    case AF_LOGISTIC:
        if (x > 35.0) { v = 1.0; d = 0.0; }
        else if (x < -35.0) { v = 0.0; d = 0.0; }
        else
        {
            double const s = 1.0 / (1.0 + exp(-x));
            v = s; d = s * (1.0 - s);
        }
        break;
    case AF_SOFTPLUS:
        if (x > 35.0) { v = x; d = 1.0; }
        else if (x < -35.0) { v = 0.0; d = 0.0; }
        else
        {
            double const ex = exp(x);
            v = log(1.0 + ex);
            d = 1.0 / (1.0 + 1.0 / ex);
        }
        break;
    case AF_RELU:
        if (x > 0.0) { v = x; d = 1.0; } else { v = 0.0; d = 0.0; }
        break;
    case AF_GAUSSIAN:
    {
        double const g = exp(-0.5 * x * x);
        v = g; d = -x * g;
        break;
    }
    case AF_COS: v = cos(x); d = -sin(x); break;
    case AF_REVLOGISTIC:
    {
        double const s = 1.0 / (1.0 + exp(-x));
        v = 1.0 - s; d = s * (s - 1.0);
        break;
    }
    case AF_EXP:
    {
        double const e = exp(-x);
        v = e; d = -e;
        break;
    }
    case AF_HARMONIC: v = x * x; d = 2.0 * x; break;
    default: v = 0.0; d = 0.0; break;
    }
}

// Member parameters of one group, staged in LDS at the start of the group
// and read with wave-uniform addresses (broadcast) inside the pair loops.
// Integer fields are made scalar with readfirstlane where they steer
// branches.
enum MemberFlags
{
    MF_INTPOW = 1,   // integer zeta (pow_int)
    MF_NEWEXP = 2,   // first member of an (eta, rs) run: new exponential
    MF_NEWLAM = 4,   // first member of an (eta, rs, lambda) run
    MF_PREFIX = 8    // zeta = 2^level: power from the run's prefix chain
};

template <typename R>
struct MParam
{
    R   lambda, zl, eta, rs, zeta, w;   // w: per-kernel weight
    int zint, flags;                    // flags | level << 8
};

template <typename R>
__device__ __forceinline__ MParam<R> make_mparam(MemberDesc const& md,
                                                 double w)
{
    MParam<R> p;
    p.lambda = (R)md.lambda;
    p.zl = (R)md.zl;
    p.eta = (R)md.eta;
    p.rs = (R)md.rs;
    p.zeta = (R)md.zeta;
    p.w = (R)w;
    p.zint = md.zint;
    p.flags = (md.useint ? MF_INTPOW : 0) | (md.calcexp ? MF_NEWEXP : 0)
            | (md.newlam ? MF_NEWLAM : 0)
            | (md.level >= 0 ? MF_PREFIX | (md.level << 8) : 0);
    return p;
}

__device__ __forceinline__ int uniform(int v)
{
    return __builtin_amdgcn_readfirstlane(v);
}

// Wave-uniform copies of floating-point values (scalar registers).
__device__ __forceinline__ float uniform_r(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

__device__ __forceinline__ double uniform_r(double v)
{
    long long const b = __double_as_longlong(v);
    int const lo = __builtin_amdgcn_readfirstlane((int)b);
    int const hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// exp(-eta s) from the exponent factor of exp_factor(eta): FP64 takes the
// library exp of -eta s; FP32 the hardware 2^x of (-eta log2 e) s.
__device__ __forceinline__ double exp_factor(double eta) { return -eta; }
__device__ __forceinline__ float exp_factor(float eta)
{
    return -eta * 1.44269504088896340736f;
}
__device__ __forceinline__ double exp_scaled(double a) { return exp(a); }
__device__ __forceinline__ float exp_scaled(float a)
{
    return __builtin_amdgcn_exp2f(a);
}

// Cutoff value and derivative for rc > r >= 0 without branches for the
// specialised types: x = (r - rci) iw clamped to [0, 1] gives f = 1, f' = 0
// below rci exactly as the branch does (the cosine form to rounding).  Other
// types take the general form.
template <int CT, typename R>
__device__ __forceinline__ void cutoff_inside(CutCfg const& c, R r, R& fc,
                                              R& dfc)
{
    if (CT == CT_COS)
    {
        R const iw = (R)c.iw;
        R sn, cs;
        // No inner radius (known when the model's one cutoff is compiled in):
        // x = r iw is in [0, 1] as it is.
        if (__builtin_constant_p(c.rci) && c.rci == 0.0)
            sincospi_scaled(r, iw, sn, cs);
        else
        {
            R x = (r - (R)c.rci) * iw;
            x = fmin(fmax(x, R(0)), R(1));
            sincospi01(x, sn, cs);
        }
        fc = fma(R(0.5), cs, R(0.5));
        dfc = R(-0.5) * iw * (R)kPi * sn;
    }
    else if (CT == CT_POLY2)
    {
        R const iw = (R)c.iw;
        R x = (r - (R)c.rci) * iw;
        x = fmin(fmax(x, R(0)), R(1));
        R const x2 = x * x;
        fc = ((R(15) - R(6) * x) * x - R(10)) * x * x2 + R(1);
        dfc = x2 * ((R(60) - R(30) * x) * x - R(30)) * iw;
    }
    else cutoff_fdf_t<CT>(c, r, fc, dfc);
}

// SymFnc::scale (SymFnc.cpp:169-195).
__device__ __forceinline__ double scale_sf(ScaleDesc const& s, double v)
{
    switch (s.type)
    {
    case ST_NONE: return v;
    case ST_SCALE: return s.smin + s.sfac * (v - s.gmin);
    case ST_CENTER: return v - s.gmean;
    case ST_SCALECENTER:
    case ST_SCALESIGMA: return s.smin + s.sfac * (v - s.gmean);
    }
    return 0.0;
}

// Butterfly sum over the 64 lanes of a wave; every lane gets the total.
// The pairing pattern is fixed, so the result is deterministic.  Float
// partials are summed in FP64.
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ int wave_sum_int(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & 63u); }

// Work index of workgroup b of nb.  The hardware deals workgroups to the 8
// XCDs round-robin (XCD = b % 8); this mapping gives each XCD one contiguous
// range of work indices, so work items that touch the same data (atoms of
// neighbouring cells) share that XCD's L2.  A bijection on [0, nb).
__device__ __forceinline__ int xcd_work_index(int b, int nb)
{
    int const x = b & 7, k = b >> 3;
    int const q = nb >> 3, r = nb & 7;   // XCD x holds q + (x < r) groups
    return x * q + (x < r ? x : r) + k;
}

// Sums M per-lane values over the wave by a transposing butterfly: at each
// of the first log2(M) steps a lane keeps half of its values, sends the
// other half to the partner lane (xor 32, 16, ...) and adds what it
// receives, then the remaining steps are a plain butterfly.  Returns the
// total of member ((lane >> (6 - log2 M)) & (M - 1)); every lane of that
// group of 64/M lanes holds it.  M - 1 + 6 - log2(M) exchanges and adds
// instead of 6 M for M separate sums; the order of the additions is fixed.
template <int M>
__device__ __forceinline__ double wave_sum_transposed(double (&v)[M])
{
    static_assert(M == 1 || M == 2 || M == 4 || M == 8 || M == 16
                  || M == 32, "power of two up to 32");
    int const lane = lane_id();
#pragma unroll
    for (int h = M / 2, o = 32; h >= 1; h >>= 1, o >>= 1)
    {
        bool const upper = (lane & o) != 0;
#pragma unroll
        for (int m = 0; m < h; ++m)
        {
            double const send = upper ? v[m] : v[m + h];
            double const keep = upper ? v[m + h] : v[m];
            v[m] = keep + __shfl_xor(send, o, kWave);
        }
    }
    double t = v[0];
#pragma unroll
    for (int o = 32 / M; o > 0; o >>= 1) t += __shfl_xor(t, o, kWave);
    return t;
}

// Orders this wave's LDS accesses around a queue hand-off between lanes,
// where the workgroup is one wave: a wave's LDS operations complete in
// issue order, so a wavefront-scope fence (no wait, unlike the workgroup
// barrier's fence) is enough and later LDS reads no longer wait for the
// queue writes before them to complete.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// Number of set bits of a 64-lane ballot below this lane (two mbcnt
// instructions).
__device__ __forceinline__ int lanes_below(uint64_t mask)
{
    return (int)__builtin_amdgcn_mbcnt_hi(
        (unsigned)(mask >> 32),
        __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// Unordered pairs {j, k} of a group's neighbour blocks in diagonal order.
// Same element (block of n at s0): pair p = c n + r is {r, (r + 1 + c) mod
// n}, at circular distance 1 + c.  The (n - 1) / 2 full diagonals
// (distance below n/2) hold n pairs each; for n even the half diagonal at
// distance n/2 follows with r < n/2.  Every unordered pair appears once
// (n (n - 1) / 2 in all) and one diagonal holds each slot at most twice.
// Different elements, smaller block s0 (ns) and larger block l0 (nl):
// p = c ns + r is {s0 + r, l0 + (r + c) mod nl}, c < nl; one diagonal holds
// each slot at most once.  A lane walks p = lane, lane + 64, ... with an
// incremental (c, r) (no division per step).
struct DiagPairs
{
    bool same;
    int s0, ns, l0, nl, d, npairs;
    int q64, r64;     // 64 = q64 d + r64
    __device__ DiagPairs(bool same_, int a0, int na, int b0, int nb)
        : same(same_)
    {
        if (same)
        {
            s0 = l0 = a0;
            ns = nl = na;
            d = na;
            npairs = na * (na - 1) / 2;
        }
        else
        {
            bool const aSmall = na <= nb;
            s0 = aSmall ? a0 : b0;
            ns = aSmall ? na : nb;
            l0 = aSmall ? b0 : a0;
            nl = aSmall ? nb : na;
            d = ns;
            npairs = na * nb;
        }
        q64 = d > 0 ? 64 / d : 0;
        r64 = 64 - q64 * d;
    }
    // Cursor (c, r) of pair p0 (one division, at the start).
    __device__ void start(int p0, int& c, int& r) const
    {
        c = 0;
        r = 0;
        if (d > 0) divmod_small(p0, d, 1.0f / (float)d, c, r);
    }
    // (c, r) of pair p -> pair p + 64.
    __device__ void advance(int& c, int& r) const
    {
        r += r64;
        c += q64;
        if (r >= d) { r -= d; ++c; }
    }
    // Staged indices of pair (c, r); only for p < npairs.
    __device__ void pair(int c, int r, int& j, int& k) const
    {
        int v = r + c + (same ? 1 : 0);
        // r < d and c < nl (c < n/2 for one block): one subtraction.
        if (v >= nl) v -= nl;
        j = s0 + r;
        k = l0 + v;
    }
};

// rij, rik < rc and (narrow only) rjk^2 < rc^2 from the staged records
// (SymGrpExpAngn.cpp:182-232; the wide type skips rjk), branch free.
template <typename R, typename V4>
__device__ __forceinline__ bool pair_in_range(V4 const& pj, V4 const& pk,
                                              bool wide, R rc, R rc2)
{
    R const dx = pk.x - pj.x;
    R const dy = pk.y - pj.y;
    R const dz = pk.z - pj.z;
    R const d2 = dx * dx + dy * dy + dz * dz;
    return (pj.w < rc) & (pk.w < rc) & (wide | (d2 < rc2));
}

// The model-specialised build says which angular types there are: 0 none of
// the wide type, 1 only it, 2 both.
#ifndef HDNNP_WIDE
#define HDNNP_WIDE 2
#endif

// Keeps a value that was read from LDS with others in that one wide read: the
// compiler otherwise splits it and reads the components that only a later
// branch needs there, with 16-byte strides that collide in the banks.
template <typename R>
__device__ __forceinline__ void read_whole(R& x)
{
    asm volatile("" : "+v"(x));
}

// Queue of a PairWalk: fewer than 64 entries when a step of 256 pairs starts,
// and one that takes what is not queued.
constexpr int kPairQueue = 64 + 256;
constexpr int kPairQueueAlloc = kPairQueue + 4;

typedef float Float4V __attribute__((ext_vector_type(4)));

// Position of staged neighbour t in FP32 and half its negative square,
// (x, y, z, -r^2 / 2), as the pair search reads it; minus infinity in place of
// the square keeps the neighbour out (r >= rc) wherever it is: the sum is that
// or NaN, also where products of coordinates overflow.  FP64 records are
// rounded as they are read: a float copy beside them cost 16 of 64 bytes of LDS
// per neighbour and with it workgroups per CU (196,608 water atoms 9,790 ->
// 9,510 us; 8,000 atoms of 366 neighbours, symmetry functions 2,530 -> 2,340
// and force 4,500 -> 3,710 us).
constexpr float kOutside = -__builtin_inff();

template <typename R>
__device__ __forceinline__ Float4V search_row(Vec4<R> const* P, R rc, int t)
{
    Vec4<R> const p = P[t];
    float const r = (float)p.w;
    return Float4V{(float)p.x, (float)p.y, (float)p.z,
                   p.w < rc ? -0.5f * (r * r) : kOutside};
}

// The pairs {j, k} of a group's neighbour blocks that can pass rij, rik < rc
// and rjk < rc (narrow types), 64 at a time in diagonal order.
//
// Narrow: the search for rjk < rc is a matrix product.  With h = -r^2 / 2,
// x_j x_k + y_j y_k + z_j z_k + h_j + h_k = -rjk^2 / 2, so five 4x4x1 MFMA
// steps over 16 independent blocks give the distances of 16 blocks of 4 x 4
// neighbours, 256 pairs, in 40 cycles of the matrix cores; the vector ALU
// only compares (4) and appends the hits to the queue.  The blocks of 4 are
// walked as DiagPairs walks single neighbours, and the four hits masks of a
// step are recombined so that the 64 pairs of one append have 64 different j
// and 64 different k (the force kernel's LDS adds collide on equal slots).
// The distances are FP32 with an error below 2e-6 rc^2 (15 roundings of terms
// up to 1.5 rc^2, h and, on the FP64 path, the rounded positions included),
// so pairs up to 8e-6 rc^2 beyond are let through and the evaluation takes
// f_c(rjk) = 0 for those (rij, rik < rc hold exactly: h).  One neighbour pair
// per lane and step (differences, squares, index arithmetic and queue: 37
// vector instructions per 64 pairs instead of about 12) made the search 40% of
// the symmetry-function kernel.
//
// Wide: no distance to search; if every neighbour of the list is inside rc
// (direct) the pairs go to the lanes as they come, else through the queue.
template <typename R>
struct PairWalk
{
    DiagPairs dp;         // neighbours (wide) or blocks of four (narrow)
    Vec4<R> const* P;
    int* Q;
    R rc;
    float thr;
    int s0, e0, l0, e1;   // first and last neighbour of each side
    int base, qn, c, r;
    bool wide, direct;

    __device__ __forceinline__ PairWalk(bool wide_, bool allIn, bool same,
                                        int a0, int na, int b0, int nb,
                                        Vec4<R> const* P_, int* Q_, R rc_,
                                        R rc2)
        : dp(same, a0, na, b0, nb), P(P_), Q(Q_), rc(rc_),
          thr(-0.5f * (1.0f + 8e-6f) * (float)rc2), base(0), qn(0), c(0),
          r(0), wide(wide_), direct(wide_ && allIn)
    {
        s0 = dp.s0;
        l0 = dp.l0;
        e0 = s0 + dp.ns - 1;
        e1 = l0 + dp.nl - 1;
        if (!wide)
        {
            // Blocks of four: the same order with the diagonal (blocks with
            // themselves) first.
            int const nbs = (dp.ns + 3) >> 2, nbl = (dp.nl + 3) >> 2;
            dp.d = nbs;
            dp.nl = nbl;
            dp.npairs = dp.npairs == 0 ? 0
                      : same ? nbs * (nbs + 1) / 2 : nbs * nbl;
            dp.q64 = nbs > 0 ? 16 / nbs : 0;
            dp.r64 = 16 - dp.q64 * nbs;
            dp.start(lane_id() >> 2, c, r);
        }
        else dp.start(lane_id(), c, r);
    }

    // 256 pairs of the narrow search.
    __device__ __forceinline__ void search()
    {
        int const lane = lane_id(), j = lane & 3;
        bool const valid = base + (lane >> 2) < dp.npairs;
        int v = r + c;
        if (v >= dp.nl) v -= dp.nl;
        int const ja = s0 + 4 * r, kb = l0 + 4 * v + j;
        // Beyond the end (also of the pairs): a neighbour in bounds, kept out.
        Float4V A = search_row(P, rc, min(ja + j, e0));
        Float4V B = search_row(P, rc, min(kb, e1));
        if (ja + j > e0) A.w = kOutside;
        if (kb > e1 || !valid) B.w = kOutside;
        Float4V d = {0.0f, 0.0f, 0.0f, 0.0f};
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(A.x, B.x, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(A.y, B.y, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(A.z, B.z, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(A.w, 1.0f, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_4x4x1f32(1.0f, B.w, d, 0, 0, 0);
        // d[i]: neighbour i of the first block, j of the second.  Rotated by
        // j, so that d[s] is the pair (i = (j + s) mod 4, j).
        bool const j1 = (j & 1) != 0, j2 = (j & 2) != 0;
        float const t0 = j1 ? d[1] : d[0], t1 = j1 ? d[2] : d[1],
                    t2 = j1 ? d[3] : d[2], t3 = j1 ? d[0] : d[3];
        float p[4] = {j2 ? t2 : t0, j2 ? t3 : t1, j2 ? t0 : t2, j2 ? t1 : t3};
        if (dp.same && base < dp.d)
        {
            // Blocks with themselves: i < j only, the s with j + s >= 4.
            int const first = c == 0 ? 4 - j : 0;
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (s < first) p[s] = kOutside;
        }
        int const code = ja | (kb << 16);
#pragma unroll
        for (int s = 0; s < 4; ++s)
        {
            uint64_t const hit = __ballot(p[s] > thr);
            // The others write behind the queue.
            int const at = __builtin_amdgcn_mbcnt_hi(
                (uint32_t)(hit >> 32),
                __builtin_amdgcn_mbcnt_lo((uint32_t)hit, qn));
            Q[p[s] > thr ? at : kPairQueue] = code + ((j + s) & 3);
            qn += __popcll(hit);
        }
        base += 16;
        dp.advance(c, r);
    }

    // 64 pairs of a wide group with neighbours beyond rc.
    __device__ __forceinline__ void filter()
    {
        bool const valid = base + lane_id() < dp.npairs;
        int j, k;
        dp.pair(c, r, j, k);
        if (!valid) j = k = dp.s0;
        bool const pass = valid & (P[j].w < rc) & (P[k].w < rc);
        uint64_t const hit = __ballot(pass);
        if (pass) Q[qn + lanes_below(hit)] = j | (k << 16);
        qn += __popcll(hit);
        base += 64;
        dp.advance(c, r);
    }

    // Calls f(e, count) for the pairs in turn: e = j | k << 16 in the first
    // `count` lanes.
    template <typename F>
    __device__ __forceinline__ void run(F const& f)
    {
        if (HDNNP_WIDE > 0 && direct)
        {
            for (; base < dp.npairs; base += 64)
            {
                int j, k;
                dp.pair(c, r, j, k);
                dp.advance(c, r);
                f(j | (k << 16), min(64, dp.npairs - base));
            }
            return;
        }
        for (;;)
        {
            while (qn < 64 && base < dp.npairs)
            {
                if (HDNNP_WIDE == 0 || (HDNNP_WIDE == 2 && !wide)) search();
                else filter();
            }
            int const count = min(64, qn);
            if (count == 0) return;
            wave_lds_fence();
            qn -= count;
            int const e = Q[qn + lane_id()];
            wave_lds_fence();
            f(e, count);
        }
    }
};

// Sums M per-lane values over the wave through LDS (M x 64 values at `s`,
// 16-byte aligned): lane l adds M of the 64 values of member l / (64 / M),
// in FP64, and a butterfly over the 64 / M lanes of a member follows.  Every
// lane of member m's lanes returns its total; the order of the additions is
// fixed.  About 35 vector instructions for 8 members; exchanging FP64 values
// between lanes register by register takes about 250.
template <int M, typename R>
__device__ __forceinline__ double wave_sum_members(R const (&v)[M], R* s)
{
    static_assert(M == 4 || M == 8 || M == 16, "4, 8 or 16 members");
    constexpr int kLanes = 64 / M, kVec = 16 / sizeof(R);
    int const lane = lane_id();
    wave_lds_fence();
#pragma unroll
    for (int m = 0; m < M; ++m) s[64 * m + lane] = v[m];
    wave_lds_fence();
    typedef R V __attribute__((ext_vector_type(16 / sizeof(R))));
    V const* row = (V const*)(s + 64 * (lane / kLanes)) + lane % kLanes;
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < M / kVec; ++q)
    {
        V const x = row[q * kLanes];
#pragma unroll
        for (int u = 0; u < kVec; ++u) t += (double)x[u];
    }
    wave_lds_fence();
#pragma unroll
    for (int o = 1; o < kLanes; o <<= 1) t += __shfl_xor(t, o, kWave);
    return t;
}

// Weight of staged neighbour t for the weighted SF types: the atomic number
// of the element block (neighbours staged partitioned by element) that
// holds it.
__device__ __forceinline__ double staged_weight(ModelTables const& T,
                                                int const* sStart,
                                                int const* sCnt, int t)
{
    double w = 0.0;
#pragma unroll
    for (int q = 0; q < kMaxElements; ++q)
        if (q < T.ne && t >= sStart[q] && t < sStart[q] + sCnt[q])
            w = T.zw[q];
    return w;
}

}  // namespace hdnnp

#endif
