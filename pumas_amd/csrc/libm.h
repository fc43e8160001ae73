/*
 * Math functions of the transport engine, rounding exactly as the host C
 * library the reference is built against (GNU C library 2.35, x86-64).
 *
 * Per-history parity of a stochastic path needs every transcendental
 * function to return the bits the reference's libm returns: a last-bit
 * difference in one log or cos moves a history by ~1e-16, and a few of
 * them, amplified along a thousand steps or flipping a comparison, move
 * it beyond 1e-12. The device libraries (OCML) are accurate to about one
 * ulp but round differently, so the engine calls these functions instead.
 * They restate published algorithms:
 *
 *  - exp, log, pow, expf, logf: the table driven methods of Szabolcs
 *    Nagy's ARM Optimized Routines (as shipped in glibc 2.28+), in the
 *    variant glibc selects on x86-64 CPUs with FMA: every multiply-add the
 *    compiler contracts there is an explicit fma() here.
 *  - sin, cos: the IBM Accurate Mathematical Library (glibc
 *    sysdeps/ieee754/dbl-64/s_sin.c after the 2018 rewrite), also in its
 *    FMA variant; sincos: the same algorithm without FMA (glibc builds
 *    sincos without the FMA variant). gcc turns sin(x) and cos(x) of one
 *    argument into one sincos(x) call, so the engine calls sincos where
 *    the reference computes both.
 *  - log10: the fdlibm method of glibc (k log10(2) + log(x) / ln 10).
 *
 * Tables are in libm_tables.h (generated by libm/gen_tables.py). Arguments
 * beyond the transport's range (|x| >= 2^26.65 for sin/cos, where the
 * reference's library switches to a multi-word reduction) fall back to the
 * platform's function.
 *
 * Checks: logf and expf agree with the host library on all 2^32 inputs;
 * exp, log, pow, sin, cos, sincos on >= 1e8 random arguments each over
 * their whole ranges (tests/test_libm.py on the CPU build, and the GPU
 * build against the host library in tests/test_gpu_libm.py).
 */
#ifndef PUMAS_LIBM_H
#define PUMAS_LIBM_H

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define LM_FN __device__ __forceinline__
#define LM_TABLE static __constant__ const
#else
#include <math.h>
#define LM_FN inline
#define LM_TABLE static const
#endif

#include "libm_tables.h"

namespace pg {
namespace lm {

LM_FN uint64_t asu64(double x) { return __builtin_bit_cast(uint64_t, x); }
LM_FN double asd(uint64_t u) { return __builtin_bit_cast(double, u); }
LM_FN uint32_t asu32(float x) { return __builtin_bit_cast(uint32_t, x); }
LM_FN float asf(uint32_t u) { return __builtin_bit_cast(float, u); }
LM_FN double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
LM_FN double fabs_(double x) { return __builtin_fabs(x); }
LM_FN double copysign_(double x, double y) { return __builtin_copysign(x, y); }

constexpr double INF = __builtin_inf();

/* ------------------------------------------------------------------------
 * exp (ARM Optimized Routines exp.c, N = 128, order 5 polynomial).
 * ------------------------------------------------------------------------ */
constexpr double EXP_INVLN2N = 0x1.71547652b82fep0 * 128;
constexpr double EXP_NEGLN2HIN = -0x1.62e42fefa0000p-8;
constexpr double EXP_NEGLN2LON = -0x1.cf79abc9e3b3ap-47;
constexpr double EXP_SHIFT = 0x1.8p52;
constexpr double EXP_C2 = 0x1.ffffffffffdbdp-2;
constexpr double EXP_C3 = 0x1.555555555543cp-3;
constexpr double EXP_C4 = 0x1.55555cf172b91p-5;
constexpr double EXP_C5 = 0x1.1111167a4d017p-7;

/* |x| > 512 or so: scale in two steps (k > 0) or round before scaling
 * into the subnormal range (k < 0). */
LM_FN double exp_special(double tmp, uint64_t sbits, uint64_t ki)
{
        if ((ki & 0x80000000) == 0) {
                sbits -= 1009ull << 52;
                const double scale = asd(sbits);
                return 0x1p1009 * fma_(scale, tmp, scale);
        }
        sbits += 1022ull << 52;
        const double scale = asd(sbits);
        /* Not contracted in the reference build: the product has a second
         * use in another block. */
        const double st = scale * tmp;
        double y = scale + st;
        if (fabs_(y) < 1.0) {
                const double one = (y < 0.0) ? -1.0 : 1.0;
                double lo = scale - y + st;
                const double hi = one + y;
                lo = one - hi + y + lo;
                y = (hi + lo) - one;
                if (y == 0.0) y = asd(sbits & 0x8000000000000000ull);
        }
        return 0x1p-1022 * y;
}

/* exp(x + xtail) with the sign of sign_bias, the common kernel of exp and
 * pow. `top12(x)` outside [2^-54, 512) is handled here. */
LM_FN double exp_kernel(double x, double xtail, uint64_t sign_bias,
    bool from_pow)
{
        uint32_t abstop = (uint32_t)(asu64(x) >> 52) & 0x7ff;
        if (abstop - 0x3c9u >= 0x408u - 0x3c9u) {
                if ((int32_t)(abstop - 0x3c9u) < 0) {
                        const double one = 1.0 + x;
                        return sign_bias ? -one : one;
                }
                if (abstop >= 0x409u) {
                        if (!from_pow) {
                                if (asu64(x) == asu64(-INF)) return 0.0;
                                if (abstop >= 0x7ffu) return 1.0 + x;
                        }
                        if (asu64(x) >> 63)
                                return sign_bias ? -0.0 : 0.0;
                        return sign_bias ? -INF : INF;
                }
                abstop = 0;
        }
        double kd = fma_(EXP_INVLN2N, x, EXP_SHIFT);
        const uint64_t ki = asu64(kd);
        kd -= EXP_SHIFT;
        double r = fma_(kd, EXP_NEGLN2LON, fma_(kd, EXP_NEGLN2HIN, x));
        if (from_pow) r += xtail;
        const uint64_t idx = 2 * (ki % 128);
        const uint64_t top = (ki + sign_bias) << 45;
        const double tail = asd(EXP_TAB[idx]);
        const uint64_t sbits = EXP_TAB[idx + 1] + top;
        const double r2 = r * r;
        const double tmp = fma_(r2 * r2, fma_(r, EXP_C5, EXP_C4),
            fma_(r2, fma_(r, EXP_C3, EXP_C2), tail + r));
        if (abstop == 0) return exp_special(tmp, sbits, ki);
        const double scale = asd(sbits);
        return fma_(scale, tmp, scale);
}

LM_FN double exp(double x) { return exp_kernel(x, 0.0, 0, false); }

/* ------------------------------------------------------------------------
 * log (ARM Optimized Routines log.c, N = 128; order 12 polynomial near 1).
 * ------------------------------------------------------------------------ */
constexpr double LN2HI = 0x1.62e42fefa3800p-1;
constexpr double LN2LO = 0x1.ef35793c76730p-45;

LM_FN double log(double x)
{
        constexpr double A0 = -0x1.0000000000001p-1, A1 = 0x1.555555551305bp-2,
                         A2 = -0x1.fffffffeb459p-3, A3 = 0x1.999b324f10111p-3,
                         A4 = -0x1.55575e506c89fp-3;
        constexpr double B0 = -0x1p-1, B1 = 0x1.5555555555577p-2,
                         B2 = -0x1.ffffffffffdcbp-3, B3 = 0x1.999999995dd0cp-3,
                         B4 = -0x1.55555556745a7p-3, B5 = 0x1.24924a344de3p-3,
                         B6 = -0x1.fffffa4423d65p-4, B7 = 0x1.c7184282ad6cap-4,
                         B8 = -0x1.999eb43b068ffp-4, B9 = 0x1.78182f7afd085p-4,
                         B10 = -0x1.5521375d145cdp-4;
        uint64_t ix = asu64(x);
        const uint32_t top = (uint32_t)(ix >> 48);
        constexpr uint64_t LO = 0x3fee000000000000ull; /* 1 - 2^-4 */
        constexpr uint64_t HI = 0x3ff1090000000000ull; /* 1 + 0x1.09p-4 */
        if (ix - LO < HI - LO) {
                if (ix == 0x3ff0000000000000ull) return 0;
                const double r = x - 1.0, r2 = r * r, r3 = r * r2;
                const double p3 = fma_(r3, B10, fma_(r2, B9, fma_(r, B8, B7)));
                const double p2 = fma_(r3, p3, fma_(r2, B6, fma_(r, B5, B4)));
                const double p1 = fma_(r3, p2, fma_(r2, B3, fma_(r, B2, B1)));
                double w = r * 0x1p27;
                const double rhi = r + w - w;
                const double rlo = r - rhi;
                w = rhi * rhi * B0;
                const double hi = r + w;
                double lo = r - hi + w;
                lo = fma_(B0 * rlo, rhi + r, lo);
                return fma_(r3, p1, lo) + hi;
        }
        if (top - 0x0010u >= 0x7ff0u - 0x0010u) {
                if (ix * 2 == 0) return -INF;
                if (ix == 0x7ff0000000000000ull) return x;
                if ((top & 0x8000) || (top & 0x7ff0) == 0x7ff0)
                        return __builtin_nan("");
                ix = asu64(x * 0x1p52);
                ix -= 52ull << 52;
        }
        const uint64_t tmp = ix - 0x3fe6000000000000ull;
        const int i = (int)((tmp >> 45) % 128);
        const int k = (int)((int64_t)tmp >> 52);
        const uint64_t iz = ix - (tmp & (0xfffull << 52));
        const double invc = LOG_TAB[i][0], logc = LOG_TAB[i][1];
        const double z = asd(iz);
        const double r = fma_(z, invc, -1.0);
        const double kd = (double)k;
        const double w = fma_(kd, LN2HI, logc);
        const double hi = w + r;
        const double lo = fma_(kd, LN2LO, w - hi + r);
        const double r2 = r * r;
        const double p = fma_(r2, fma_(r, A4, A3), fma_(r, A2, A1));
        return fma_(r * r2, p, fma_(r2, A0, lo)) + hi;
}

/* log10 (glibc e_log10.c, fdlibm; not contracted in the reference's
 * build). */
LM_FN double log10(double x)
{
        constexpr double TWO54 = 1.80143985094819840000e+16;
        constexpr double IVLN10 = 4.34294481903251816668e-01;
        constexpr double LOG10_2HI = 3.01029995663611771306e-01;
        constexpr double LOG10_2LO = 3.69423907715893078616e-13;
        uint64_t ix = asu64(x);
        int32_t hx = (int32_t)(ix >> 32);
        int32_t k = 0;
        if (hx < 0x00100000) {
                if (((hx & 0x7fffffff) | (uint32_t)ix) == 0)
                        return -INF;
                if (hx < 0) return __builtin_nan("");
                k -= 54;
                x *= TWO54;
                ix = asu64(x);
                hx = (int32_t)(ix >> 32);
        }
        if (hx >= 0x7ff00000) return x + x;
        k += (hx >> 20) - 1023;
        const int32_t i = (int32_t)(((uint32_t)k & 0x80000000u) >> 31);
        hx = (hx & 0x000fffff) | ((0x3ff - i) << 20);
        const double y = (double)(k + i);
        x = asd(((uint64_t)(uint32_t)hx << 32) | (uint32_t)ix);
        const double z = y * LOG10_2LO + IVLN10 * lm::log(x);
        return z + y * LOG10_2HI;
}

/* ------------------------------------------------------------------------
 * pow (ARM Optimized Routines pow.c: log with a 128 bit result, then exp).
 * ------------------------------------------------------------------------ */
LM_FN double pow_log(uint64_t ix, double * tail)
{
        constexpr double P0 = -0x1p-1, P1 = 0x1.555555555556p-2 * -2,
                         P2 = -0x1.0000000000006p-2 * -2,
                         P3 = 0x1.999999959554ep-3 * 4,
                         P4 = -0x1.555555529a47ap-3 * 4,
                         P5 = 0x1.2495b9b4845e9p-3 * -8,
                         P6 = -0x1.0002b8b263fc3p-3 * -8;
        const uint64_t tmp = ix - 0x3fe6955500000000ull;
        const int i = (int)((tmp >> 45) % 128);
        const int k = (int)((int64_t)tmp >> 52);
        const uint64_t iz = ix - (tmp & (0xfffull << 52));
        const double z = asd(iz), kd = (double)k;
        const double invc = POW_LOG_TAB[i][0], logc = POW_LOG_TAB[i][1],
                     logctail = POW_LOG_TAB[i][2];
        const double r = fma_(z, invc, -1.0);
        const double t1 = fma_(kd, LN2HI, logc);
        const double t2 = t1 + r;
        const double lo1 = fma_(kd, LN2LO, logctail);
        const double lo2 = t1 - t2 + r;
        const double ar = P0 * r, ar2 = r * ar, ar3 = r * ar2;
        const double hi = t2 + ar2;
        const double lo3 = fma_(ar, r, -ar2);
        const double lo4 = t2 - hi + ar2;
        const double q = fma_(ar2, fma_(ar2, fma_(r, P6, P5), fma_(r, P4, P3)),
            fma_(r, P2, P1));
        const double lo = fma_(ar3, q, lo1 + lo2 + lo3 + lo4);
        const double y = hi + lo;
        *tail = hi - y + lo;
        return y;
}

/* 0: not an integer, 1: odd integer, 2: even integer. */
LM_FN int pow_checkint(uint64_t iy)
{
        const int e = (int)(iy >> 52 & 0x7ff);
        if (e < 0x3ff) return 0;
        if (e > 0x3ff + 52) return 2;
        if (iy & ((1ull << (0x3ff + 52 - e)) - 1)) return 0;
        if (iy & (1ull << (0x3ff + 52 - e))) return 1;
        return 2;
}

LM_FN bool pow_zeroinfnan(uint64_t i)
{
        return 2 * i - 1 >= 2 * 0x7ff0000000000000ull - 1;
}

LM_FN double pow(double x, double y)
{
        constexpr uint64_t SIGN_BIAS = 0x800ull << 7;
        constexpr uint64_t ONE = 0x3ff0000000000000ull;
        constexpr uint64_t PINF = 0x7ff0000000000000ull;
        uint64_t sign_bias = 0;
        uint64_t ix = asu64(x);
        const uint64_t iy = asu64(y);
        uint32_t topx = (uint32_t)(ix >> 52);
        const uint32_t topy = (uint32_t)(iy >> 52);
        if (topx - 0x001u >= 0x7ffu - 0x001u ||
            (topy & 0x7ff) - 0x3beu >= 0x43eu - 0x3beu) {
                if (pow_zeroinfnan(iy)) {
                        if (2 * iy == 0) return 1.0;
                        if (ix == ONE) return 1.0;
                        if (2 * ix > 2 * PINF || 2 * iy > 2 * PINF)
                                return x + y;
                        if (2 * ix == 2 * ONE) return 1.0;
                        if ((2 * ix < 2 * ONE) == !(iy >> 63)) return 0.0;
                        return y * y;
                }
                if (pow_zeroinfnan(ix)) {
                        double x2 = x * x;
                        if ((ix >> 63) && pow_checkint(iy) == 1) x2 = -x2;
                        return (iy >> 63) ? 1 / x2 : x2;
                }
                if (ix >> 63) {
                        const int yint = pow_checkint(iy);
                        if (yint == 0) return __builtin_nan("");
                        if (yint == 1) sign_bias = SIGN_BIAS;
                        ix &= 0x7fffffffffffffffull;
                        topx &= 0x7ff;
                }
                if ((topy & 0x7ff) - 0x3beu >= 0x43eu - 0x3beu) {
                        if (ix == ONE) return 1.0;
                        if ((topy & 0x7ff) < 0x3be)
                                return (ix > ONE) ? 1.0 + y : 1.0 - y;
                        return ((ix > ONE) == (topy < 0x800)) ? INF : 0.0;
                }
                if (topx == 0) {
                        ix = asu64(x * 0x1p52);
                        ix &= 0x7fffffffffffffffull;
                        ix -= 52ull << 52;
                }
        }
        double lo;
        const double hi = pow_log(ix, &lo);
        const double ehi = y * hi;
        const double elo = fma_(y, lo, fma_(y, hi, -ehi));
        return exp_kernel(ehi, elo, sign_bias, true);
}

/* ------------------------------------------------------------------------
 * sin, cos, sincos (IBM Accurate Mathematical Library, glibc s_sin.c).
 * ------------------------------------------------------------------------ */
constexpr double SC_S1 = -0x1.5555555555555p-3, SC_S2 = 0x1.1111111110ECEp-7,
                 SC_S3 = -0.00019841269834414642,
                 SC_S4 = 0x1.71DE27B9A7ED9p-19,
                 SC_S5 = -0x1.ADDFFC2FCDF59p-26;
constexpr double SC_SN3 = -1.66666666666664880952546298448555E-01,
                 SC_SN5 = 8.33333214285722277379541354343671E-03,
                 SC_CS2 = 4.99999999999999999999950396842453E-01,
                 SC_CS4 = -4.16666666666664434524222570944589E-02,
                 SC_CS6 = 1.38888874007937613028114285595617E-03;
constexpr double SC_BIG = 0x1.8p45, SC_HP0 = 0x1.921FB54442D18p0,
                 SC_HP1 = 0x1.1A62633145C07p-54,
                 SC_MP1 = 0x1.921FB58000000p0, SC_MP2 = -0x1.DDE973C000000p-27,
                 SC_PP3 = -0x1.CB3B398000000p-55,
                 SC_PP4 = -0x1.d747f23e32ed7p-83,
                 SC_HPINV = 0x1.45F306DC9C883p-1, SC_TOINT = 0x1.8p52;

/* FUSED: the FMA variant (sin, cos) or the plain one (sincos). */
template <bool FUSED>
LM_FN double sc_mad(double a, double b, double c)
{
        if (FUSED) return fma_(a, b, c);
        return a * b + c;
}

/* sin(x + dx) for |x| <= 0.855469: Taylor series below 0.126, else a
 * table point k/128 and short series for the remainder. */
template <bool FUSED>
LM_FN double sc_do_sin(double x, double dx)
{
        const double xold = x;
        if (fabs_(x) < 0.126) {
                const double xx = x * x;
                double p;
                if (FUSED) {
                        p = fma_(fma_(fma_(fma_(SC_S5, xx, SC_S4), xx, SC_S3),
                                     xx, SC_S2),
                            xx, SC_S1);
                        const double t = fma_(fma_(p, x, -(0.5 * dx)), xx, dx);
                        return x + t;
                }
                p = (((SC_S5 * xx + SC_S4) * xx + SC_S3) * xx + SC_S2) * xx +
                    SC_S1;
                const double t = (p * x - 0.5 * dx) * xx + dx;
                return x + t;
        }
        if (x <= 0) dx = -dx;
        const double u = SC_BIG + fabs_(x);
        x = fabs_(x) - (u - SC_BIG);
        const double xx = x * x;
        double s, c, cor;
        const int k = (int)((uint32_t)asu64(u) << 2);
        const double sn = SINCOS_TAB[k], ssn = SINCOS_TAB[k + 1],
                     cs = SINCOS_TAB[k + 2], ccs = SINCOS_TAB[k + 3];
        if (FUSED) {
                s = x + fma_(x * xx, fma_(xx, SC_SN5, SC_SN3), dx);
                c = fma_(x, dx,
                    xx * fma_(xx, fma_(xx, SC_CS6, SC_CS4), SC_CS2));
                cor = fma_(cs, s, fma_(-sn, c, fma_(s, ccs, ssn)));
        } else {
                s = x + (dx + x * xx * (SC_SN3 + xx * SC_SN5));
                c = x * dx + xx * (SC_CS2 + xx * (SC_CS4 + xx * SC_CS6));
                cor = (ssn + s * ccs - sn * c) + cs * s;
        }
        return copysign_(sn + cor, xold);
}

/* cos(x + dx) for |x| <= 0.855469. */
template <bool FUSED>
LM_FN double sc_do_cos(double x, double dx)
{
        if (x < 0) dx = -dx;
        const double u = SC_BIG + fabs_(x);
        x = fabs_(x) - (u - SC_BIG) + dx;
        const double xx = x * x;
        const int k = (int)((uint32_t)asu64(u) << 2);
        const double sn = SINCOS_TAB[k], ssn = SINCOS_TAB[k + 1],
                     cs = SINCOS_TAB[k + 2], ccs = SINCOS_TAB[k + 3];
        double s, c, cor;
        if (FUSED) {
                s = fma_(x * xx, fma_(xx, SC_SN5, SC_SN3), x);
                c = xx * fma_(xx, fma_(xx, SC_CS6, SC_CS4), SC_CS2);
                cor = fma_(-sn, s, fma_(-cs, c, fma_(-s, ssn, ccs)));
        } else {
                s = x + x * xx * (SC_SN3 + xx * SC_SN5);
                c = xx * (SC_CS2 + xx * (SC_CS4 + xx * SC_CS6));
                cor = (ccs - s * ssn - cs * c) - sn * s;
        }
        return cs + cor;
}

/* x = n pi/2 + (a + da), |a| <= pi/4, for |x| < 105414350. */
template <bool FUSED>
LM_FN int sc_reduce(double x, double * a, double * da)
{
        double t, xn, y, t2, db, b;
        if (FUSED) {
                t = fma_(x, SC_HPINV, SC_TOINT);
                xn = t - SC_TOINT;
                y = fma_(-xn, SC_MP2, fma_(-xn, SC_MP1, x));
                t2 = fma_(-xn, SC_PP3, y);
                db = fma_(-xn, SC_PP3, y - t2);
                b = fma_(-xn, SC_PP4, t2);
                db += fma_(-xn, SC_PP4, t2 - b);
        } else {
                t = x * SC_HPINV + SC_TOINT;
                xn = t - SC_TOINT;
                y = (x - xn * SC_MP1) - xn * SC_MP2;
                double t1 = xn * SC_PP3;
                t2 = y - t1;
                db = (y - t2) - t1;
                t1 = xn * SC_PP4;
                b = t2 - t1;
                db += (t2 - b) - t1;
        }
        *a = b;
        *da = db;
        return (int)((uint32_t)asu64(t) & 3);
}

template <bool FUSED>
LM_FN double sc_do_sincos(double a, double da, int n)
{
        const double r = (n & 1) ? sc_do_cos<FUSED>(a, da) :
                                   sc_do_sin<FUSED>(a, da);
        return (n & 2) ? -r : r;
}

/* Beyond the simple reduction: the platform's function. */
LM_FN double sin_far(double x) { return ::sin(x); }
LM_FN double cos_far(double x) { return ::cos(x); }

LM_FN double sin(double x)
{
        const uint32_t k = (uint32_t)(asu64(x) >> 32) & 0x7fffffff;
        if (k < 0x3e500000) return x;
        if (k < 0x3feb6000) return sc_do_sin<true>(x, 0);
        if (k < 0x400368fd) {
                const double t = SC_HP0 - fabs_(x);
                return copysign_(sc_do_cos<true>(t, SC_HP1), x);
        }
        if (k < 0x419921FB) {
                double a, da;
                const int n = sc_reduce<true>(x, &a, &da);
                return sc_do_sincos<true>(a, da, n);
        }
        return sin_far(x);
}

LM_FN double cos(double x)
{
        const uint32_t k = (uint32_t)(asu64(x) >> 32) & 0x7fffffff;
        if (k < 0x3e400000) return 1.0;
        if (k < 0x3feb6000) return sc_do_cos<true>(x, 0);
        if (k < 0x400368fd) {
                const double y = SC_HP0 - fabs_(x);
                const double a = y + SC_HP1;
                const double da = (y - a) + SC_HP1;
                return sc_do_sin<true>(a, da);
        }
        if (k < 0x419921FB) {
                double a, da;
                const int n = sc_reduce<true>(x, &a, &da);
                return sc_do_sincos<true>(a, da, n + 1);
        }
        return cos_far(x);
}

/*
 * The three argument ranges of glibc's sincos (below 0.855469, below
 * 2.426265, below 105414350) differ in their reduction only: each then
 * evaluates sc_do_sin and sc_do_cos once on its reduced argument and assigns
 * them, swapped and negated by range and quadrant. The reduction of every
 * range is computed and selected first, so that lanes of a wavefront in
 * different ranges evaluate the two series together instead of once per
 * range; each lane's operations are those of its range.
 */
LM_FN void sincos_near(double x, double * sx, double * cx)
{
        const uint32_t k = (uint32_t)(asu64(x) >> 32) & 0x7fffffff;
        if (k < 0x3e400000) {
                *sx = x;
                *cx = 1.0;
                return;
        }
        /* Range 2: pi/2 - |x|. */
        const double y = SC_HP0 - fabs_(x);
        const double a2 = y + SC_HP1;
        const double da2 = (y - a2) + SC_HP1;
        /* Range 3: x = n pi/2 + a. */
        double a3, da3;
        const int n = sc_reduce<false>(x, &a3, &da3);
        const bool r1 = k < 0x3feb6000;
        const bool r2 = !r1 && (k < 0x400368fd);
        const double a = r1 ? x : (r2 ? a2 : a3);
        const double da = r1 ? 0. : (r2 ? da2 : da3);
        const double s = sc_do_sin<false>(a, da);
        const double c = sc_do_cos<false>(a, da);
        if (r1) {
                *sx = s;
                *cx = c;
        } else if (r2) {
                *sx = copysign_(c, x);
                *cx = s;
        } else {
                const double rs = (n & 1) ? c : s;
                const double rc = (n & 1) ? s : c;
                *sx = (n & 2) ? -rs : rs;
                *cx = ((n + 1) & 2) ? -rc : rc;
        }
}

/* Any argument (sincos_near: |x| < 105414350, the reductions above). */
LM_FN void sincos(double x, double * sx, double * cx)
{
        const uint32_t k = (uint32_t)(asu64(x) >> 32) & 0x7fffffff;
        if (k >= 0x419921FB) {
                *sx = sin_far(x);
                *cx = cos_far(x);
                return;
        }
        sincos_near(x, sx, cx);
}

/* ------------------------------------------------------------------------
 * logf, expf (ARM Optimized Routines logf.c, expf.c).
 * ------------------------------------------------------------------------ */
/* {1/c, log(c)} for 16 subintervals of [0x1.66p-1, 0x1.66p0). */
LM_TABLE double LOGF_TAB[16][2] = {
        { 0x1.661ec79f8f3bep+0, -0x1.57bf7808caadep-2 },
        { 0x1.571ed4aaf883dp+0, -0x1.2bef0a7c06ddbp-2 },
        { 0x1.49539f0f010bp+0, -0x1.01eae7f513a67p-2 },
        { 0x1.3c995b0b80385p+0, -0x1.b31d8a68224e9p-3 },
        { 0x1.30d190c8864a5p+0, -0x1.6574f0ac07758p-3 },
        { 0x1.25e227b0b8eap+0, -0x1.1aa2bc79c81p-3 },
        { 0x1.1bb4a4a1a343fp+0, -0x1.a4e76ce8c0e5ep-4 },
        { 0x1.12358f08ae5bap+0, -0x1.1973c5a611cccp-4 },
        { 0x1.0953f419900a7p+0, -0x1.252f438e10c1ep-5 },
        { 0x1p+0, 0x0p+0 },
        { 0x1.e608cfd9a47acp-1, 0x1.aa5aa5df25984p-5 },
        { 0x1.ca4b31f026aap-1, 0x1.c5e53aa362eb4p-4 },
        { 0x1.b2036576afce6p-1, 0x1.526e57720db08p-3 },
        { 0x1.9c2d163a1aa2dp-1, 0x1.bc2860d22477p-3 },
        { 0x1.886e6037841edp-1, 0x1.1058bc8a07ee1p-2 },
        { 0x1.767dcf5534862p-1, 0x1.4043057b6ee09p-2 },
};

LM_FN float logf(float x)
{
        constexpr double LN2 = 0x1.62e42fefa39efp-1;
        constexpr double A0 = -0x1.00ea348b88334p-2, A1 = 0x1.5575b0be00b6ap-2,
                         A2 = -0x1.ffffef20a4123p-2;
        uint32_t ix = asu32(x);
        if (ix == 0x3f800000u) return 0.f;
        if (ix - 0x00800000u >= 0x7f800000u - 0x00800000u) {
                if (ix * 2 == 0) return -__builtin_inff();
                if (ix == 0x7f800000u) return x;
                if ((ix & 0x80000000u) || ix * 2 >= 0xff000000u)
                        return __builtin_nanf("");
                ix = asu32(x * 0x1p23f);
                ix -= 23u << 23;
        }
        const uint32_t tmp = ix - 0x3f330000u;
        const int i = (int)((tmp >> 19) % 16);
        const int k = (int32_t)tmp >> 23;
        const uint32_t iz = ix - (tmp & 0xff800000u);
        const double invc = LOGF_TAB[i][0], logc = LOGF_TAB[i][1];
        const double z = (double)asf(iz);
        const double r = fma_(z, invc, -1.0);
        const double y0 = fma_((double)k, LN2, logc);
        const double r2 = r * r;
        double y = fma_(A1, r, A2);
        y = fma_(A0, r2, y);
        y = fma_(y, r2, y0 + r);
        return (float)y;
}

LM_FN float expf(float x)
{
        constexpr double INVLN2N = 0x1.71547652b82fep+0 * 32;
        constexpr double SHIFT = 0x1.8p+52;
        constexpr double C0 = 0x1.c6af84b912394p-5 / 32 / 32 / 32,
                         C1 = 0x1.ebfce50fac4f3p-3 / 32 / 32,
                         C2 = 0x1.62e42ff0c52d6p-1 / 32;
        const double xd = (double)x;
        const uint32_t abstop = (asu32(x) >> 20) & 0x7ff;
        if (abstop >= 0x42bu) { /* |x| >= 88 or NaN */
                if (asu32(x) == 0xff800000u) return 0.f;
                if (abstop >= 0x7f8u) return x + x;
                if (x > 0x1.62e42ep6f) return __builtin_inff();
                if (x < -0x1.9fe368p6f) return 0.f;
        }
        double kd = fma_(INVLN2N, xd, SHIFT);
        const uint64_t ki = asu64(kd);
        kd -= SHIFT;
        const double r = fma_(INVLN2N, xd, -kd);
        uint64_t t = EXP2F_TAB[ki % 32];
        t += ki << 47;
        const double s = asd(t);
        const double z = fma_(C0, r, C1);
        const double r2 = r * r;
        double y = fma_(C2, r, 1.0);
        y = fma_(z, r2, y);
        y = y * s;
        return (float)y;
}

} /* namespace lm */
} /* namespace pg */

#endif
