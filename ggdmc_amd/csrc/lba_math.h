/*
 * LBA trial log-likelihood arithmetic for the HIP sampler.
 *
 * Reference semantics (external ggdmcHeaders/likelihood.h `sumloglike`, called
 * at src/de.cpp:145,187,604,653; per-trial floor R/phi.R:3-13): for a trial of
 * cell c with responding accumulator w and each accumulator j with
 * t = rt - t0_j > 0,
 *     zs = t*s, chi = b - t*v, z1 = chi/zs, z2 = (chi - A)/zs, den = max(Phi(v/s), 1e-10)
 *     pdf_j = (v*(Phi(z1)-Phi(z2)) + s*(phi(z2)-phi(z1))) / (A*den)
 *     F_j   = (1 + (zs*(phi(z2)-phi(z1)) + (chi-A)*Phi(z2) - chi*Phi(z1)) / A) / den
 *     density = max(pdf_w, 1e-10) * prod_{j != w} (1 - max(F_j, 1e-10))
 *     term = log(density > 0 ? density : DBL_EPSILON)
 * (t <= 0 gives pdf = F = 0.)
 *
 * Two evaluations are provided:
 *
 *  - `naive_*`: the formula above, term by term, in FP64 (the plain FP64 path).
 *
 *  - `mixed_*` / `*_factor`: the batched path, bound by the issue rate of the
 *    vector ALU. On CDNA4 every FP64 instruction (multiply-add, compare,
 *    convert, rndne, ldexp) measured 4.4 cycles per wave and SIMD, 32-bit
 *    integer and FP32 adds 2.8, v_rcp_f64 16.9 (v_rcp_f32 8.5 plus two
 *    conversions of 4.4 for its FP64 use), so the arithmetic stays FP64 and
 *    what counts is the number of instructions:
 *      * exp(-z^2/2) = 2^y, y = -z^2/2*log2(e): 2^n * 2^(j/64) (table) * 2^f
 *        (short polynomial), scaling and rounding folded into multiply-adds;
 *      * the accumulator's three reciprocals (1/zs and both tails' arguments)
 *        from one v_rcp_f64 and one Newton step (mixed_core);
 *      * Q(|z|) = exp(-z^2/2) * R(|z|), R the Mills-ratio factor
 *        Q(z)*exp(z^2/2), approximated as t*sum_k c_k t^k, k = 0..10, with
 *        t = 1/(1+0.2625|z|) (coefficients fitted for this library to
 *        0.5*erfcx(z/sqrt(2)) on [0, 14] by least squares reweighted toward
 *        the minimax relative error; max relative error 2.9e-10);
 *      * the small tail of Phi is always the one computed, so
 *        Phi(z1) - Phi(z2) is taken as Q(z2) - Q(z1) when z2 >= 0; where
 *        the reference's own FP64 value RN(1 - Q(z1)) - RN(1 - Q(z2)) could
 *        differ from that by more than the tolerance (the winner's far right
 *        tail), that rounded difference is reproduced from the computed
 *        tails whenever their error cannot move either rounding;
 *      * the survivor of a loser is formed from the complement 1 - G of the
 *        untruncated CDF (written without cancellation, see below) and then
 *        passed through the reference's own FP64 operations G = 1 + (G - 1),
 *        F = G/den, 1 - max(F, 1e-10). Where the reference's survivor is
 *        quantised by FP64 rounding (survivors of 1e-16 .. 1e-10 of sharp
 *        accumulators, whose F sits within a few ulps of 1), this reproduces
 *        the rounding itself, not just its scale; the DBL_EPSILON replacement
 *        and its sign rule follow from the same FP64 values. Phi follows R's
 *        pnorm: for z > 0 it is 1 - Q(z) rounded in FP64, Q the accurate
 *        upper tail;
 *      * each factor's error bound is first tested in a loose form of three
 *        or four instructions; the full bound (and the winner's rounding
 *        reproduction) is evaluated only by waves in which a trial fails it
 *        (6 of 60,000 simulated trials).
 *    The complement, with Phi2 = Phi(z2):
 *        1 - G = Phi2 + (chi*(Phi1 - Phi2) + zs*(phi1 - phi2)) / A
 *    (integrating the drift density over the start point: P(drift < (b - a)/t)
 *    averaged over a ~ U(0, A)).
 *    A trial's density is the reference's own FP64 product of the floored
 *    winner pdf and the survivors, in accumulator order; a lane takes one log
 *    of its two trials' product: log(x) = e*ln2 + log2(m)*ln2 with the FP32
 *    log2 applied to the mantissa only, so its error is absolute ~1e-8
 *    whatever the magnitude of log(x).
 *    Against two trials of 2 accumulators in about 720 vector instructions
 *    (both forms of G, a reciprocal and its seed conversions per quotient, the
 *    full error bound everywhere, a log per trial) this takes about 500: 33
 *    vectors x 100608 trials of 4 accumulators on 33 workgroups fell from 1111
 *    to 804 us, a 62-iteration run of 1024 subjects x 2048 trials of 4
 *    accumulators from 182 to 160 ms (about 80 ms of it host work).
 */
#ifndef GGDMC_LBA_MATH_H
#define GGDMC_LBA_MATH_H

#include <cmath>
#include <cstdint>
#include <cstring>

#ifdef __HIPCC__
#define GGDMC_FN __host__ __device__ __forceinline__
#else
#define GGDMC_FN inline
#endif

namespace ggdmc {

constexpr double kFloor = 1e-10;
constexpr double kLogFloor = -23.025850929940457;          /* log(1e-10)           */
constexpr double kInvSqrt2Pi = 0.3989422804014327;
constexpr double kLog2e = 1.4426950408889634;
constexpr double kLn2 = 0.6931471805599453;
constexpr double kMillsK = 0.2625;
constexpr int kMillsDeg = 10;
/* R(z) ~= t * sum_{k=0}^{10} c_k t^k, t = 1/(1 + 0.2625 z), z >= 0 */
constexpr double kMills[kMillsDeg + 1] = {
    0.10471908204997292, 0.10480896722129296, 0.09649084604609494,  0.090014727337448,
    0.032247173067295534, 0.13170626451118267, -0.1694328833813132, 0.2609796199857909,
    -0.23411156866613111, 0.09871999173116763, -0.016142220044834274};

/* Per (chain, cell, accumulator) constants, computed once per proposal. eL
 * and wU scale the quick error tests of losers and winners; they are NaN for
 * constants outside the range in which mixed_core may be trusted (A or s not
 * above 1e-30, any of them 1e30 or larger, NaN), so that such an accumulator
 * always takes the reference formula. Ten doubles: a 16-byte stride in LDS. */
struct AccK {
    double A, b, v, s, t0;
    double invA, den, inv_den, eL, wU;
};

/* ---------------------------------------------------------------- host/device
 * Policy interface (Ops): float log2(float), float rcp(float), double
 * exp2_frac(int).
 */

/* 1/x from the hardware seed (v_rcp_f64: 2^-24 relative over the whole double
 * range, at the issue cost of v_rcp_f32 with its two conversions) and one
 * Newton step; 0, infinities and NaN give infinities or NaN. The host takes a
 * quotient truncated to 24 bits for the seed. */
GGDMC_FN double rcp64(double x) {
#ifdef __HIP_DEVICE_COMPILE__
    const double r = __builtin_amdgcn_rcp(x);
#else
    double r = 1.0 / x;
    uint64_t u;
    std::memcpy(&u, &r, sizeof(u));
    u &= ~((uint64_t(1) << 29) - 1);
    std::memcpy(&r, &u, sizeof(u));
#endif
    return std::fma(std::fma(-x, r, 1.0), r, r);
}

/* The low 32 bits of a double. */
GGDMC_FN int32_t low_word(double x) {
    uint64_t u;
    std::memcpy(&u, &x, sizeof(u));
    return (int32_t)(uint32_t)u;
}

/* exp(-z^2/2) = 2^y, y = -(z^2/2) log2(e), in FP64 arithmetic: 64 y = k + f
 * with k the nearest integer and |f| <= 1/2; 2^(k/64) from a 64-entry table of
 * correctly rounded values (Ops::exp2_frac) and an exponent shift, 2^(f/64)
 * from its Taylor series to degree 5 (truncation below 4e-17), the powers of
 * ln(2)/64 folded into its coefficients. k is read from the low word of
 * 64 y + 1.5 2^52 and f is one multiply-add, exact but for its own rounding,
 * so the argument needs no separate product, scaling, rounding and
 * conversion instructions. z^2 is cut at 1492 (2^-1076, which rounds to 0); a
 * NaN z also gives 0 (fmin), so callers carry NaN through another factor
 * (the Mills ratio of the same argument). */
constexpr double kExpScale = -0.5 * kLog2e * 64.0;
constexpr double kLn2_64 = kLn2 / 64.0;
template <class Ops>
GGDMC_FN double exp_half_square(double z) {
    constexpr double kMagic = 6755399441055744.0; /* 1.5 2^52 */
    constexpr double c1 = kLn2_64, c2 = c1 * c1 / 2.0, c3 = c2 * c1 / 3.0, c4 = c3 * c1 / 4.0,
                     c5 = c4 * c1 / 5.0;
    const double zz = std::fmin(z * z, 1492.0);
    const double km = std::fma(zz, kExpScale, kMagic);
    const double f = std::fma(zz, kExpScale, kMagic - km);
    const int ki = low_word(km);
    /* Horner: one constant per multiply-add, which GFX9's single constant-bus
     * read per instruction takes straight from a scalar register */
    const double p = f * std::fma(f, std::fma(f, std::fma(f, std::fma(f, c5, c4), c3), c2), c1);
    const double tab = Ops::exp2_frac(ki & 63);
    return std::ldexp(std::fma(tab, p, tab), ki >> 6);
}

/* 2^(j/64), j = 0..63, correctly rounded to FP64 (the table of
 * exp_half_square). */
inline void fill_exp2_table(double *t) {
    for (int j = 0; j < 64; ++j) t[j] = (double)std::exp2((long double)j / 64.0L);
}

/* The Mills-ratio coefficients: kMills, or Ops's copy of them (the kernels keep
 * one in constant memory). */
template <class Ops>
GGDMC_FN auto mills_coefs(int) -> decltype(Ops::mills_coefs()) {
    return Ops::mills_coefs();
}
template <class Ops>
GGDMC_FN const double *mills_coefs(long) {
    return kMills;
}

/* e = exp(-z^2/2) and qa = Q(|z|), the upper normal tail beyond |z|, given
 * t = 1/(1 + 0.2625 |z|) (NaN for a NaN t). */
template <class Ops>
GGDMC_FN void mixed_tail_t(double z, double t, double &e, double &qa) {
    e = exp_half_square<Ops>(z);
    /* sum_k c_k t^k, k = 0..10, by Horner's rule: each multiply-add reads one
     * coefficient (a scalar register), so no coefficient is first moved into
     * vector registers; the two trials and two tails a lane evaluates give the
     * dependency chains to interleave */
    const double *c = mills_coefs<Ops>(0);
    double h = c[kMillsDeg];
#pragma unroll
    for (int j = kMillsDeg - 1; j >= 0; --j) h = std::fma(t, h, c[j]);
    qa = e * (t * h);
}

/* The same for a bare z. */
template <class Ops>
GGDMC_FN void mixed_tail(double z, double &e, double &qa) {
    mixed_tail_t<Ops>(z, rcp64(std::fma(kMillsK, std::fabs(z), 1.0)), e, qa);
}

/* log(x) for normal x > 0, FP32 log2 on the mantissa in [sqrt(1/2), sqrt(2));
 * mantissa and exponent by integer operations on the high word (half the
 * issue cost of the FP64 frexp, compare and select they replace). */
template <class Ops>
GGDMC_FN double mixed_log(double x) {
    uint64_t u;
    std::memcpy(&u, &x, sizeof(u));
    const int32_t hi = (int32_t)(u >> 32);
    const int32_t ex = (hi - 0x3FE6A09E) >> 20; /* high word of sqrt(1/2) */
    u = ((uint64_t)(uint32_t)(hi - (ex << 20)) << 32) | (uint32_t)u;
    double m;
    std::memcpy(&m, &u, sizeof(u));
    const float mf = (float)m;
    /* log(m) = log(mf) + r with r = (m - mf)/mf, |r| < 2^-24: an FP32 reciprocal suffices */
    const double r = (m - (double)mf) * (double)Ops::rcp(mf);
    return std::fma((double)Ops::log2(mf) + (double)ex, kLn2, r);
}

/* Shared core of one accumulator at time t > 0: z1 = chi/zs, z2 = (chi - A)/zs,
 * their tails q = Q(|z|) and e = exp(-z^2/2), dP = Phi(z1) - Phi(z2) and
 * de = e2 - e1. One reciprocal serves the three divisions: with
 * D1 = zs + K|chi|, D2 = zs + K|chi - A| the tails' arguments are
 * 1/(1 + K|z|) = zs/D, so r = 1/(zs D1 D2) gives 1/zs = D1 D2 r,
 * zs/D1 = zs^2 D2 r and zs/D2 = zs^2 D1 r. With a = q with the sign of z,
 * Phi(z) = [z >= 0] - a, so dP = (a2 - a1) + [z1 >= 0 > z2] is Q(z2) - Q(z1)
 * or Q(-z1) - Q(-z2) without cancellation when both z have one sign (A > 0,
 * so z1 >= z2; chi and chi - A are never -0). */
struct Core {
    double zs, chi, chiA, z1, z2, D, a1, a2, e1, e2, dP, de;
};

template <class Ops>
GGDMC_FN Core mixed_core(const AccK &k, double t) {
    Core c;
    c.zs = t * k.s;
    c.chi = std::fma(-t, k.v, k.b);
    c.chiA = c.chi - k.A;
    const double D1 = std::fma(kMillsK, std::fabs(c.chi), c.zs);
    const double D2 = std::fma(kMillsK, std::fabs(c.chiA), c.zs);
    c.D = D1 + D2;
    const double D12 = D1 * D2;
    const double r = rcp64(c.zs * D12);
    const double w = c.zs * (c.zs * r);
    const double r0 = D12 * r;
    c.z1 = c.chi * r0;
    c.z2 = c.chiA * r0;
    double q1, q2;
    mixed_tail_t<Ops>(c.z1, w * D2, c.e1, q1);
    mixed_tail_t<Ops>(c.z2, w * D1, c.e2, q2);
    c.a1 = std::copysign(q1, c.z1);
    c.a2 = std::copysign(q2, c.z2);
    c.dP = (c.a2 - c.a1) + (c.z1 >= 0.0 && c.z2 < 0.0 ? 1.0 : 0.0);
    c.de = c.e2 - c.e1;
    return c;
}

/* ------------------------------------------------------------- naive FP64 */
/* P = Phi(z) and d = phi(z): in one step where Ops has one (the kernels: the
 * same bits, from tables in LDS). */
template <class Ops>
GGDMC_FN auto normal_parts(double z, double &P, double &d, int) -> decltype(Ops::normal(z, P, d)) {
    Ops::normal(z, P, d);
}
template <class Ops>
GGDMC_FN void normal_parts(double z, double &P, double &d, long) {
    P = Ops::pnorm(z);
    d = Ops::dnorm(z);
}

/* x / d correctly rounded for finite x, y = 1/d correctly rounded: q = x*y,
 * then r = x - q*d exactly (one FMA) and RN(q + r*y) = RN(x/d) (Markstein's
 * correction step), while nothing overflows and x is 0 or above 1e-290. */
GGDMC_FN double div_finite(double x, double d, double y) {
    const double q = x * y;
    return std::fma(std::fma(-q, d, x), y, q);
}

/* The reference's intermediate values of one accumulator at t > 0. The two
 * quotients by zs share one division and correct its reciprocal (the same bits
 * as two divisions, of about 15 issue slots each); fine: the operands lie where
 * that holds (a quotient that the correction could round differently is below
 * 1e-190). */
struct NaiveParts {
    double zs, chi, chimA, P1, P2, d1, d2;
    bool fine;
};

template <class Ops>
GGDMC_FN NaiveParts naive_parts(const AccK &k, double t) {
    NaiveParts n;
    n.zs = t * k.s;
    n.chi = k.b - t * k.v;
    n.chimA = n.chi - k.A;
    n.fine = k.eL == k.eL && n.zs > 1e-100 && n.zs < 1e100 && std::fabs(n.chi) < 1e100;
    const double y = 1.0 / n.zs;
    double z1 = div_finite(n.chi, n.zs, y), z2 = div_finite(n.chimA, n.zs, y);
    if (__builtin_expect(!n.fine, 0)) {
        z1 = n.chi / n.zs;
        z2 = n.chimA / n.zs;
    }
    normal_parts<Ops>(z1, n.P1, n.d1, 0);
    normal_parts<Ops>(z2, n.P2, n.d2, 0);
    return n;
}

template <class Ops>
GGDMC_FN double naive_pdf(const AccK &k, double t) {
    if (!(t > 0.0)) return t == t ? 0.0 : t;
    const NaiveParts n = naive_parts<Ops>(k, t);
    return (k.v * (n.P1 - n.P2) + k.s * (n.d2 - n.d1)) / (k.A * k.den);
}

template <class Ops>
GGDMC_FN double naive_cdf(const AccK &k, double t) {
    if (!(t > 0.0)) return t == t ? 0.0 : t;
    const NaiveParts n = naive_parts<Ops>(k, t);
    const double num = n.zs * (n.d2 - n.d1) + n.chimA * n.P2 - n.chi * n.P1;
    /* quotients by A and den from their stored reciprocals */
    double cdf = div_finite(1.0 + div_finite(num, k.A, k.invA), k.den, k.inv_den);
    if (__builtin_expect(!n.fine, 0)) cdf = (1.0 + num / k.A) / k.den;
    return cdf;
}

template <class Ops>
GGDMC_FN void naive_pdf_cdf(const AccK &k, double t, double &pdf, double &cdf) {
    pdf = naive_pdf<Ops>(k, t);
    cdf = naive_cdf<Ops>(k, t);
}

/* Error model of the mixed evaluation: a computed tail carries a relative error
 * of up to kTailErr, exp(-z^2/2) of up to kExpErr; a result whose
 * bound exceeds kCondTol relative, or whose reference FP64 value carries more
 * rounding noise than that where the rounding is not reproduced (Phi rounded
 * near 1, ulp 1.1e-16, scaled by the formula's coefficients), is flagged
 * ill-conditioned and the trial is evaluated with the reference's FP64
 * formula instead. */
constexpr double kTailErr = 1e-9;   /* the Mills-ratio fit (2.9e-10; measured with the rest under 4e-10) */
constexpr double kExpErr = 1e-15;   /* exp(-z^2/2) in FP64 arithmetic */
constexpr double kCondTol = 1e-5;
constexpr double kUlp1 = 1.1102230246251565e-16;
/* a loser's reference noise per unit of D1 + D2 > K (|chi| + |chi - A|) */
constexpr double kLoserUlp = 4.3e-16; /* above kUlp1 / kMillsK */

/* div_finite for any x: x = +-inf takes x*y, which is x/d there. */
GGDMC_FN double div_rn(double x, double d, double y) {
    return std::isinf(x) ? x * y : div_finite(x, d, y);
}

/* One accumulator of a trial: its factor of the density, and whether the quick
 * error test vouches for it. */
struct Factor {
    Core c;
    double t, val, num;
    bool pos, ok;
};

/* x, or a negative number where !keep: cleared below by a floor. Only the high
 * word is selected. */
GGDMC_FN double or_negative(double x, bool keep) {
    uint64_t u;
    std::memcpy(&u, &x, sizeof(u));
    const uint32_t hi = keep ? (uint32_t)(u >> 32) : 0xBFF00000u;
    u = ((uint64_t)hi << 32) | (uint32_t)u;
    std::memcpy(&x, &u, sizeof(u));
    return x;
}

/* Winner: max(pdf, 1e-10), the reference's floored density. The numerator's
 * error is at most |v| (1e-9 (q1 + q2) + 2 ulp) + s 1e-15 (e1 + e2)/sqrt(2 pi);
 * with e1 + e2 <= 2 the test |num| >= 1e5 times that takes a multiply, two adds
 * and a multiply-add (wU holds the constant part), and only trials that fail
 * it (densities far in a tail, NaN, t <= 0) go through winner_careful. t <= 0
 * is evaluated as it stands and replaced. */
template <class Ops>
GGDMC_FN Factor winner_factor(const AccK &k, double rt) {
    Factor f;
    f.t = rt - k.t0;
    f.pos = f.t > 0.0;
    f.c = mixed_core<Ops>(k, f.t);
    f.num = std::fma(kInvSqrt2Pi, k.s * f.c.de, k.v * f.c.dP);
    f.val = std::fmax(or_negative(f.num * k.invA * k.inv_den, f.pos), kFloor);
    const double q = std::fabs(f.c.a1) + std::fabs(f.c.a2);
    f.ok = std::fma(std::fabs(k.v) * (kTailErr / kCondTol), q, k.wU) <= std::fabs(f.num);
    return f;
}

/* A winner that the quick test does not vouch for: the error bound in full,
 * the reference's own rounding in the far right tail, and ill where neither
 * suffices. */
GGDMC_FN void winner_careful(const AccK &k, Factor &f, bool &ill) {
    const Core &c = f.c;
    if (!f.pos) {
        ill |= f.t != f.t;
        return;
    }
    const double q1 = std::fabs(c.a1), q2 = std::fabs(c.a2);
    /* |v| (kTailErr (q1 + q2) + [z2 > 0] 2 ulp) + s (e1 + e2) kExpErr / sqrt(2 pi) */
    const double tv = std::fma(kTailErr, q1 + q2, c.z2 > 0.0 ? 2.0 * kUlp1 : 0.0);
    const double ex = k.s * (kExpErr * kInvSqrt2Pi) * (c.e1 + c.e2);
    double num = f.num;
    double err = std::fma(std::fabs(k.v), tv, ex);
    if (c.z2 > 0.0 && err > kCondTol * std::fabs(num)) {
        /* the far right tail, where the reference's Phi(z1) - Phi(z2) is the
         * difference of two values rounded near 1: take that difference,
         * RN(1 - Q1) - RN(1 - Q2), itself. 1 - q = p + r exactly (Fast2Sum,
         * p = RN(1 - q)); when r lies further than q's error from the rounding
         * midpoint p -+ ulp/2 (ulp = 2^-53 on [1/2, 1]), the reference's 1 - Q
         * rounds to p as well and the quantised difference is reproduced
         * exactly; otherwise it may be one ulp off */
        const double p1 = 1.0 - q1, p2 = 1.0 - q2;
        const double r1 = -q1 - (p1 - 1.0), r2 = -q2 - (p2 - 1.0);
        const double eq1 = kTailErr * q1, eq2 = kTailErr * q2;
        const double dP = p1 - p2;
        /* |v| (error of dP + 4 ulp of it for the products) + the exp term */
        const double tr = (0.5 * kUlp1 - std::fabs(r1) > eq1 ? 0.0 : eq1 + kUlp1) +
                          (0.5 * kUlp1 - std::fabs(r2) > eq2 ? 0.0 : eq2 + kUlp1) + 4.0 * kUlp1 * dP;
        num = std::fma(kInvSqrt2Pi, k.s * c.de, k.v * dP);
        err = std::fma(std::fabs(k.v), tr, ex);
    }
    f.val = std::fmax(num * k.invA * k.inv_den, kFloor);
    /* both floored unless the pdf or its uncertainty reaches the floor; NaN
     * and constants out of range (wU) are left to the reference formula */
    ill |= !(err <= kCondTol * std::fabs(num) || (std::fabs(num) + err) * k.invA * k.inv_den <= 0.5 * kFloor) ||
           k.wU != k.wU;
}

/* Loser: the reference's FP64 survivor 1 - max(F, 1e-10) (may be <= 0), from
 * 1 - G without cancellation and the reference's own FP64 steps
 * F = (1 + (G - 1)) / den: the rounding of 1 + (G - 1) is what quantises the
 * reference's survivor where F is near 1, and it is reproduced exactly
 * whenever 1 - G is accurate to well under half an ulp of 1. (Where F is small
 * 1 - F is as accurate either way: the survivor needs F's absolute error
 * only.) F's error is at most
 *   (|chi| (1e-9 q1 + ulp) + |chi - A| (1e-9 q2 + ulp) + 1e-15 zs (e1 + e2)/sqrt(2 pi)) / (A den);
 * as |z| Q(|z|) < 0.17 and K |chi| < D1, that is below
 * (0.345e-9 zs + 4.3e-16 (D1 + D2)) / (A den), tested against the survivor in
 * four instructions (eL holds 1e5 4.3e-16 / (A den)); trials that fail it go
 * through loser_careful. */
template <class Ops>
GGDMC_FN Factor loser_factor(const AccK &k, double rt) {
    Factor f;
    f.t = rt - k.t0;
    f.pos = f.t > 0.0;
    f.c = mixed_core<Ops>(k, f.t);
    const double P2 = (f.c.z2 < 0.0 ? 0.0 : 1.0) - f.c.a2;
    f.num = std::fma(std::fma(-kInvSqrt2Pi, f.c.zs * f.c.de, f.c.chi * f.c.dP), k.invA, P2); /* 1 - G */
    const double F = div_finite(1.0 - f.num, k.den, k.inv_den);
    f.val = 1.0 - std::fmax(or_negative(F, f.pos), kFloor);
    f.ok = std::fma(f.c.zs, 0.345e-9 / kLoserUlp, f.c.D) * k.eL <= std::fabs(f.val);
    return f;
}

/* A loser that the quick test does not vouch for. */
GGDMC_FN void loser_careful(const AccK &k, Factor &f, bool &ill) {
    const Core &c = f.c;
    if (!f.pos) {
        ill |= f.t != f.t;
        return;
    }
    if (std::isinf(f.num)) f.val = 1.0 - std::fmax(div_rn(1.0 - f.num, k.den, k.inv_den), kFloor);
    /* error of F from the tails, plus the reference's own noise from Phi
     * values rounded near 1 (z > 0), against the survivor */
    const double u1 = std::fma(kTailErr, std::fabs(c.a1), c.z1 > 0.0 ? kUlp1 : 0.0);
    const double u2 = std::fma(kTailErr, std::fabs(c.a2), c.z2 > 0.0 ? kUlp1 : 0.0);
    const double errF = std::fma(std::fabs(c.chi), u1,
                                 std::fma(std::fabs(c.chiA), u2, c.zs * (kExpErr * kInvSqrt2Pi) * (c.e1 + c.e2))) *
                        k.invA * k.inv_den;
    /* below a hundredth of an ulp of 1 the reference's own rounding of F is
     * reproduced exactly, whatever the survivor; NaN and constants out of
     * range (eL) are left to the reference formula */
    ill |= !(errF <= kCondTol * std::fabs(f.val) || errF <= 1e-18) || k.eL != k.eL;
}

/* max(pdf, 1e-10) of a winner; NaN sets ill. */
template <class Ops>
GGDMC_FN double mixed_winner_pdf(const AccK &k, double rt, bool &ill) {
    Factor f = winner_factor<Ops>(k, rt);
    if (!f.ok) winner_careful(k, f, ill);
    return f.val;
}

/* Winner: log(max(pdf, 1e-10)). */
template <class Ops>
GGDMC_FN double mixed_winner_logpdf(const AccK &k, double rt, bool &ill) {
    const double pf = mixed_winner_pdf<Ops>(k, rt, ill);
    return pf == kFloor ? kLogFloor : mixed_log<Ops>(pf);
}

/* Loser: the survivor; NaN sets ill. */
template <class Ops>
GGDMC_FN double mixed_loser_survivor(const AccK &k, double rt, bool &ill) {
    Factor f = loser_factor<Ops>(k, rt);
    if (!f.ok) loser_careful(k, f, ill);
    return f.val;
}

/* Reference FP64 trial term (src formula above), for the plain path and for
 * the batched path's ill-conditioned trials. */
template <class Ops>
GGDMC_FN double naive_trial_term(const AccK *kc, int n_acc, int w, double rt) {
    const double pdf = naive_pdf<Ops>(kc[w], rt - kc[w].t0);
    double dens = pdf != pdf ? pdf : (pdf > kFloor ? pdf : kFloor);
    /* losers in accumulator order; indexing the l-th loser (rather than
     * skipping j == w) keeps every lane of a wave on the same iteration */
    for (int l = 0; l + 1 < n_acc; ++l) {
        const int j = l + (l >= w);
        const double cdf = naive_cdf<Ops>(kc[j], rt - kc[j].t0);
        const double F = cdf != cdf ? cdf : (cdf > kFloor ? cdf : kFloor);
        dens *= (1.0 - F);
    }
    return Ops::log(dens <= 0.0 ? 2.220446049250313e-16 : dens);
}

/* Batched-path trial density, mixed evaluation: the reference's
 * max(pdf_w, 1e-10) * prod_{j != w} (1 - max(F_j, 1e-10)), multiplied in FP64
 * in accumulator order as the reference does, and DBL_EPSILON for a product
 * <= 0. A survivor is 0, or at least 2^-53 in magnitude, so the product of
 * n_acc - 1 <= 7 of them and the floored pdf is above 1e-122: normal, and so is
 * the product of two trials'. ill is set when any accumulator's evaluation is
 * ill-conditioned or NaN (the caller then takes naive_trial_term instead). */
GGDMC_FN double density_or_eps(double dens) { return dens <= 0.0 ? 2.220446049250313e-16 : dens; }

template <class Ops>
GGDMC_FN double mixed_density(const AccK *kc, int n_acc, int w, double rt, bool &ill) {
    double dens = mixed_winner_pdf<Ops>(kc[w], rt, ill);
    for (int l = 0; l + 1 < n_acc; ++l) dens *= mixed_loser_survivor<Ops>(kc[l + (l >= w)], rt, ill);
    return density_or_eps(dens);
}

/* Two independent trials' densities (A and B) in one body: both winner
 * factors, then each loser step of both, so that the two dependency chains
 * interleave in a wave that has few neighbours to hide latency with; one
 * branch covers both trials' careful forms. Per trial the same operations as
 * mixed_density, hence the same values. */
template <class Ops>
GGDMC_FN void mixed_density2(const AccK *kA, int wA, double rtA, const AccK *kB, int wB, double rtB,
                             int n_acc, double &outA, double &outB, bool &illA, bool &illB) {
    Factor fA = winner_factor<Ops>(kA[wA], rtA), fB = winner_factor<Ops>(kB[wB], rtB);
    if (__builtin_expect(!(fA.ok && fB.ok), 0)) {
        if (!fA.ok) winner_careful(kA[wA], fA, illA);
        if (!fB.ok) winner_careful(kB[wB], fB, illB);
    }
    double dA = fA.val, dB = fB.val;
    for (int l = 0; l + 1 < n_acc; ++l) {
        const int jA = l + (l >= wA), jB = l + (l >= wB);
        fA = loser_factor<Ops>(kA[jA], rtA);
        fB = loser_factor<Ops>(kB[jB], rtB);
        if (__builtin_expect(!(fA.ok && fB.ok), 0)) {
            if (!fA.ok) loser_careful(kA[jA], fA, illA);
            if (!fB.ok) loser_careful(kB[jB], fB, illB);
        }
        dA *= fA.val;
        dB *= fB.val;
    }
    outA = density_or_eps(dA);
    outB = density_or_eps(dB);
}

/* Batched-path trial term: mixed evaluation, or the reference formula when
 * any accumulator's evaluation is ill-conditioned. */
template <class Ops>
GGDMC_FN double mixed_trial_term(const AccK *kc, int n_acc, int w, double rt) {
    bool ill = false;
    const double dens = mixed_density<Ops>(kc, n_acc, w, rt, ill);
    return ill ? naive_trial_term<Ops>(kc, n_acc, w, rt) : mixed_log<Ops>(dens);
}

/* ----------------------------------------------------------- per (cell, acc)
 * Resolves the six families from theta / constants and fills AccK.
 * par_src / par_const are [n_acc * 6] for the cell. Returns false if st0 != 0
 * (the path implements st0 = 0 only).
 */
template <class Ops>
GGDMC_FN bool make_acck(const double *theta, const int32_t *src6, const double *const6,
                        AccK &k) {
    double f[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) f[i] = src6[i] >= 0 ? theta[src6[i]] : const6[i];
    k.A = f[0];
    k.b = f[0] + f[1];
    k.v = f[2];
    k.s = f[3];
    k.t0 = f[5];
    k.invA = 1.0 / k.A;
    const double x = k.v / k.s;
    /* q = Phi(-|x|) */
    const double q = Ops::qtail(std::fabs(x));
    const double Pv = x >= 0.0 ? 1.0 - q : (x == x ? q : x);   /* Phi(v/s)  */
    k.den = Pv > kFloor ? Pv : (Pv == Pv ? kFloor : Pv);
    k.inv_den = 1.0 / k.den;
    const bool fine = std::fmin(k.A, k.s) > 1e-30 &&
                      std::fmax(std::fmax(k.A, k.s), std::fmax(std::fabs(k.b), std::fabs(k.v))) < 1e30 &&
                      x == x && k.b == k.b;
    k.eL = fine ? kLoserUlp / kCondTol * k.invA * k.inv_den : NAN;
    k.wU = fine ? std::fma(2.0 * kUlp1 / kCondTol, std::fabs(k.v), 2.0 * kExpErr / kCondTol * kInvSqrt2Pi * k.s)
                : NAN;
    return f[4] == 0.0;
}

} // namespace ggdmc

#endif
