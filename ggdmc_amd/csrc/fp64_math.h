/*
 * Accurate FP64 exp, log and normal tail for the reference-formula evaluations
 * of the HIP kernels (the plain FP64 path, the batched path's fallback for
 * ill-conditioned trials, the likelihood constants and the priors), written
 * for this library so that no math-library routine (with its register-resident
 * constant tables) is inlined into the kernels.
 *
 *  exp_acc(x)   e^x for x <= 709: x = k ln2/64 + r with ln2/64 in two parts
 *               (Cody & Waite argument reduction), 2^(k/64) from the 64-entry
 *               table, e^r by its Taylor series to degree 6 (|r| <= ln2/128,
 *               truncation below 3e-20); about 2 ulp.
 *  log_acc(x)   x > 0: x = m 2^e with m in [sqrt(1/2), sqrt(2)),
 *               log m = 2 atanh(s), s = (m - 1)/(m + 1), by 11 terms of the
 *               atanh series (|s| <= 0.172, truncation below 1e-18), plus
 *               e ln2 with ln2 in two parts; about 2 ulp.
 *  qtail_acc(a) upper normal tail Q(a) = P(Z > a), a >= 0, as
 *               exp(-a^2/2) R(a): a^2 split exactly (one FMA), R the Mills
 *               ratio from the piecewise polynomials below (1 ulp); about 4 ulp.
 *
 * Tables: generated for this library with 50-digit arithmetic.
 */
#ifndef GGDMC_FP64_MATH_H
#define GGDMC_FP64_MATH_H

#include <cmath>

#ifdef __HIPCC__
#define GGDMC_MFN __host__ __device__ __forceinline__
#else
#define GGDMC_MFN inline
#endif

namespace ggdmc {

/* 2^(j/64), j = 0..63, correctly rounded. */
constexpr double kExp2Tab[64] = {
    1.0, 1.0108892860517005, 1.0218971486541166, 1.0330248790212284,
    1.0442737824274138, 1.0556451783605572, 1.0671404006768237, 1.0787607977571199,
    1.0905077326652577, 1.102382583307841, 1.1143867425958924, 1.1265216186082418,
    1.1387886347566916, 1.1511892299529827, 1.1637248587775775, 1.1763969916502812,
    1.189207115002721, 1.202156731452703, 1.215247359980469, 1.22848053610687,
    1.241857812073484, 1.255380757024691, 1.2690509571917332, 1.2828700160787783,
    1.2968395546510096, 1.3109612115247644, 1.3252366431597413, 1.339667524053303,
    1.3542555469368927, 1.3690024229745905, 1.383909881963832, 1.3989796725383112,
    1.4142135623730951, 1.42961333839197, 1.4451808069770467, 1.460917794180647,
    1.4768261459394993, 1.4929077282912648, 1.5091644275934228, 1.5255981507445384,
    1.5422108254079407, 1.559004400237837, 1.5759808451078865, 1.593142151342267,
    1.6104903319492543, 1.6280274218573478, 1.645755478153965, 1.6636765803267364,
    1.681792830507429, 1.7001063537185235, 1.718619298122478, 1.7373338352737062,
    1.7562521603732995, 1.7753764925265212, 1.7947090750031072, 1.8142521755003989,
    1.8340080864093424, 1.8539791250833855, 1.8741676341103, 1.8945759815869656,
    1.9152065613971474, 1.9360617934922943, 1.9571441241754002, 1.978456026387951,
};
/* Mills ratio R(a) = Q(a) exp(a^2/2) in 9 pieces of degree 16: piece k < 8 covers
 * a in [k, k+1) in s = 2(a - k) - 1; piece 8 covers a >= 8 as R(a) = P(s)/a,
 * s = 128/a^2 - 1. Chebyshev interpolants of the exact function (computed
 * with 50-digit arithmetic), converted to monomial coefficients. */
constexpr int kMillsPieceDeg = 16;
constexpr double kMillsPieces[9][17] = {
    {0.34961883472039806, -0.11206643152061682, 0.029694050399972655, -0.006864365093387165, 0.0014268553316616193, -0.0002718754880841504, 4.812416014874036e-05, -7.991118868216706e-06, 1.2541575418953088e-06, -1.8713776998622836e-07, 2.6675488309109142e-08, -3.6469544873483034e-09, 4.797721003481152e-10, -6.08163613947021e-11, 7.46979328787379e-12, -9.41128236705851e-13, 1.0850267550855344e-13},
    {0.2057806669773947, -0.045135639967670324, 0.008796718384297965, -0.0015621237345647056, 0.00025689669878774165, -3.957168191002321e-05, 5.7575688773917115e-06, -7.963919745285434e-07, 1.0526227986744934e-07, -1.3350141570624807e-08, 1.6302961953977497e-09, -1.9225776672335474e-10, 2.194871558542579e-11, -2.4288195649224335e-12, 2.61498556698211e-13, -2.8647625777412395e-14, 2.921937325969836e-15},
    {0.1413313313805753, -0.0228069759749972, 0.0034120564381986624, -0.0004788911486669909, 6.36000434289818e-05, -8.044546576102266e-06, 9.740546061857315e-07, -1.1336691233911623e-07, 1.272562639310673e-08, -1.381632749846506e-09, 1.4543655799112663e-10, -1.487393519045426e-11, 1.4805738666579809e-12, -1.4359627793509724e-13, 1.3603991004734039e-14, -1.304226869334686e-15, 1.1802119522101067e-16},
    {0.10634515363370545, -0.013367121341731807, 0.0015969130301978494, -0.0001823941775289052, 2.0009611718469557e-05, -2.1163447749808218e-06, 2.1646659556679066e-07, -2.1467093072491167e-08, 2.068654502028983e-09, -1.9406976354712032e-10, 1.775415343481403e-11, -1.5861557431671185e-12, 1.3856464581540963e-13, -1.1846066613370294e-14, 9.92801093102512e-16, -8.389123111896433e-17, 6.7638046998180986e-18},
    {0.08480339210780034, -0.008663507958165556, 0.0008539775605387919, -8.147582610970247e-05, 7.54344534696686e-06, -6.792408993500299e-07, 5.959488553402168e-08, -5.103104626606365e-09, 4.270919967194693e-10, -3.4979906978595645e-11, 2.8068208076733228e-12, -2.208757054710886e-13, 1.7061304963633323e-14, -1.2944141577267493e-15, 9.657138178474875e-17, -7.24640341062719e-18, 5.232589514498543e-19},
    {0.07034269402512788, -0.006028731631614648, 0.000503330759670845, -4.100777293627943e-05, 3.265328585735706e-06, -2.544579246593325e-07, 1.942880893679336e-08, -1.4550366555253123e-09, 1.0698142893946525e-10, -7.728914909692574e-12, 5.490841191683529e-13, -3.838615048103997e-14, 2.6424331203823483e-15, -1.7919393823403013e-16, 1.198100217159116e-17, -8.043514956326451e-19, 5.231585086728447e-20},
    {0.06001567534317183, -0.00442019533540789, 0.0003191419978586574, -2.2612446937111967e-05, 1.5737617297626162e-06, -1.0767722250989765e-07, 7.2482432139144124e-09, -4.803593117507837e-10, 3.1361630036262454e-11, -2.0182811452613537e-12, 1.280993781660465e-13, -8.022485104374498e-15, 4.959815239911595e-16, -3.0280351620552016e-17, 1.8266272370002272e-18, -1.1051897009778467e-19, 6.512714304342635e-21},
    {0.052293097118194715, -0.003372026007486157, 0.00021408837573779502, -1.3391697618269317e-05, 8.258069664847036e-07, -5.022965604993818e-08, 3.0150885723179435e-09, -1.7869026661323662e-10, 1.0460455410010803e-11, -6.050954293396255e-13, 3.460059916661774e-14, -1.956510401573256e-15, 1.0943644673917867e-16, -6.056606773421078e-18, 3.3179279563956184e-19, -1.8216680098611244e-20, 9.782286674709372e-22},
    {0.39589588482488375, -0.0029786255133119914, 6.532711140277205e-05, -2.322953707299462e-06, 1.1261446442046953e-07, -6.842138987167744e-09, 4.957107754952934e-10, -4.14442709631715e-11, 3.90690284052492e-12, -4.0818255565966057e-13, 4.664116704597881e-14, -5.76840999040235e-15, 7.654950476350089e-16, -1.0761111519583064e-16, 1.6098155568961464e-17, -2.8997265905586032e-18, 4.859094890846157e-19},
};
constexpr double kLn2By64Hi = 0.010830424696249145, kLn2By64Lo = 3.623510646634843e-19;
constexpr double kLn2Hi = 0.6931471805599453, kLn2Lo = 2.3190468138462996e-17;

/* e^x; x > 709.78 overflows to +inf, x < -745.2 underflows to 0, NaN passes.
 * tab: the 64 values above or a copy of them. */
GGDMC_MFN double exp_acc(double x, const double *tab = kExp2Tab) {
    const bool in = x > -745.2 && x < 709.8;
    const double xc = in ? x : 0.0;
    const double k = std::rint(xc * 92.33248261689366);   /* 64 / ln 2 */
    double r = std::fma(-k, kLn2By64Hi, xc);
    r = std::fma(-k, kLn2By64Lo, r);
    const double p =
        1.0 + r * (1.0 + r * (0.5 + r * (0.16666666666666666 +
                                         r * (0.041666666666666664 +
                                              r * (0.008333333333333333 + r * 0.001388888888888889)))));
    const int ki = (int)k;
    const double v = std::ldexp(tab[ki & 63] * p, ki >> 6);
    return in ? v : (x != x ? x : (x > 0.0 ? HUGE_VAL : 0.0));
}

/* log(x); 0 gives -inf, negative or NaN gives NaN, +inf gives +inf. */
GGDMC_MFN double log_acc(double x) {
    int e;
    double m = std::frexp(x, &e);            /* x = m 2^e, m in [0.5, 1) */
    const bool lo = m < 0.7071067811865476;
    m = lo ? 2.0 * m : m;
    e = lo ? e - 1 : e;
    const double s = (m - 1.0) / (m + 1.0);
    const double s2 = s * s;
    /* atanh(s)/s = sum s^(2k)/(2k+1), k = 0..10 */
    double h = 1.0 / 21.0;
    h = 1.0 / 19.0 + s2 * h;
    h = 1.0 / 17.0 + s2 * h;
    h = 1.0 / 15.0 + s2 * h;
    h = 1.0 / 13.0 + s2 * h;
    h = 1.0 / 11.0 + s2 * h;
    h = 1.0 / 9.0 + s2 * h;
    h = 1.0 / 7.0 + s2 * h;
    h = 1.0 / 5.0 + s2 * h;
    h = 1.0 / 3.0 + s2 * h;
    const double lm = 2.0 * s + 2.0 * s * (s2 * h);
    const double ed = (double)e;
    const double v = ed * kLn2Hi + (ed * kLn2Lo + lm);
    const bool finite = x > 0.0 && x < HUGE_VAL;
    return finite ? v : (x == 0.0 ? -HUGE_VAL : (x == HUGE_VAL ? x : (x - x) / 0.0 * 0.0 + NAN));
}

/* The Mills ratio R(a) = Q(a) exp(a^2/2), a >= 0. pieces: kMillsPieces or a
 * copy. The asymptotic piece and its two divisions stand behind a branch that
 * few waves take. */
GGDMC_MFN double mills_acc(double a, const double *pieces = &kMillsPieces[0][0]) {
    const int k = a < 8.0 ? (int)a : 8;
    double s = 2.0 * (a - (double)k) - 1.0;
    if (!(a < 8.0)) s = 128.0 / (a * a) - 1.0;
    const double *c = pieces + k * (kMillsPieceDeg + 1);
    double h = c[kMillsPieceDeg];
#pragma unroll
    for (int j = kMillsPieceDeg - 1; j >= 0; --j) h = c[j] + s * h;
    if (!(a < 8.0)) h = h / a;
    return h;
}

/* Q(a) = P(Z > a) for a >= 0 (a = +inf gives 0, NaN passes). */
GGDMC_MFN double qtail_acc(double a, const double *tab = kExp2Tab, const double *pieces = &kMillsPieces[0][0]) {
    if (!(a < 1e300)) return a != a ? a : 0.0;
    const double a2 = a * a;
    const double a2l = std::fma(a, a, -a2);         /* a^2 = a2 + a2l exactly */
    const double e = exp_acc(-0.5 * a2, tab);
    return std::fma(e, -0.5 * a2l, e) * mills_acc(a, pieces);
}

/* Phi(z) as R's pnorm rounds it: the lower tail directly, above 0 as
 * 1 - the upper tail. */
GGDMC_MFN double pnorm_acc(double z) {
    return z > 0.0 ? 1.0 - qtail_acc(z) : qtail_acc(-z);
}

/* P = pnorm_acc(z) and e = exp_acc(-z^2/2), the same bits from one exponential
 * (z^2/2 is the argument of both) and without the range selects that a
 * non-positive argument does not need: |z| is cut at 40, where Q is 0. A NaN z
 * gives a NaN P (through the Mills ratio). */
GGDMC_MFN void normal_acc(double z, const double *tab, const double *pieces, double &P, double &e) {
    double a = std::fabs(z);
    a = a > 40.0 ? 40.0 : a;
    const double a2 = a * a;
    const double a2l = std::fma(a, a, -a2);
    const double x = -0.5 * a2;
    const double k = std::rint(x * 92.33248261689366);   /* 64 / ln 2 */
    double r = std::fma(-k, kLn2By64Hi, x);
    r = std::fma(-k, kLn2By64Lo, r);
    const double p =
        1.0 + r * (1.0 + r * (0.5 + r * (0.16666666666666666 +
                                         r * (0.041666666666666664 +
                                              r * (0.008333333333333333 + r * 0.001388888888888889)))));
    const int ki = (int)k;
    e = std::ldexp(tab[ki & 63] * p, ki >> 6);
    const double q = std::fma(e, -0.5 * a2l, e) * mills_acc(a, pieces);
    P = z > 0.0 ? 1.0 - q : q;
}

} // namespace ggdmc

#endif
