// mr_dec_core.h -- squaring modulo a search-form number in base 10^13, with
// transforms over two 50-bit primes in FP64 arithmetic.
//
// A candidate N = 10^D - Q has a sparse decimal Q (a few digits and 1), so in
// base B = 10^13 a product reduces modulo N by adding shifted multiples of
// its high (or low) half by the digits of Q: one transform product per
// squaring, where a general Montgomery step needs three.  (50 000 digits,
// 256 numbers: 136 us per squaring in mr_core.h's Montgomery step.)
//
// Why FP64: a modular product by two fused multiply-adds (h = a w, l = the
// exact remainder a w - h, q = rint(h / p), r = (h - q p) + l) takes 6
// instructions for a 50-bit prime, and gfx950 issues FP64 instructions at the
// rate of 32-bit integer multiplies (measured: fma_f64 29, mul_lo_u32 32 T
// lane-operations/s), so one point of a 50-bit prime costs what one point of
// a 31-bit prime costs, at 1.6 times the bits.  All values are integers below
// 2^53 in magnitude and every operation is exact; the bounds that make it so
// are stated where they are used and tracked at compile time (Plan).
//
// Primes p = y^4 + 1: y is a primitive 8th root of one, so multiplying by a
// power of y is a = a1 y^j + a0 -> a0 y^(4-j) - a1, 4 instructions without a
// table.  P0 = 5072^4 + 1, P1 = 5232^4 + 1 (both 1 mod 2^16).
//
// Digits are balanced (|d| <= B/2 and a little) and never fully carried: a
// number is any digit vector with that value, and one local carry per
// squaring keeps the digits bounded.
//
// This file compiles for the device and, with PF_DEC_HOST, for the host
// (threads and barriers emulated), where a test compares it with big-integer
// arithmetic.
#pragma once
#include <stdint.h>
#ifdef PF_DEC_HOST
#include <math.h>
#define PF_DEC_FN inline
#define PF_DEC_HD inline
namespace mr { namespace dec {
int  tid();
void sync_waves();
void sync_wave();
void sync_global();
double lane_up(double x);          // the value of the lane below (lane 0: unspecified)
inline double fma_(double a, double b, double c) { return fma(a, b, c); }
inline double rint_(double a) { return rint(a); }
inline int uniform(int x) { return x; }
inline double uniform_d(double x) { return x; }
} }
#else
#include <hip/hip_runtime.h>
#define PF_DEC_FN __device__ __forceinline__
#define PF_DEC_HD __host__ __device__ inline
namespace mr { namespace dec {
// The thread index through an empty asm: otherwise every index derived from
// it is hoisted out of the squaring loop and spills.
__device__ __forceinline__ int tid()
{
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}
// LDS hand-off between the waves of a block; global loads stay in flight.
__device__ __forceinline__ void sync_waves()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// LDS hand-off inside one wave: its LDS operations complete in order, so only
// the compiler has to keep them in order.
__device__ __forceinline__ void sync_wave() { asm volatile("" ::: "memory"); }
// Hand-off through global memory within the block.
__device__ __forceinline__ void sync_global() { __syncthreads(); }
__device__ __forceinline__ double lane_up(double x)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, 0x138, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), 0x138, 0xF, 0xF, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ double rint_(double a) { return __builtin_rint(a); }
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ double uniform_d(double x)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = (unsigned)uniform((int)(unsigned)u), hi = (unsigned)uniform((int)(unsigned)(u >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
} }
#endif
#pragma clang fp contract(off)

namespace mr { namespace dec {

constexpr int    DIGITS = 13;                   // decimal digits per limb
constexpr double B = 1e13, IB = 1e-13;

constexpr uint64_t Y0 = 5072, Y1 = 5232;
constexpr uint64_t P0 = Y0 * Y0 * Y0 * Y0 + 1, P1 = Y1 * Y1 * Y1 * Y1 + 1;

constexpr uint64_t mulmod(uint64_t a, uint64_t b, uint64_t p)
{
    return (uint64_t)((unsigned __int128)a * b % p);
}
constexpr uint64_t powmod(uint64_t a, uint64_t e, uint64_t p)
{
    uint64_t r = 1;
    for (a %= p; e; e >>= 1) {
        if (e & 1) r = mulmod(r, a, p);
        a = mulmod(a, a, p);
    }
    return r;
}
// The representative of x in (-p/2, p/2).
constexpr double balanced(uint64_t x, uint64_t p)
{
    return x > p / 2 ? -(double)(p - x) : (double)x;
}
// A primitive 2^16-th root w of one mod p = y^4 + 1 whose 2^13-th power is y
// (so that the 8th root is y itself): g^((p-1)/2^16) to the odd power that
// does it, for the first g that is no square.
constexpr uint64_t root16(uint64_t y, uint64_t p)
{
    for (uint64_t g = 2;; g++) {
        if (powmod(g, (p - 1) / 2, p) != p - 1) continue;
        const uint64_t w = powmod(g, (p - 1) >> 16, p);
        for (uint64_t e = 1; e < 8; e += 2)
            if (powmod(w, e << 13, p) == y) return powmod(w, e, p);
    }
}

// Constants of one prime: W the 32nd root with W^4 = y, r[k] = W^k (k < 16; the
// multiples of 4 are powers of y and not used).
struct Fp {
    double p, ip, y, y2, y3, iy, iy2, iy3, r[16];
};
constexpr Fp make_fp(uint64_t y, uint64_t p)
{
    const uint64_t w = powmod(root16(y, p), 1u << 11, p);
    const double d = (double)y;
    Fp f = {(double)p, 1.0 / (double)p, d, d * d, d * d * d, 1.0 / d, 1.0 / (d * d), 1.0 / (d * d * d), {}};
    for (int k = 0; k < 16; k++) f.r[k] = balanced(powmod(w, (uint64_t)k, p), p);
    return f;
}
constexpr Fp FP0 = make_fp(Y0, P0), FP1 = make_fp(Y1, P1);

// CRT of coefficients V, |V| < P0 P1 / 2: V = r0 + P0 u with
// u = (r1 - r0) P0^-1 mod P1; then V in base B from P0 = CA B + CA0.
constexpr double INV01 = balanced(powmod(P0 % P1, P1 - 2, P1), P1);
struct Base10 {                     // search-form candidates
    static constexpr double B = 1e13, IB = 1e-13, CA = (double)((P0 + 5000000000000ull) / 10000000000000ull),
                            CA0 = (double)((int64_t)P0 - (int64_t)CA * 10000000000000ll);
};
struct Base2 {                      // any odd modulus
    static constexpr int BITS = 43;
    static constexpr double B = 8796093022208.0, IB = 1.0 / B,
                            CA = (double)((P0 + (1ull << 42)) >> 43), CA0 = (double)((int64_t)P0 - ((int64_t)CA << 43));
};

// a w mod p for |w| <= p/2: |result| <= (0.5 + 0.125 |a|/p) p, exact while
// |a w| / p < 2^52 (q's three roundings lose at most 0.125 |a|/p).
PF_DEC_FN double mulmod_d(double a, double w, double p, double ip)
{
    const double h = a * w;
    const double q = rint_(h * ip);
    const double l = fma_(a, w, -h);
    return fma_(-q, p, h) + l;
}
// a to within p/2.
PF_DEC_FN double reduce(double a, double p, double ip)
{
    return fma_(-rint_(a * ip), p, a);
}

// a W^E for the 32nd root W (E mod 32, a compile-time constant after
// unrolling): multiples of 4 by powers of y (4 instructions, |result| <= p/2 +
// 2^41), the others by a constant.
PF_DEC_FN double mul_w(const Fp &F, double a, int E)
{
    E &= 31;
    const bool neg = E >= 16;
    E &= 15;
    if (E == 0) return neg ? -a : a;
    if (E & 3) return mulmod_d(neg ? -a : a, F.r[E], F.p, F.ip);
    // E = 4, 8, 12: y^j with a = a1 y^(4-j) + a0
    const double ih = E == 4 ? F.iy3 : E == 8 ? F.iy2 : F.iy;
    const double hi = E == 4 ? F.y3 : E == 8 ? F.y2 : F.y;
    const double lo = E == 4 ? F.y : E == 8 ? F.y2 : F.y3;
    const double a1 = rint_(a * ih);
    const double a0 = fma_(-a1, hi, a);
    return neg ? fma_(-a0, lo, a1) : fma_(a0, lo, -a1);
}

// ---- bounds -------------------------------------------------------------
// Magnitudes in units of p, tracked through a radix-2^LR butterfly network at
// compile time.  An element is reduced (3 instructions) before a level when
// it exceeds PLAN_T; sums stay below 2 PLAN_T p < 2^53 (2^53 / P1 = 12.0).
constexpr double PLAN_T = 3.5;
constexpr double rho(double a) { return 0.501 + 0.125 * a; }
struct Plan {
    bool red[5][32];
    double m[32], out;              // output magnitudes, the largest
};
// inv = false: natural in, bit-reversed out (decimation in frequency);
// inv = true: the mirror.  b0: bound of element 0, b: of the others.
constexpr Plan make_plan(int LR, bool inv, double b0, double b)
{
    Plan P = {};
    const int R = 1 << LR;
    double m[32] = {};
    for (int i = 0; i < R; i++) m[i] = i ? b : b0;
    for (int l = 0; l < LR; l++) {
        const int h = inv ? 1 << l : R >> (l + 1);
        for (int i = 0; i < R; i++) {
            P.red[l][i] = m[i] > PLAN_T;
            if (P.red[l][i]) m[i] = 0.501;
        }
        for (int s = 0; s < R; s += 2 * h)
            for (int j = 0; j < h; j++) {
                const int e = j * 32 / (2 * h);
                if (inv) {
                    const double c = e == 0 ? m[s + j + h] : (e & 3) ? rho(m[s + j + h]) : 0.501;
                    m[s + j] = m[s + j + h] = m[s + j] + c;
                } else {
                    const double t = m[s + j] + m[s + j + h];
                    m[s + j] = t;
                    m[s + j + h] = e == 0 ? t : (e & 3) ? rho(t) : 0.501;
                }
            }
    }
    for (int i = 0; i < R; i++) {
        P.m[i] = m[i];
        P.out = m[i] > P.out ? m[i] : P.out;
    }
    return P;
}
// Squares x^2 mod p: |x^2| / p < 2^52 up to SQ_T p, off by at most 0.25 x^2 /
// p^2 before the final half.
constexpr double SQ_T = 2.2;
constexpr double rho_sq(double a) { return 0.501 + 0.25 * a * a; }
// Inputs of a scaled pass: every element but the first was just multiplied
// (rho of at most 2 PLAN_T: 1.376).
constexpr double SCALED = rho(2 * PLAN_T);

// DFT of 2^LR elements, element bounds (thousandths of p) as for make_plan.
// HALF: the upper half of the inputs is zero (and not read).
template <int LR, bool INV, int B0_1000, int B_1000, bool HALF = false>
PF_DEC_FN void dft(double *x, const Fp &F)
{
    constexpr Plan P = make_plan(LR, INV, B0_1000 * 1e-3, B_1000 * 1e-3);
    static_assert(P.out <= 2 * PLAN_T, "sums stay exact");
    constexpr int R = 1 << LR;
#pragma unroll
    for (int l = 0; l < LR; l++) {
        const int h = INV ? 1 << l : R >> (l + 1);
#pragma unroll
        for (int i = 0; i < R; i++)
            if (P.red[l][i]) x[i] = reduce(x[i], F.p, F.ip);
#pragma unroll
        for (int s = 0; s < R; s += 2 * h)
#pragma unroll
            for (int j = 0; j < h; j++) {
                const int e = j * 32 / (2 * h);
                const double a = x[s + j], c = HALF && l == 0 ? 0.0 : x[s + j + h];
                if (HALF && l == 0) {
                    x[s + j + h] = mul_w(F, a, e);
                } else if (INV) {
                    const double d = mul_w(F, c, -e);
                    x[s + j] = a + d;
                    x[s + j + h] = a - d;
                } else {
                    x[s + j] = a + c;
                    x[s + j + h] = mul_w(F, a - c, e);
                }
            }
    }
}

// ---- geometry -------------------------------------------------------------
// A product of M = 2^LM points.  Forward: the ring X^M - 1 is split level by
// level (block b of 2^d blocks is modulo X^(M/2^d) - zeta_d^brv(b)); a pass
// takes LR levels: scale x_k by gamma_b^k, then a plain DFT of R = 2^LR
// elements at stride Q.  The first pass has gamma = 1 (no table); from the
// second pass on the data of a wave (64 R consecutive points) stay with it, so
// only the first pass and its mirror need block barriers.
constexpr int MIN_LM = 7, MAX_LM = 14;
#ifndef PF_LR
#define PF_LR(lm) (lm >= 14 ? 5 : lm >= 13 ? 4 : lm >= 11 ? 3 : 2)
#endif
constexpr int lr_of(int lm) { return PF_LR(lm); }

template <int LM_>
struct G {
    static constexpr int LM = LM_, LR = lr_of(LM_), M = 1 << LM, R = 1 << LR;
    static constexpr bool SEQ = LM > 13;                 // primes one after the other (LDS)
    static constexpr int TP = M / R;                     // threads per prime
    static constexpr int THREADS = SEQ ? TP : 2 * TP;
    static constexpr int NS = (LM + LR - 1) / LR - 1;    // strided passes
    static constexpr int TL = LM - LR * NS;              // levels of the tail
    static constexpr int C = R / 2;                      // coefficients a thread carries
    static constexpr int XP = M + M / 16;                // padded words of a transform buffer
    static constexpr int LDS = SEQ ? XP : 2 * XP;
    static_assert(M <= 64 * R * R, "passes after the first stay in a wave");
    static_assert(TL >= 1 && TL <= LR, "tail");
};
// Pad of two words per 32: the strided passes, the contiguous tail and the
// contiguous coefficient runs all spread over the 64 banks.
PF_DEC_FN int pd(int i) { return i + ((i >> 5) << 1); }
// pd(base + d) - pd(base) for a compile-time d with base mod 32 + d mod 32 <
// 32: an element's offset from its thread's first one, an immediate of the LDS
// instruction instead of an address register.
PF_DEC_HD constexpr int po(int d) { return d + ((d >> 5) << 1); }

// Twiddle tables of a class: per prime and direction, per pass from the
// second on (nb blocks) and then the tail, (radix - 1) x nb values
// gamma_b^(+-k) at (k - 1) nb + b.
constexpr int tab_off(int lm, int pass)
{
    int o = 0;
    for (int s = 1; s < pass; s++) o += ((1 << lr_of(lm)) - 1) << (lr_of(lm) * s);
    return o;
}
template <int LM>
constexpr int tab_size()
{
    return tab_off(LM, G<LM>::NS) + (((1 << G<LM>::TL) - 1) << (G<LM>::LR * G<LM>::NS));
}
constexpr int tab_size_rt(int lm)
{
    const int lr = lr_of(lm), ns = (lm + lr - 1) / lr - 1, tl = lm - lr * ns;
    return tab_off(lm, ns) + (((1 << tl) - 1) << (lr * ns));
}

// The tables of class lm: out[4 tab_size], [prime][forward, inverse].
inline void build_tables(int lm, double *out)
{
    const int lr = lr_of(lm), ns = (lm + lr - 1) / lr - 1, ts = tab_size_rt(lm);
    for (int q = 0; q < 2; q++) {
        const uint64_t p = q ? P1 : P0, w = root16(q ? Y1 : Y0, p);
        for (int inv = 0; inv < 2; inv++)
            for (int pass = 1; pass <= ns; pass++) {
                const int d = lr * pass, rad = 1 << (pass < ns ? lr : lm - lr * ns), nb = 1 << d;
                const int lv = pass < ns ? d + lr : lm;         // gamma is a power of zeta_lv
                double *o = out + (2 * q + inv) * ts + tab_off(lm, pass);
                const uint64_t zeta = powmod(w, (inv ? (1ull << 16) - 1u : 1ull) << (16 - lv), p);
                for (int b = 0; b < nb; b++) {
                    int r = 0;
                    for (int i = 0; i < d; i++) r |= ((b >> i) & 1) << (d - 1 - i);
                    const uint64_t gamma = powmod(zeta, (uint64_t)r, p);
                    uint64_t x = 1;
                    for (int k = 1; k < rad; k++) {
                        x = mulmod(x, gamma, p);
                        o[(k - 1) * nb + b] = balanced(x, p);
                    }
                }
            }
    }
}

// ---- a candidate's form -----------------------------------------------------
// N = 10^D - sum c_i 10^(e_i) (c_i > 0; Q's terms, the 1 among them).
// mode TOP: arithmetic modulo N 10^z, z = 13 Lw - D, where B^Lw = Q 10^z:
//   the limbs from Lw up fold down by Q 10^z.
// mode BOTTOM: Montgomery with R = B^Lw >= 10^(D + 8): adding t_p B^p N clears
//   limb p below Lw, since N = -1 modulo 10^(least e_i).
// mode DENSE: BOTTOM with all of m = T N' mod R at once, N' = -N^-1 mod R, by
//   a second transform product, then T + m N by the sparse terms.
// Each term adds coef * (t shifted by 13 E + s digits); a fold round of TOP or
// BOTTOM clears at most `gap` limbs, so that its targets lie outside its
// sources.
//
// The multiple is a unit (Q's 1, or 10^D) and groups of up to six digits, so
// that a candidate with k, j below 10^6 has one group for each.
constexpr int MAX_TERMS = 16, TOP = 0, BOTTOM = 1, DENSE = 2;
struct Term {
    double c;                       // signed coefficient, |c| < 10^6
    double ts, tc, itc;             // 10^s, 10^(13 - s) and its inverse
    int32_t E, s;                   // target offset in limbs (TOP: less Lw), digit shift
};
struct Form {
    int32_t lm;                     // class, 0: not handled here
    int32_t mode, Lw, gap, nt;      // gap: limbs per fold round
    int32_t D, z, f;                // f = 13 Lw - D
    int32_t omin, omax;             // least and largest offset over the terms
    Term t[MAX_TERMS];              // the unit (TOP: Q's 1, else 10^D), then the groups
};

// How a candidate with D digits whose Q has its terms (but the 1) at exponents
// [lo, hi) is handled: class and mode, or lm = 0.  TOP and BOTTOM need a gap
// of at least one limb between sources and targets; lo >= 2 makes N - 1 = 2
// mod 4 (one squaring chain, s = 1); hi < D keeps Q below N/10.  Where the
// fewer of the two modes' rounds would cost more than a second product
// (dense_from rounds, measured), DENSE; its N' comes from BOTTOM's rounds, run
// once, or, where lo leaves them no gap, limb by limb (solve).
constexpr int MAX_ROUNDS = 64, MIN_DIGITS = 40, MAX_BASE = 511;
constexpr int dense_from(int lm) { return lm <= 8 ? 7 : lm <= 11 ? 8 : 10; }
struct Choice { int32_t lm, mode; };
PF_DEC_HD Choice choose(int64_t D, int64_t lo, int64_t hi)
{
    Choice c = {0, TOP};
    if (D < MIN_DIGITS || lo < 2 || hi >= D) return c;
    const int64_t Lt = (D + DIGITS - 1) / DIGITS, Lb = (D + 8 + DIGITS - 1) / DIGITS;
    const int64_t z = DIGITS * Lt - D;
    const int64_t gt = Lt - (hi - 1 + z) / DIGITS - 2, gb = lo / DIGITS;
    const int64_t none = 1 << 30;
    const int64_t rt = gt >= 1 ? (Lt + gt) / gt : none, rb = gb >= 1 ? (Lb + gb - 1) / gb : none;
    if (rb == none && rt > MAX_ROUNDS) return c;
    c.mode = rt <= rb ? TOP : BOTTOM;
    const int64_t L = c.mode == TOP ? Lt : Lb;
    for (int lm = MIN_LM; lm <= MAX_LM && !c.lm; lm++)
        if ((1ll << lm) >= 2 * L + 4) c.lm = lm;
    if (c.lm && (rt < rb ? rt : rb) >= dense_from(c.lm)) {
        const int lm = 2 * Lb + 4 <= (1ll << c.lm) ? c.lm : c.lm < MAX_LM ? c.lm + 1 : 0;
        if (lm || gb >= 1) c = {lm, DENSE};
    }
    return c;
}

// The form of N = sum of coef 10^exp over terms[0 .. nterm) (pairs, in any
// order, unused ones zero): +1 at D, the rest negative.
PF_DEC_HD void make_form(const int64_t *terms, int nterm, int64_t D, int lm, int mode, Form &f)
{
    int64_t e[MAX_TERMS * 2], g[MAX_TERMS * 2];
    int n = 0;
    for (int i = 0; i < nterm; i++) {           // Q less its 1, by exponent
        int64_t c = -terms[2 * i], x = terms[2 * i + 1];
        if (x == 0 && c > 0) c--;
        if (c <= 0 || n == MAX_TERMS * 2) continue;
        int at = n++;
        for (; at > 0 && e[at - 1] > x; at--) { e[at] = e[at - 1]; g[at] = g[at - 1]; }
        e[at] = x;
        g[at] = c;
    }
    f.mode = mode;
    f.D = (int32_t)D;
    f.Lw = (int32_t)((D + (mode == TOP ? 0 : 8) + DIGITS - 1) / DIGITS);
    f.f = DIGITS * f.Lw - f.D;
    f.z = mode == TOP ? f.f : 0;
    f.nt = 0;
    f.lm = lm;
    f.omin = 1 << 30;
    f.omax = -(1 << 30);
    auto put = [&](int64_t x, double c) {
        if (f.nt == MAX_TERMS) { f.lm = 0; return; }
        Term &t = f.t[f.nt++];
        t.c = c;
        t.s = (int32_t)(x % DIGITS);
        t.E = (int32_t)(x / DIGITS) - (mode == TOP ? f.Lw : 0);
        t.ts = 1.0;
        for (int i = 0; i < t.s; i++) t.ts *= 10.0;
        t.tc = B / t.ts;                        // exact
        t.itc = t.ts / B;
        f.omin = t.E < f.omin ? t.E : f.omin;
        f.omax = t.E > f.omax ? t.E : f.omax;
    };
    put(mode == TOP ? f.z : D, 1.0);
    for (int i = 0; i < n;) {                   // neighbouring digits below 10^6 together
        int64_t c = 0, w = 1, at = e[i];
        for (; i < n && e[i] - at <= 5; i++) {
            for (w = 1; w < 1000000 && at + (w < 10 ? 0 : w < 100 ? 1 : w < 1000 ? 2 : w < 10000 ? 3 : w < 100000 ? 4 : 5) < e[i];) w *= 10;
            if (c + g[i] * w >= 1000000) break;
            c += g[i] * w;
        }
        if (c == 0) { c = g[i]; i++; }          // (10^6 itself, as k or j)
        put(at + f.z, mode == TOP ? (double)c : -(double)c);
    }
    f.gap = mode == TOP ? -f.omax - 2 : f.omin;
    if (f.gap < 1 && mode != DENSE) f.lm = 0;
}

// Group k >= 1 of Q as limbs: lo at limb E, hi at limb E + 1.
struct Share { int32_t E; int64_t lo, hi; };
PF_DEC_HD Share share_of(const Form &f, int k)
{
    const Term &t = f.t[k];
    const int64_t x = (int64_t)DIGITS * (t.E + (f.mode == TOP ? f.Lw : 0)) + t.s - f.z;
    const int64_t c = (int64_t)(t.c < 0.0 ? -t.c : t.c);
    int64_t ts = 1;
    for (int i = 0; i < (int)(x % DIGITS); i++) ts *= 10;
    const int64_t tc = 10000000000000ll / ts;
    return {(int32_t)(x / DIGITS), c % tc * ts, c / tc};
}

// Whether the digits v[0 .. Lw) of a number are m N + add (m 0 or 1; sh: the
// shares of groups 1 .. nt - 1): their difference is carried up from the lowest
// limb, where nearly every number that differs ends it.
template <class V>
PF_DEC_HD bool equals(const V *v, const Form &f, const Share *sh, int m, int add)
{
    const int64_t Bi = 10000000000000ll;
    const int ED = f.D / DIGITS;
    int64_t c = m - add, top = m;               // N = 10^D - 1 - groups
    for (int i = 0; i < f.D % DIGITS; i++) top *= 10;
    for (int i = 0; i < f.Lw + 2; i++) {
        c += i < f.Lw ? (int64_t)v[i] : 0;
        if (m) {
            c -= i == ED ? top : 0;
            for (int k = 1; k < f.nt; k++)
                c += (i == sh[k].E ? sh[k].lo : 0) + (i == sh[k].E + 1 ? sh[k].hi : 0);
        }
        if (c % Bi) return false;
        c /= Bi;
    }
    return c == 0;
}

// Where T waits during a DENSE squaring: in the LDS, behind the transforms (and
// the zero word), where it fits; its limbs come back a barrier later instead of
// a trip to memory.
template <int LM>
constexpr bool park_lds() { return LM <= 12; }
template <int LM>
constexpr int lds_words() { return G<LM>::LDS + 2 + (park_lds<LM>() ? G<LM>::M : 0); }

// A block of one wave needs no barrier (its LDS operations stay in order).
template <int LM>
PF_DEC_FN void sync_block()
{
    if constexpr (G<LM>::THREADS > 64) sync_waves();
    else sync_wave();
}

// ---- transform ----------------------------------------------------------------
// v[k] scaled by gamma^(+-k) with the table row at tab (entries nb apart).
template <int N>
PF_DEC_FN void load_tw(double (&w)[N - 1], const double *tab, int nb)
{
#pragma unroll
    for (int k = 1; k < N; k++) w[k - 1] = tab[(k - 1) * nb];
}

// A thread's twiddles of everything but the first pass, for one direction.
// Where the registers allow (few waves per SIMD), they are loaded once for a
// whole chunk of squarings: at these lengths a squaring is a chain of LDS
// round trips, and a table load in each pass doubles the chain.
template <int LM>
struct Twid {
    using g = G<LM>;
    static constexpr int NB = g::R >> g::TL, T = 1 << g::TL;
    double w[g::NS > 1 ? g::NS - 1 : 1][g::R - 1], tail[NB][T - 1];
    PF_DEC_FN void load(const double *tab, int t)
    {
#pragma unroll
        for (int P = 1; P < g::NS; P++)
            load_tw<g::R>(w[P - 1], tab + tab_off(LM, P) + block_of(P, t), 1 << (g::LR * P));
#pragma unroll
        for (int m = 0; m < NB; m++)
            load_tw<T>(tail[m], tab + tab_off(LM, g::NS) + t * NB + m, 1 << (g::LR * g::NS));
    }
    static PF_DEC_FN int block_of(int P, int t) { return (int)((unsigned)t >> (LM - g::LR * (P + 1))); }
};

// The middle of a product: from the first pass's outputs in X (natural order)
// to the inverse of everything but the first pass, in place; the pointwise
// step squares (Nt == nullptr) or multiplies by the transform Nt (point k of
// thread t at k TP + t).  out: store the transform there instead, and stop.
// Waves work on their own points.  h: hoisted twiddles (forward, inverse).
template <int LM, bool HOIST>
PF_DEC_FN void middle(double *X, const Fp &F, const double *tf, const double *ti, int t, const Twid<LM> *h,
                      const double *Nt, double *out = nullptr)
{
    using g = G<LM>;
    constexpr int R = g::R, LR = g::LR;
    constexpr int S1 = (int)(SCALED * 1000) + 1, S0 = (int)(2 * PLAN_T * 1000);
    double v[R];
#pragma unroll
    for (int P = 1; P < g::NS; P++) {
        const int S = g::M >> (LR * P), Q = S >> LR, nb = 1 << (LR * P);
        const int b = Twid<LM>::block_of(P, t);
        double *Xb = X + pd(b * S + (t & (Q - 1)));
        double l[R - 1];
        if (!HOIST) load_tw<R>(l, tf + tab_off(LM, P) + b, nb);
        const double *w = HOIST ? h[0].w[P - 1] : l;
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = Xb[po(k * Q)];
#pragma unroll
        for (int k = 1; k < R; k++) v[k] = mulmod_d(v[k], w[k - 1], F.p, F.ip);
        dft<LR, false, S0, S1>(v, F);
#pragma unroll
        for (int k = 0; k < R; k++) Xb[po(k * Q)] = v[k];
        sync_wave();
    }
    {   // tail: R / 2^TL blocks of 2^TL consecutive points, squared in registers
        constexpr int TL = g::TL, T = 1 << TL, NB = R / T;
        constexpr int nb = 1 << (LR * g::NS), off = tab_off(LM, g::NS);
        constexpr Plan P = make_plan(TL, false, S0 * 1e-3, S1 * 1e-3);
        constexpr int SQ = (int)(1000 * rho_sq(P.out < SQ_T ? P.out : SQ_T)) + 1;
        double *Xb = X + pd(t * R);
        double l[NB][T - 1], li[NB][T - 1];
        if (!HOIST)
#pragma unroll
            for (int m = 0; m < NB; m++) load_tw<T>(l[m], tf + off + t * NB + m, nb);
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = Xb[po(k)];
#pragma unroll
        for (int m = 0; m < NB; m++) {
            double *u = v + m * T;
            const double *w = HOIST ? h[0].tail[m] : l[m];
#pragma unroll
            for (int k = 1; k < T; k++) u[k] = mulmod_d(u[k], w[k - 1], F.p, F.ip);
            dft<TL, false, S0, S1>(u, F);
#pragma unroll
            for (int k = 0; k < T; k++)
                if (P.m[k] > SQ_T) u[k] = reduce(u[k], F.p, F.ip);
        }
        if (out) {
#pragma unroll
            for (int k = 0; k < R; k++) out[k * g::TP + t] = reduce(v[k], F.p, F.ip);
            return;
        }
        if (Nt) {
#pragma unroll
            for (int k = 0; k < R; k++) v[k] = mulmod_d(v[k], Nt[k * g::TP + t], F.p, F.ip);
        } else {
#pragma unroll
            for (int k = 0; k < R; k++) v[k] = mulmod_d(v[k], v[k], F.p, F.ip);
        }
        if (!HOIST) {
            if (R > 16) sync_wave();        // (loaded earlier, the second half of the twiddles spills)
#pragma unroll
            for (int m = 0; m < NB; m++) load_tw<T>(li[m], ti + off + t * NB + m, nb);
        }
#pragma unroll
        for (int m = 0; m < NB; m++) {
            double *u = v + m * T;
            const double *wi = HOIST ? h[1].tail[m] : li[m];
            dft<TL, true, SQ, SQ>(u, F);
            u[0] = reduce(u[0], F.p, F.ip);
#pragma unroll
            for (int k = 1; k < T; k++) u[k] = mulmod_d(u[k], wi[k - 1], F.p, F.ip);
        }
#pragma unroll
        for (int k = 0; k < R; k++) Xb[po(k)] = v[k];
        sync_wave();
    }
#pragma unroll
    for (int P = g::NS - 1; P >= 1; P--) {
        const int S = g::M >> (LR * P), Q = S >> LR, nb = 1 << (LR * P);
        const int b = Twid<LM>::block_of(P, t);
        double *Xb = X + pd(b * S + (t & (Q - 1)));
        double l[R - 1];
        if (!HOIST) load_tw<R>(l, ti + tab_off(LM, P) + b, nb);
        const double *w = HOIST ? h[1].w[P - 1] : l;
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = Xb[po(k * Q)];
        dft<LR, true, S1, S1>(v, F);
        v[0] = reduce(v[0], F.p, F.ip);
#pragma unroll
        for (int k = 1; k < R; k++) v[k] = mulmod_d(v[k], w[k - 1], F.p, F.ip);
#pragma unroll
        for (int k = 0; k < R; k++) Xb[po(k * Q)] = v[k];
        sync_wave();
    }
}

// ---- digits of coefficients -------------------------------------------------
struct Split { double d0, d1, d2; };
// The coefficient V = M^-1 (r0 mod P0, r1 mod P1), |V| < 2^97.4, in base B.
// M^-1 a = a1 - a0 (p - 1)/M for a = a1 M + a0.
template <class S, int LM>
PF_DEC_FN Split crt_split(double r0, double r1)
{
    constexpr double Md = (double)(1 << LM), iM = 1.0 / Md;
    constexpr double K0 = (double)((P0 - 1) >> LM), K1 = (double)((P1 - 1) >> LM);
    const double a = rint_(r0 * iM);
    const double x0 = fma_(-fma_(-a, Md, r0), K0, a);
    const double b = rint_(r1 * iM);
    const double x1 = fma_(-fma_(-b, Md, r1), K1, b);
    constexpr double p1 = (double)P1, ip1 = 1.0 / (double)P1;
    double u = mulmod_d(x1 - x0, INV01, p1, ip1);
    if (LM > 13) u = reduce(u, p1, ip1);        // |V / P0| reaches 0.43 P1: q's rounding may be one off
    const double u1 = rint_(u * S::IB), u0 = fma_(-u1, S::B, u);
    const double h = u0 * S::CA0, l = fma_(u0, S::CA0, -h);
    const double q = rint_(h * S::IB);
    const double s0 = (fma_(-q, S::B, h) + l) + x0;
    const double q0 = rint_(s0 * S::IB);
    const double s1 = fma_(S::CA, u0, fma_(S::CA0, u1, q + q0));
    const double q1 = rint_(s1 * S::IB);
    Split o;
    o.d0 = fma_(-q0, S::B, s0);
    o.d1 = fma_(-q1, S::B, s1);
    o.d2 = fma_(S::CA, u1, q1);
    return o;
}

// A run of C coefficients -> limbs, first half: z[i] = mul (d0[i] + d1[i-1] +
// d2[i-2]) as far as the run knows them.  o0, o1: what the next run's first
// two limbs still get; oc: the carry out of z[C-1] (run_finish takes the same
// one out of it).
template <class S, int C, int LM, class LD0, class LD1>
PF_DEC_FN void run_digits(double (&z)[C], LD0 r0, LD1 r1, double mul, double &o0, double &o1, double &oc)
{
    double p1 = 0.0, p2 = 0.0, q2 = 0.0;        // d1[i-1], d2[i-1], d2[i-2]
#pragma unroll
    for (int i = 0; i < C; i++) {
        const Split s = crt_split<S, LM>(r0(i), r1(i));
        z[i] = mul * (s.d0 + p1 + q2);
        p1 = s.d1;
        q2 = p2;
        p2 = s.d2;
    }
    o0 = mul * (p1 + q2);
    o1 = mul * p2;
    oc = rint_(z[C - 1] * S::IB);
}
// Second half: with the run below's o0, o1, oc.  Limbs stay below
// B/2 + 2^12: |z| <= 512 (B + 2^12), an exact carry of at most 2^10 each.
template <class S, int C>
PF_DEC_FN void run_finish(double (&z)[C], double i0, double i1, double ic, double oc)
{
    z[0] += i0;
    z[1] += i1;
    double cin = ic;
#pragma unroll
    for (int i = 0; i < C; i++) {
        const double c = i == C - 1 ? oc : rint_(z[i] * S::IB);
        z[i] = fma_(-c, S::B, z[i]) + cin;
        cin = c;
    }
}

// ---- fold rounds ----------------------------------------------------------------
// A target limb i gathers, per term with offset o, c times the shifted limb
//   w = 10^s (t[i-o] mod 10^(13-s)) + (t[i-o-1] div 10^(13-s))
// (balanced remainders).  c w < 2^63 splits exactly into a carry and a
// remainder of at most B/2 (h = c w rounded, l = c w - h).  Lanes take
// consecutive targets, 62 new ones a wave: the quotient by 10^(13-s) comes from
// the lane below, whose own limb it is (lane 0), and so does the carry (lane
// 1).  A round is one LDS latency and a chain of arithmetic: the unit and two
// groups wait in scalar registers, a limb outside the sources is read from a
// zero word (index zi) instead of branched around.  (Groups of two digits, terms
// in LDS and branches took 1 800 cycles a round.)
constexpr int NT = 2;               // groups held in registers
struct Terms {
    int nt, Lw, gap, mode, omin, omax, E[NT + 1];
    double c[NT + 1], ts[NT + 1], tc[NT + 1], itc[NT + 1];
};
PF_DEC_FN void load_terms(Terms &u, const Form &f)
{
    u.nt = uniform(f.nt); u.Lw = uniform(f.Lw); u.gap = uniform(f.gap); u.mode = uniform(f.mode);
    u.omin = uniform(f.omin); u.omax = uniform(f.omax);
#pragma unroll
    for (int k = 0; k <= NT; k++) {
        const bool on = k < u.nt;
        const Term &m = f.t[on ? k : 0];
        u.E[k] = uniform(on ? m.E : 1 << 29);       // out of every range
        u.c[k] = uniform_d(m.c); u.ts[k] = uniform_d(m.ts);
        u.tc[k] = uniform_d(m.tc); u.itc[k] = uniform_d(m.itc);
    }
}

// acc + the terms' multiples of the source limbs S[s0 .. s1) at target i; what
// they carry out of the limb is added to car.  (Leaving out the terms that
// reach no limb of a strip was slower: 100 000 digits, two rounds 54.6 -> 61 us.)
PF_DEC_FN double gather(double acc, double &car, const double *S, int s0, int s1, int zi, int i,
                        const Form &f, const Terms &u)
{
    double a[NT + 1];
    const unsigned n = (unsigned)(s1 - s0);
#pragma unroll
    for (int k = 0; k <= NT; k++) {
        const int p = i - u.E[k];
        a[k] = S[(unsigned)(p - s0) < n ? pd(p) : zi];
    }
    {
        const double q = rint_(a[0] * u.itc[0]);
        acc += fma_(u.ts[0], fma_(-q, u.tc[0], a[0]), lane_up(q));
    }
    auto group = [&](double x, double c, double ts, double tc, double itc) {
        const double q = rint_(x * itc), w = fma_(ts, fma_(-q, tc, x), lane_up(q));
        const double h = c * w, g = rint_(h * IB);
        acc += fma_(-g, B, h) + fma_(c, w, -h);
        car += g;
    };
#pragma unroll
    for (int k = 1; k <= NT; k++) group(a[k], u.c[k], u.ts[k], u.tc[k], u.itc[k]);
    for (int k = NT + 1; k < u.nt; k++) {
        const Term &m = f.t[k];
        const int p = i - m.E;
        group(S[(unsigned)(p - s0) < n ? pd(p) : zi], m.c, m.ts, m.tc, m.itc);
    }
    return acc;
}

// v = q B + r, 0 <= r < B, for |v| < 2^92: the quotient estimated in FP64 (below
// 2^49, off by a unit or two), r exact.
PF_DEC_FN int64_t split(__int128 v, int64_t &r)
{
    const int64_t Bi = 10000000000000ll;
    const double e = (double)(int64_t)(v >> 64) * 18446744073709551616.0 + (double)(uint64_t)v;
    int64_t q = (int64_t)(e * IB);
    v -= (__int128)q * Bi;
    while (v < 0) { v += Bi; q--; }
    while (v >= Bi) { v -= Bi; q++; }
    r = (int64_t)v;
    return q;
}

// T (limbs in LDS, padded; limbs from Lw up zero) -> m with T + m N = 0 mod R at
// limbs [0, Lw), and, with high, (T + m N) / R at [Lw, 2 Lw): what BOTTOM's
// rounds compute, limb by limb for terms that leave them no gap (digits of Q
// below 10^13: a limb of m is the limb of the sum so far over the lowest limb of
// 1 + Q's groups, a unit since every exponent is at least 2).  One thread; once
// per candidate and per round, where up to MAX_ROUNDS fold rounds in every
// squaring cost up to 13.7 us in class 8 against 4 (a batch of 300 numbers with one
// such: 95 -> 64 ms).
PF_DEC_FN void solve(double *T, const Form &f, bool high)
{
    const int64_t Bi = 10000000000000ll;
    const int Lw = f.Lw, ED = f.D / DIGITS;
    Share sh[MAX_TERMS];
    int64_t u0 = 1, top = 1;
    for (int i = 0; i < f.D % DIGITS; i++) top *= 10;
    for (int k = 1; k < f.nt; k++) {
        sh[k] = share_of(f, k);
        if (sh[k].E == 0) u0 += sh[k].lo;
    }
    int64_t w = 1, x;                           // 1 / u0 mod B: 2, 4, 8, 16 digits
    for (int n = 0; n < 3; n++) {
        split((__int128)(u0 % Bi) * w, x);
        split((__int128)w * (2 - x), w);
    }
    int64_t carry = 0;
    for (int i = 0; i < (high ? 2 * Lw : Lw); i++) {
        auto m = [&](int p) { return p >= 0 && p < Lw && p < i ? (int64_t)T[pd(p)] : (int64_t)0; };
        __int128 v = (__int128)(int64_t)T[pd(i)] + carry + (__int128)top * m(i - ED);
        for (int k = 1; k < f.nt; k++) v -= (__int128)sh[k].lo * m(i - sh[k].E) + (__int128)sh[k].hi * m(i - sh[k].E - 1);
        int64_t d;
        carry = split(v, d);
        if (i < Lw) {
            split((__int128)d * w, d);
            if (d > Bi / 2) d -= Bi;
            carry = split(v - (__int128)d * u0, x);
        } else if (d > Bi / 2) {
            d -= Bi;
            carry++;
        }
        T[pd(i)] = (double)d;
    }
}

// T (limbs in LDS, padded) -> the product reduced, at limbs [0, Lw) (TOP) or
// [Lw, 2 Lw) (BOTTOM).  A round's targets lie outside its sources and span at
// most Lw + 2 limbs.  T[zi] is zero.  (Cutting the targets into one window per
// group saved work but cost more in bookkeeping: 380 digits, two rounds 3.4 ->
// 6.4 us a squaring.)  rec (BOTTOM on T = 1): the limbs cleared, N'.
template <int LM>
PF_DEC_FN void fold(double *T, int zi, const Form &f, const Terms &u, int t, double *rec = nullptr)
{
    constexpr int W = G<LM>::THREADS / 64, STEP = 62 * W, NI = (G<LM>::M / 2 + 1 + STEP) / STEP;
    const int lane = t & 63, wave = uniform(t >> 6);
    const int Lw = u.Lw, gap = u.gap;
    if (rec && gap < 1) {
        if (t == 0) solve(T, f, false);
        sync_block<LM>();
        for (int i = t; i < Lw; i += G<LM>::THREADS) rec[i] = T[pd(i)];
        return;
    }
    const bool top = u.mode == TOP;
    const int first = top ? Lw : 0, last = top ? 2 * Lw + 1 : Lw;
    for (int done = 0; first + done < last; done += gap) {
        int s0, s1;
        if (top) { s1 = last - done; s0 = s1 - gap < Lw ? Lw : s1 - gap; }
        else { s0 = done; s1 = s0 + gap > Lw ? Lw : s0 + gap; }
        const int lo = s0 + u.omin, hi = s1 + u.omax + 1;       // targets [lo, hi]
        if (rec)
            for (int i = s0 + t; i < s1; i += G<LM>::THREADS) rec[i] = T[pd(i)];
        double out[NI];
#pragma unroll
        for (int n = 0; n < NI; n++) {
            const int i0 = lo + n * STEP + wave * 62 - 2, i = i0 + lane;
            if (i0 + 2 <= hi) {
                double car = 0.0;
                const double acc = gather(T[i >= lo && i <= hi ? pd(i) : zi],   // (limb lo - 1 keeps its carry)
                                          car, T, s0, s1, zi, i, f, u);
                const double c = i < hi ? rint_(acc * IB) : 0.0;    // (limb hi only takes one in)
                out[n] = fma_(-c, B, acc) + lane_up(c + car);
            }
        }
        sync_block<LM>();
#pragma unroll
        for (int n = 0; n < NI; n++) {
            const int i = lo + n * STEP + wave * 62 - 2 + lane;
            if (lane > 1 && i <= hi) T[pd(i)] = out[n];
        }
        sync_block<LM>();
    }
}

// DENSE: m's limbs [0, Lw) in X (LDS), T's limbs in park -> (T + m N) / R at
// X's limbs [Lw, 2 Lw).  The limbs below Lw come to zero: after the carries
// their digits are at most B/2 and a little, so the multiple of B^Lw that they
// sum to is zero, and only limb Lw - 1's carry is needed from them.
template <int LM>
PF_DEC_FN void dense_tail(double *X, int zi, const double *park, const Form &f, const Terms &u, int t)
{
    constexpr int W = G<LM>::THREADS / 64;
    const int lane = t & 63, wave = uniform(t >> 6), Lw = u.Lw;
    for (int st = wave; st * 62 < Lw; st += W) {
        const int i = Lw + st * 62 - 2 + lane;
        double acc = i >= Lw - 1 && i <= 2 * Lw ? park[i] : 0.0;
        if (st == 0) acc -= X[i == Lw - 1 ? pd(i) : zi];        // N's -1 ends at Lw - 1
        double car = 0.0;
        acc = gather(acc, car, X, 0, Lw, zi, i, f, u);
        const double c = rint_(acc * IB);
        acc = fma_(-c, B, acc) + lane_up(c + car);
        if (lane > 1 && i < 2 * Lw) X[pd(i)] = acc;
    }
    sync_block<LM>();
}

// ---- products ------------------------------------------------------------------
template <int LM>
constexpr bool hoisted() { return LM <= 11; }

PF_DEC_FN Fp prime_of(int q)
{
    Fp F;
    F.p = q ? FP1.p : FP0.p; F.ip = q ? FP1.ip : FP0.ip;
    F.y = q ? FP1.y : FP0.y; F.y2 = q ? FP1.y2 : FP0.y2; F.y3 = q ? FP1.y3 : FP0.y3;
    F.iy = q ? FP1.iy : FP0.iy; F.iy2 = q ? FP1.iy2 : FP0.iy2; F.iy3 = q ? FP1.iy3 : FP0.iy3;
#pragma unroll
    for (int k = 0; k < 16; k++) F.r[k] = q ? FP1.r[k] : FP0.r[k];
    return F;
}

// X: G<LM>::LDS words; the digits of x at limbs [off, off + n).  Leaves mul x^2,
// or mul x times the number whose transform is at Nt (per prime M words), as
// limbs [0, live + 2) at X (live: limbs of the result that are needed).  bnd: 3
// words per wave.  tab: the class's tables, [prime][forward, inverse]; h: this
// thread's hoisted twiddles (hoisted classes), F0 its prime's constants (chosen
// once: the choice costs as much as a pass); keep: 3 M/2 words of global memory
// (SEQ classes).  Begins after a barrier and ends with one.
template <class S, int LM>
PF_DEC_FN void product(double *X, double *bnd, const Fp &F0, int n, int off, int live, const double *tab,
                       double mul, const Twid<LM> *h, const double *Nt, double *keep)
{
    using g = G<LM>;
    constexpr int R = g::R, Q = g::M / R, C = g::C, TS = tab_size<LM>();
    constexpr int S1 = (int)(SCALED * 1000) + 1;
    const int t = tid(), lane = t & 63, wave = t >> 6;
    double i0, i1, ic, oc;
    auto hand_on = [&](double o0, double o1, double c) {     // to the next thread's run
        i0 = lane_up(o0);
        i1 = lane_up(o1);
        ic = lane_up(c);
        if (lane == 63) { bnd[3 * wave] = o0; bnd[3 * wave + 1] = o1; bnd[3 * wave + 2] = c; }
    };
    auto take = [&](bool first) {
        if (lane == 0) {
            i0 = first ? 0.0 : bnd[3 * wave - 3];
            i1 = first ? 0.0 : bnd[3 * wave - 2];
            ic = first ? 0.0 : bnd[3 * wave - 1];
        }
    };
    if constexpr (!g::SEQ) {
        const int q = g::TP >= 64 ? uniform(t / g::TP) : t / g::TP, tp = t & (g::TP - 1);
        const Fp &F = F0;
        const double *tf = tab + 2 * q * TS, *ti = tf + TS;
        double *Y = X + q * g::XP, *Yb = Y + pd(tp);
        const double *Xd = X + pd(off + tp);
        double v[R];
#pragma unroll
        for (int k = 0; k < R / 2; k++) {
            const int i = tp + k * Q;
            v[k] = i < n ? Xd[po(k * Q)] : 0.0;
        }
        sync_block<LM>();
        dft<g::LR, false, 10, 10, true>(v, F);      // |digit| < 2^42.4: 0.01 p
#pragma unroll
        for (int k = 0; k < R; k++) Yb[po(k * Q)] = v[k];
        sync_block<LM>();
        middle<LM, hoisted<LM>()>(Y, F, tf, ti, tp, h, Nt ? Nt + q * g::M : nullptr);
        sync_block<LM>();
#pragma unroll
        for (int k = 0; k < R; k++) v[k] = Yb[po(k * Q)];
        dft<g::LR, true, S1, S1>(v, F);
#pragma unroll
        for (int k = 0; k < R; k++) Yb[po(k * Q)] = v[k];
        sync_block<LM>();
        double z[C], o0 = 0.0, o1 = 0.0, *Xr = X + pd(t * C);
        const bool in = uniform(t & ~63) * C <= live + 2;       // waves above what is needed stay out
        oc = 0.0;
        if (in)
            run_digits<S, C, LM>(z, [&](int i) { return Xr[po(i)]; },
                              [&](int i) { return Xr[g::XP + po(i)]; }, mul, o0, o1, oc);
        hand_on(o0, o1, oc);
        sync_block<LM>();
        take(t == 0);
        if (in) {
            run_finish<S, C>(z, i0, i1, ic, oc);
#pragma unroll
            for (int i = 0; i < C; i++) Xr[po(i)] = z[i];
        }
    } else {
        // the first prime's residues and the digits wait in keep (point k of thread
        // t at k TP + t): in registers they spilled
        double v[R], *Xb = X + pd(t), *Xr = X + pd(t * C);
        const double *Xd = X + pd(off + t);
#pragma unroll
        for (int k = 0; k < R / 2; k++) {
            const int i = t + k * Q;
            v[k] = i < n ? Xd[po(k * Q)] : 0.0;
            keep[g::M + k * g::TP + t] = v[k];
        }
#pragma clang loop unroll(disable)
        for (int q = 0; q < 2; q++) {
            const Fp F = prime_of(q);
            const double *tf = tab + 2 * q * TS, *ti = tf + TS;
            if (q)
#pragma unroll
                for (int k = 0; k < R / 2; k++) v[k] = keep[g::M + k * g::TP + t];
            sync_block<LM>();
            dft<g::LR, false, 10, 10, true>(v, F);
#pragma unroll
            for (int k = 0; k < R; k++) Xb[po(k * Q)] = v[k];
            sync_block<LM>();
            middle<LM, false>(X, F, tf, ti, t, nullptr, Nt ? Nt + q * g::M : nullptr);
            sync_block<LM>();
#pragma unroll
            for (int k = 0; k < R; k++) v[k] = Xb[po(k * Q)];
            dft<g::LR, true, S1, S1>(v, F);
            if (q) {
#pragma unroll
                for (int k = 0; k < R; k++) Xb[po(k * Q)] = v[k];
            } else {
#pragma unroll
                for (int k = 0; k < R; k++) keep[k * Q + t] = v[k];
            }
        }
        sync_global();
        // a run in each half of the coefficients
        constexpr int H = g::M / 2;
        double b0 = 0.0, b1 = 0.0, b2 = 0.0;        // what the lower half's last run hands on
#pragma unroll
        for (int h2 = 0; h2 < 2; h2++) {
            double z[C], o0 = 0.0, o1 = 0.0;
            const bool in = h2 * H + uniform(t & ~63) * C <= live + 2;
            const double *r0 = keep + h2 * H + t * C;
            oc = 0.0;
            if (in)
                run_digits<S, C, LM>(z, [&](int i) { return r0[i]; },
                                  [&](int i) { return Xr[po(h2 * H) + po(i)]; }, mul, o0, o1, oc);
            hand_on(o0, o1, oc);
            sync_block<LM>();
            take(t == 0);
            if (t == 0) { i0 = b0; i1 = b1; ic = b2; }
            constexpr int E = 3 * (g::THREADS / 64) - 3;
            b0 = bnd[E]; b1 = bnd[E + 1]; b2 = bnd[E + 2];
            if (in) {
                run_finish<S, C>(z, i0, i1, ic, oc);
#pragma unroll
                for (int i = 0; i < C; i++) Xr[po(h2 * H) + po(i)] = z[i];
            }
            sync_block<LM>();
        }
    }
    sync_block<LM>();
}

// X: lds_words(), X[LDS] zero.  mul x^2 (TOP) or mul x^2 R^-1 modulo N, x at limbs [off, off + Lw), left at
// limbs [0, Lw) or [Lw, 2 Lw).  DENSE: Nt the transform of N'.  park: global
// memory, 2 Lw + 2 words (DENSE), then 3 M/2 (SEQ classes).
template <int LM>
PF_DEC_FN void square_step(double *X, double *bnd, const Fp &F, const Form &f, const Terms &u, const double *tab, int off,
                           double mul, const Twid<LM> *h, const double *Nt, double *park)
{
    const int Lw = u.Lw;
    // one product instance: a second one would double the code and its registers
#pragma clang loop unroll(disable)
    for (int second = 0;; second = 1) {
        product<Base10, LM>(X, bnd, F, Lw, second ? 0 : off, second ? Lw : 2 * Lw, tab, second ? 1.0 : mul, h,
                    second ? Nt : nullptr, park + 2 * Lw + 2);
        if (second || u.mode != DENSE) break;
        if constexpr (park_lds<LM>()) {
            for (int i = tid(); i <= 2 * Lw; i += G<LM>::THREADS) X[G<LM>::LDS + 2 + i] = X[pd(i)];
        } else {
            for (int i = tid(); i <= 2 * Lw; i += G<LM>::THREADS) park[i] = X[pd(i)];
        }
        sync_block<LM>();
    }
    if (u.mode == DENSE) {
        if constexpr (park_lds<LM>()) {
            dense_tail<LM>(X, G<LM>::LDS, X + G<LM>::LDS + 2, f, u, tid());
        } else {
            sync_global();
            dense_tail<LM>(X, G<LM>::LDS, park, f, u, tid());
        }
    } else {
        fold<LM>(X, G<LM>::LDS, f, u, tid());
    }
}

// ---- any odd modulus ------------------------------------------------------------
// The same transforms in base 2^43 carry the Montgomery step of a modulus
// without structure: T = mul x y, m = T N' mod R, (T + m N) / R with R =
// 2^(43 Lw), three products, digits balanced as above.  R is at least 2^16
// times the 2^(24 L) of the 24-bit form (sh = 43 Lw - 24 L), so that |x| stays
// below N whatever the base (below 512) multiplied in.
struct Gen {
    int32_t lm, Lw, sh, L;
};
PF_DEC_HD Gen gen_of(int L)
{
    Gen g = {0, 0, 0, L};
    g.Lw = (24 * L + 16 + Base2::BITS - 1) / Base2::BITS;
    g.sh = Base2::BITS * g.Lw - 24 * L;
    for (int lm = MIN_LM; lm <= MAX_LM && !g.lm; lm++)
        if ((1 << lm) >= 2 * g.Lw + 4) g.lm = lm;
    return g;
}

// Limb i (43 bits, balanced) of 2^sh times the number of n 24-bit limbs at v
// (one per word W).
template <class W>
PF_DEC_FN double gen_limb(const W *v, int n, int sh, int i)
{
    auto raw = [&](int k) {
        const int at = 43 * k - sh;                     // first bit, maybe below 0
        if (at + 43 <= 0) return 0ull;
        const int j = at >= 0 ? at / 24 : -1, o = at - 24 * j;      // o in [0, 24), or from limb -1
        unsigned long long x = 0;
        const unsigned long long a0 = j >= 0 && j < n ? v[j] & 0xFFFFFF : 0, a1 = j + 1 < n ? v[j + 1] & 0xFFFFFF : 0,
                                 a2 = j + 2 < n ? v[j + 2] & 0xFFFFFF : 0;
        if (at >= 0) {
            x = (a0 >> o) | (a1 << (24 - o)) | (a2 << (48 - o));
        } else {                                        // starts -at bits below the number
            const int d = -at;                          // 1 .. 42
            const unsigned long long b0 = n > 0 ? v[0] & 0xFFFFFF : 0, b1 = n > 1 ? v[1] & 0xFFFFFF : 0;
            x = (b0 << d) | (d < 19 ? b1 << (24 + d) : 0ull);
        }
        return x & ((1ull << 43) - 1);
    };
    const unsigned long long x = raw(i), y = i > 0 ? raw(i - 1) : 0ull, h = 1ull << 42;
    return (double)(long long)x - (x >= h ? Base2::B : 0.0) + (y >= h ? 1.0 : 0.0);
}

// x at X's limbs [off, off + Lw) -> mul x^2 R^-1, or mul x y R^-1 for the
// transform y0 of y, at limbs [Lw, 2 Lw).  Np, Nt: transforms of N' and N.
// park: global memory, 2 Lw + 2 words (from class 13), then 3 M/2 (SEQ).
template <int LM>
PF_DEC_FN void mont_step(double *X, double *bnd, const Fp &F, int Lw, const double *tab, int off, double mul,
                         const Twid<LM> *h, const double *y0, const double *Np, const double *Nt, double *park)
{
    constexpr int W = G<LM>::THREADS / 64;
    double *Tl = X + G<LM>::LDS + 2;
#pragma clang loop unroll(disable)
    for (int k = 0; k < 3; k++) {
        product<Base2, LM>(X, bnd, F, Lw, k ? 0 : off, k == 1 ? Lw : 2 * Lw, tab, k ? 1.0 : mul, h,
                           k == 0 ? y0 : k == 1 ? Np : Nt, park + 2 * Lw + 2);
        if (k) continue;
        for (int i = Lw - 1 + tid(); i < 2 * Lw; i += G<LM>::THREADS) {
            if constexpr (park_lds<LM>()) Tl[i] = X[pd(i)];
            else park[i] = X[pd(i)];
        }
        sync_block<LM>();
    }
    if constexpr (!park_lds<LM>()) sync_global();
    // the limbs below Lw come to zero (as in dense_tail); lane 0 gives the carry
    constexpr int NI = (G<LM>::M / 2 + 63 * W - 1) / (63 * W);
    const int t = tid(), lane = t & 63, wave = uniform(t >> 6);
    double out[NI];
#pragma unroll
    for (int n = 0; n < NI; n++) {
        const int i = Lw - 1 + (wave + n * W) * 63 + lane;
        double acc = 0.0;
        if (i < 2 * Lw) {
            if constexpr (park_lds<LM>()) acc = X[pd(i)] + Tl[i];
            else acc = X[pd(i)] + park[i];
        }
        const double c = rint_(acc * Base2::IB);
        out[n] = fma_(-c, Base2::B, acc) + lane_up(c);
    }
    sync_block<LM>();
#pragma unroll
    for (int n = 0; n < NI; n++) {
        const int i = Lw - 1 + (wave + n * W) * 63 + lane;
        if (lane > 0 && i < 2 * Lw) X[pd(i)] = out[n];
    }
    sync_block<LM>();
}

// The transform of the n digits at X's limbs [0, n), per prime M words at out.
template <int LM>
PF_DEC_FN void transform(double *X, int n, const double *tab, double *out)
{
    using g = G<LM>;
    constexpr int R = g::R, Q = g::M / R, TS = tab_size<LM>();
    const int t = tid(), tp = t & (g::TP - 1);
    double x[R / 2], v[R];
#pragma unroll
    for (int k = 0; k < R / 2; k++) {
        const int i = tp + k * Q;
        x[k] = i < n ? X[pd(i)] : 0.0;
    }
    for (int s = 0; s < (g::SEQ ? 2 : 1); s++) {
        const int q = g::SEQ ? s : t / g::TP;
        const Fp F = prime_of(q);
        double *Y = g::SEQ ? X : X + q * g::XP, *Yb = Y + pd(tp);
#pragma unroll
        for (int k = 0; k < R / 2; k++) v[k] = x[k];
        sync_block<LM>();
        dft<g::LR, false, 10, 10, true>(v, F);
#pragma unroll
        for (int k = 0; k < R; k++) Yb[po(k * Q)] = v[k];
        sync_block<LM>();
        middle<LM, false>(Y, F, tab + 2 * q * TS, nullptr, tp, nullptr, nullptr, out + q * g::M);
    }
}

} } // namespace mr::dec
