// mr_dec.hip -- exponentiation of search-form candidates in base 10^13
// (mr_dec_core.h): one workgroup owns one candidate for a chunk of squarings,
// its digits and both transforms in LDS.
#include "mr_dec.h"
#include <mutex>
#include <vector>

namespace mr { namespace dec {

namespace {

__device__ __forceinline__ int slot_of(const Args &A)
{
    return A.list ? A.list[blockIdx.x] : (int)blockIdx.x;
}

template <int LM>
__device__ __forceinline__ void copy_form(Form &f, const Form *src)
{
    static_assert(sizeof(Form) % 4 == 0, "copied by words");
    for (int i = threadIdx.x; i < (int)(sizeof(Form) / 4); i += G<LM>::THREADS)
        ((uint32_t *)&f)[i] = ((const uint32_t *)src)[i];
}

// Left-to-right binary powering: a squaring per exponent bit, times the base
// (below 512, folded into the digits' carry step) where the bit is set.
// Bit i of d is bit i + s of N.
template <int LM>
__global__ __launch_bounds__(G<LM>::THREADS) void exp_kernel(Args A, const double *__restrict__ tab, int steps)
{
    __shared__ double X[lds_words<LM>()];
    __shared__ double bnd[3 * (G<LM>::THREADS / 64)];
    __shared__ Form f;
    const int c = slot_of(A);
    if (A.run && !A.run[c]) return;
    if (A.path[c] != LM || !A.alive[c] || A.pre[c]) return;
    const int s = A.sval[c];
    int bp = A.bitpos[c];
    if (bp < s) return;
    copy_form<LM>(f, A.form + c);
    __syncthreads();
    const int Lw = f.Lw;
    const double base = (double)A.base[c];
    const uint32_t *Nl = A.N + (size_t)c * A.nstride;
    double *dig = A.dig + (size_t)c * A.dstride;
    const double *Nt = A.Nt + (size_t)c * A.tstride;
    double *park = A.park + (size_t)c * A.pstride;
    for (int i = threadIdx.x; i < Lw; i += G<LM>::THREADS) X[pd(i)] = dig[i];
    if (threadIdx.x == 0) X[G<LM>::LDS] = 0.0;
    const int out = f.mode == TOP ? 0 : Lw;
    int off = 0;
    Terms u;
    load_terms(u, f);
    const int q0 = threadIdx.x / G<LM>::TP;
    const Fp F = prime_of(G<LM>::TP >= 64 ? uniform(q0) : q0);
    Twid<LM> h[hoisted<LM>() ? 2 : 1];
    if constexpr (hoisted<LM>()) {
        const int q = threadIdx.x / G<LM>::TP, t = threadIdx.x & (G<LM>::TP - 1);
        h[0].load(tab + 2 * q * tab_size<LM>(), t);
        h[1].load(tab + (2 * q + 1) * tab_size<LM>(), t);
    }
    __syncthreads();
    // a limb of exponent bits at a time: loaded in every step, the barriers of
    // the step waited for it
    uint32_t bits = Nl[bp / 24] << (31 - bp % 24);
    for (int k = 0; k < steps && bp >= s; k++, bp--) {
        const uint32_t bit = bits >> 31;
        bits <<= 1;
        if (bp % 24 == 0 && bp) bits = Nl[bp / 24 - 1] << 8;
        square_step<LM>(X, bnd, F, f, u, tab, off, bit ? base : 1.0, h, Nt, park);
        off = out;
    }
    for (int i = threadIdx.x; i < Lw; i += G<LM>::THREADS) dig[i] = X[pd(off + i)];
    if (threadIdx.x == 0) A.bitpos[c] = bp;
}

// One thread: digits at X[pd(off + i)], i < n, carried into [0, B); returns
// what leaves the top (0 or -1 for values of magnitude below B^n).
__device__ double carry_all(double *X, int off, int n)
{
    constexpr int U = 8;
    double c = 0.0;
    for (int i0 = 0; i0 < n; i0 += U) {
        double v[U];
#pragma unroll
        for (int i = 0; i < U; i++) v[i] = i0 + i < n ? X[pd(off + i0 + i)] : 0.0;
#pragma unroll
        for (int i = 0; i < U; i++)
            if (i0 + i < n) {
                const double x = v[i] + c;
                double q = __builtin_floor(x * IB), r = fma_(-q, B, x);
                if (r < 0.0) { r += B; q -= 1.0; }
                if (r >= B) { r -= B; q += 1.0; }
                v[i] = r;
                c = q;
            }
#pragma unroll
        for (int i = 0; i < U; i++)
            if (i0 + i < n) X[pd(off + i0 + i)] = v[i];
    }
    return c;
}

// The value at X's limbs [off, off + Lw) (|value| < 0.6 of the modulus) as
// digits of a number in [0, 1.1 N) congruent to it mod N.  One thread.
__device__ void canonical(double *X, int off, const Form &f)
{
    const int Lw = f.Lw;
    if (carry_all(X, off, Lw) < 0.0) {          // negative: plus the modulus
        if (f.mode != TOP) X[pd(off)] -= 1.0;
        for (int k = 0; k < f.nt; k++) {
            const Term &t = f.t[k];
            const double c = f.mode == TOP ? -t.c : t.c, h = __builtin_trunc(c / t.tc);
            const int E = off + t.E + (f.mode == TOP ? Lw : 0);
            X[pd(E)] += (c - h * t.tc) * t.ts;
            if (h != 0.0) X[pd(E + 1)] += h;
        }
        (void)carry_all(X, off, Lw);
    }
    if (f.mode == TOP && f.z) {                 // modulo N 10^z -> modulo N
        double w = 1.0;
        for (int i = 0; i < DIGITS - f.z; i++) w *= 10.0;
        double &top = X[pd(off + Lw - 1)];
        const double h = __builtin_floor(top / w);
        top -= h * w;
        for (int k = 0; k < f.nt; k++) {
            const Term &t = f.t[k];
            const int e = DIGITS * (t.E + Lw) + t.s - f.z, E = e / DIGITS, s = e % DIGITS;
            double ts = 1.0;
            for (int i = 0; i < s; i++) ts *= 10.0;
            // h c < 10^18 at limb E, s digits up
            const unsigned long long v = (unsigned long long)h * (unsigned long long)t.c;
            const unsigned long long tc = (unsigned long long)(B / ts), lim = (unsigned long long)B;
            X[pd(off + E)] += (double)(v % tc) * ts;
            X[pd(off + E + 1)] += (double)(v / tc % lim);
            if (v / tc >= lim) X[pd(off + E + 2)] += (double)(v / tc / lim);
        }
        (void)carry_all(X, off, Lw);
    }
}

template <int LM>
__global__ __launch_bounds__(G<LM>::THREADS) void norm_kernel(Args A)
{
    __shared__ double X[G<LM>::XP + 2];
    __shared__ Form f;
    const int c = slot_of(A);
    if (A.path[c] != LM || A.pre[c]) return;
    copy_form<LM>(f, A.form + c);
    __syncthreads();
    const int Lw = f.Lw, t = threadIdx.x;
    const double *dig = A.dig + (size_t)c * A.dstride;
    for (int i = t; i < G<LM>::M; i += G<LM>::THREADS) X[pd(i)] = i < Lw ? dig[i] : 0.0;
    if (t == 0) X[G<LM>::XP] = 0.0;
    __syncthreads();
    const int off = f.mode == TOP ? 0 : Lw;
    Terms u;
    load_terms(u, f);
    if (f.mode == DENSE && f.gap < 1) {                        // out of Montgomery form
        if (t == 0) solve(X, f, true);
    } else if (f.mode != TOP) {
        fold<LM>(X, G<LM>::XP, f, u, t);
    }
    __syncthreads();
    if (t == 0) canonical(X, off, f);
    __syncthreads();
    double *out = (double *)(A.scr + (size_t)c * A.sstride);
    for (int i = t; i < Lw; i += G<LM>::THREADS) out[i] = X[pd(off + i)];
}

// N' = -N^-1 mod B^Lw: the limbs that BOTTOM's rounds clear from T = 1 (1 + N' N
// = 0 mod B^Lw), and its transform.
template <int LM>
__global__ __launch_bounds__(G<LM>::THREADS) void prepare_kernel(Args A, const double *__restrict__ tab)
{
    __shared__ double X[G<LM>::LDS + 2];
    __shared__ Form f;
    const int c = slot_of(A), t = threadIdx.x;
    if (A.form[c].lm != LM || A.form[c].mode != DENSE) return;
    copy_form<LM>(f, A.form + c);
    for (int i = t; i < G<LM>::M; i += G<LM>::THREADS) X[pd(i)] = i == 0 ? 1.0 : 0.0;
    if (t == 0) X[G<LM>::LDS] = 0.0;
    __syncthreads();
    double *rec = A.park + (size_t)c * A.pstride;
    Terms u;
    load_terms(u, f);
    fold<LM>(X, G<LM>::LDS, f, u, t, rec);
    __syncthreads();
    for (int i = t; i < f.Lw; i += G<LM>::THREADS) X[pd(i)] = rec[i];
    __syncthreads();
    transform<LM>(X, f.Lw, tab, A.Nt + (size_t)c * A.tstride);
}

// Digits of 2^sh times a number of 24-bit limbs into X's limbs [0, Lw).
template <int LM, class W>
__device__ __forceinline__ void gen_load(double *X, const W *v, int L, int sh, int Lw)
{
    for (int i = threadIdx.x; i < Lw; i += G<LM>::THREADS) X[pd(i)] = gen_limb(v, L, sh, i);
    __syncthreads();
}

template <int LM>
struct GenSlot {
    double *Nt, *Np, *One, *OneR, *Y, *park;
    __device__ GenSlot(const GenArgs &A, int c)
    {
        constexpr int P = 2 * G<LM>::M;
        Nt = A.tab + (size_t)c * 5 * P;
        Np = Nt + P;
        One = Np + P;
        OneR = One + P;
        Y = OneR + P;
        park = A.park + (size_t)c * A.pstride;
    }
};

template <int LM>
__device__ __forceinline__ void load_twid(Twid<LM> (&h)[hoisted<LM>() ? 2 : 1], const double *tab)
{
    if constexpr (hoisted<LM>()) {
        const int q = threadIdx.x / G<LM>::TP, t = threadIdx.x & (G<LM>::TP - 1);
        h[0].load(tab + 2 * q * tab_size<LM>(), t);
        h[1].load(tab + (2 * q + 1) * tab_size<LM>(), t);
    }
}

// The transforms a modulus needs: N, 2^(24 L) and R mod N, and N' = -N^-1 mod
// R = 2^(43 Lw), by one Newton step y (2 + N y) from the N' mod 2^(24 L) at scr.
template <int LM>
__global__ __launch_bounds__(G<LM>::THREADS) void gen_prepare_kernel(GenArgs A, const double *__restrict__ tab)
{
    __shared__ double X[lds_words<LM>()];
    __shared__ double bnd[3 * (G<LM>::THREADS / 64)];
    const int c = blockIdx.x, L = A.g.L, Lw = A.g.Lw;
    if (A.pre[c]) return;
    GenSlot<LM> S(A, c);
    const int q0 = threadIdx.x / G<LM>::TP;
    const Fp F = prime_of(G<LM>::TP >= 64 ? uniform(q0) : q0);
    Twid<LM> h[hoisted<LM>() ? 2 : 1];
    load_twid<LM>(h, tab);
    if (threadIdx.x == 0) X[G<LM>::LDS] = 0.0;
    double *keep = S.park + 2 * Lw + 2;
    gen_load<LM>(X, A.N + (size_t)c * A.nstride, L, 0, Lw);
    transform<LM>(X, Lw, tab, S.Nt);
    __syncthreads();
    gen_load<LM>(X, A.one + (size_t)c * A.nstride, L, 0, Lw);
    transform<LM>(X, Lw, tab, S.One);
    __syncthreads();
    const uint32_t *y = A.scr + (size_t)c * A.sstride;
    gen_load<LM>(X, y + A.sstride / 2, L, 0, Lw);
    transform<LM>(X, Lw, tab, S.OneR);
    __syncthreads();
    gen_load<LM>(X, y, L, 0, Lw);
    product<Base2, LM>(X, bnd, F, Lw, 0, Lw, tab, 1.0, h, S.Nt, keep);
    if (threadIdx.x == 0) X[0] += 2.0;
    __syncthreads();
    transform<LM>(X, Lw, tab, S.Y);
    __syncthreads();
    gen_load<LM>(X, y, L, 0, Lw);
    product<Base2, LM>(X, bnd, F, Lw, 0, Lw, tab, 1.0, h, S.Y, keep);
    transform<LM>(X, Lw, tab, S.Np);
}

template <int LM>
__global__ __launch_bounds__(G<LM>::THREADS) void gen_exp_kernel(GenArgs A, const double *__restrict__ tab, int steps)
{
    __shared__ double X[lds_words<LM>()];
    __shared__ double bnd[3 * (G<LM>::THREADS / 64)];
    const int c = blockIdx.x, L = A.g.L, Lw = A.g.Lw;
    if (!A.alive[c] || A.pre[c] || A.base[c] > (uint32_t)MAX_BASE || (A.path && A.path[c])) return;
    const int s = A.sval[c];
    int bp = A.bitpos[c];
    if (bp < s) return;
    const double base = (double)A.base[c];
    const uint32_t *Nl = A.N + (size_t)c * A.nstride;
    GenSlot<LM> S(A, c);
    const int q0 = threadIdx.x / G<LM>::TP;
    const Fp F = prime_of(G<LM>::TP >= 64 ? uniform(q0) : q0);
    Twid<LM> h[hoisted<LM>() ? 2 : 1];
    load_twid<LM>(h, tab);
    // x 2^(24 L) 2^sh = x R, times R mod N: x R below N
    gen_load<LM>(X, A.res + (size_t)c * A.nstride, L, A.g.sh, Lw);
    mont_step<LM>(X, bnd, F, Lw, tab, 0, 1.0, h, S.OneR, S.Np, S.Nt, S.park);
    uint32_t bits = Nl[bp / 24] << (31 - bp % 24);
    bool last = false;
    for (int k = 0; !last; k++) {
        last = k == steps || bp < s;            // then times 2^(24 L) mod N: x R -> x 2^(24 L)
        const uint32_t bit = bits >> 31;
        mont_step<LM>(X, bnd, F, Lw, tab, Lw, bit && !last ? base : 1.0, h, last ? S.One : nullptr, S.Np, S.Nt,
                      S.park);
        bits <<= 1;
        if (bp % 24 == 0 && bp) bits = Nl[bp / 24 - 1] << 8;
        if (!last) bp--;
    }
    double *dig = A.dig + (size_t)c * A.dstride;
    for (int i = threadIdx.x; i < Lw; i += G<LM>::THREADS) dig[i] = X[pd(Lw + i)];
    if (threadIdx.x == 0) { A.bitpos[c] = bp; A.flag[c] = 1; }
}

template <int LM>
__global__ __launch_bounds__(G<LM>::THREADS) void gen_mul_kernel(GenArgs A, const double *__restrict__ tab,
                                                                 const uint64_t *a, const uint64_t *b, int ld)
{
    __shared__ double X[lds_words<LM>()];
    __shared__ double bnd[3 * (G<LM>::THREADS / 64)];
    const int c = blockIdx.x, L = A.g.L, Lw = A.g.Lw;
    if (A.pre[c]) return;
    GenSlot<LM> S(A, c);
    const int q0 = threadIdx.x / G<LM>::TP;
    const Fp F = prime_of(G<LM>::TP >= 64 ? uniform(q0) : q0);
    Twid<LM> h[hoisted<LM>() ? 2 : 1];
    load_twid<LM>(h, tab);
    if (b) {
        gen_load<LM>(X, b + (size_t)c * ld, L, 0, Lw);
        transform<LM>(X, Lw, tab, S.Y);
        __syncthreads();
    }
    // 2^sh a b R^-1 = a b 2^(-24 L)
    gen_load<LM>(X, a + (size_t)c * ld, L, b ? A.g.sh : A.g.sh / 2, Lw);
    mont_step<LM>(X, bnd, F, Lw, tab, 0, !b && (A.g.sh & 1) ? 2.0 : 1.0, h, b ? S.Y : nullptr, S.Np, S.Nt, S.park);
    double *dig = A.dig + (size_t)c * A.dstride;
    for (int i = threadIdx.x; i < Lw; i += G<LM>::THREADS) dig[i] = X[pd(Lw + i)];
    if (threadIdx.x == 0) A.flag[c] = 1;
}

__global__ void form_kernel(const int32_t *list, int n, const int64_t *terms, int nterm,
                            const int32_t *choice, Form *form, uint32_t *err)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Form &f = form[list ? list[i] : i];
    const int32_t *ch = choice + 3 * i;
    if (ch[1] == 0) { f.lm = 0; return; }
    make_form(terms + (size_t)i * 2 * nterm, nterm, ch[0], ch[1], ch[2], f);
    if (f.lm != ch[1]) atomicOr(err, 4u);
}

template <class F>
void by_class(int lm, F f)
{
    switch (lm) {
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 11: f(std::integral_constant<int, 11>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 13: f(std::integral_constant<int, 13>{}); break;
    case 14: f(std::integral_constant<int, 14>{}); break;
    }
}

std::mutex g_mu;
double *g_tab[64][MAX_LM + 1];

} // namespace

const double *tables(int device, int lm)
{
    if (device < 0 || device >= 64 || lm < MIN_LM || lm > MAX_LM) return nullptr;
    std::lock_guard<std::mutex> lk(g_mu);
    double *&t = g_tab[device][lm];
    if (!t) {
        const size_t n = 4 * (size_t)tab_size_rt(lm);
        std::vector<double> h(n);
        build_tables(lm, h.data());
        double *d = nullptr;
        if (hipMalloc(&d, n * sizeof(double)) != hipSuccess) return nullptr;
        if (hipMemcpy(d, h.data(), n * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(d);
            return nullptr;
        }
        t = d;
    }
    return t;
}

void launch_exp(int lm, const Args &A, const double *tab, int n, int steps, hipStream_t st)
{
    by_class(lm, [&](auto c) {
        constexpr int LM = decltype(c)::value;
        exp_kernel<LM><<<n, G<LM>::THREADS, 0, st>>>(A, tab, steps);
    });
}

void launch_prepare(int lm, const Args &A, const double *tab, int n, hipStream_t st)
{
    by_class(lm, [&](auto c) {
        constexpr int LM = decltype(c)::value;
        prepare_kernel<LM><<<n, G<LM>::THREADS, 0, st>>>(A, tab);
    });
}

void launch_norm(int lm, const Args &A, int n, hipStream_t st)
{
    by_class(lm, [&](auto c) {
        constexpr int LM = decltype(c)::value;
        norm_kernel<LM><<<n, G<LM>::THREADS, 0, st>>>(A);
    });
}

void launch_gen_prepare(const GenArgs &A, const double *tab, int n, hipStream_t st)
{
    by_class(A.g.lm, [&](auto c) {
        constexpr int LM = decltype(c)::value;
        gen_prepare_kernel<LM><<<n, G<LM>::THREADS, 0, st>>>(A, tab);
    });
}

void launch_gen_exp(const GenArgs &A, const double *tab, int n, int steps, hipStream_t st)
{
    by_class(A.g.lm, [&](auto c) {
        constexpr int LM = decltype(c)::value;
        gen_exp_kernel<LM><<<n, G<LM>::THREADS, 0, st>>>(A, tab, steps);
    });
}

void launch_gen_mul(const GenArgs &A, const double *tab, int n, const uint64_t *a, const uint64_t *b, int ld,
                    hipStream_t st)
{
    by_class(A.g.lm, [&](auto c) {
        constexpr int LM = decltype(c)::value;
        gen_mul_kernel<LM><<<n, G<LM>::THREADS, 0, st>>>(A, tab, a, b, ld);
    });
}

void launch_form(const int32_t *list, int n, const int64_t *terms, int nterm, const int32_t *choice,
                 Form *form, uint32_t *err, hipStream_t st)
{
    form_kernel<<<(n + 63) / 64, 64, 0, st>>>(list, n, terms, nterm, choice, form, err);
}

} } // namespace mr::dec
