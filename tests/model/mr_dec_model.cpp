// Host model of the base-10^13 squaring (mr_dec_core.h): one std::thread per
// lane, barriers for the block's and the wave's hand-offs.
#include <barrier>
#include <memory>
#include <string.h>
#include <thread>
#include <vector>
#define PF_DEC_HOST
#include "mr_dec_core.h"
namespace mr { namespace dec {
static thread_local int t_id;
static std::barrier<> *g_block;
static std::vector<std::unique_ptr<std::barrier<>>> *g_wave;
static double g_lane[1024];
int tid() { return t_id; }
void sync_waves() { g_block->arrive_and_wait(); }
void sync_global() { sync_waves(); }
void sync_wave() { (*g_wave)[t_id >> 6]->arrive_and_wait(); }
double lane_up(double x)
{
    g_lane[t_id] = x;
    sync_wave();
    const double r = t_id & 63 ? g_lane[t_id - 1] : -1e300;
    sync_wave();
    return r;
}
} }
using namespace mr::dec;
template <int LM>
static void run(const Form &f, double *dig, const double *mul, int steps)
{
    using g = G<LM>;
    std::vector<double> X(lds_words<LM>(), 1e300), bnd(3 * (g::THREADS / 64) + 3), tab(4 * tab_size<LM>()), Y(g::LDS + 2), Nt(2 * g::M), park(3 * g::M + 4);
    build_tables(LM, tab.data());
    for (int i = 0; i < f.Lw; i++) X[pd(i)] = dig[i];
    X[g::LDS] = Y[g::LDS] = 0.0;
    std::barrier<> blk(g::THREADS);
    std::vector<std::unique_ptr<std::barrier<>>> wv;
    for (int w = 0; w < g::THREADS / 64; w++) wv.emplace_back(new std::barrier<>(64));
    g_block = &blk;
    g_wave = &wv;
    std::vector<std::thread> th;
    for (int t = 0; t < g::THREADS; t++)
        th.emplace_back([&, t] {
            t_id = t;
            int off = 0;
            Terms u;
            load_terms(u, f);
            Twid<LM> h[hoisted<LM>() ? 2 : 1];
            if (hoisted<LM>()) {
                const int q = t / g::TP;
                for (int i = 0; i < (hoisted<LM>() ? 2 : 0); i++)
                    h[i].load(tab.data() + (2 * q + i) * tab_size<LM>(), t & (g::TP - 1));
            }
            if (f.mode == DENSE) {                  // N' and its transform
                for (int i = t; i < g::M; i += g::THREADS) Y[pd(i)] = i ? 0.0 : 1.0;
                sync_waves();
                fold<LM>(Y.data(), g::LDS, f, u, t, park.data());
                sync_waves();
                for (int i = t; i < f.Lw; i += g::THREADS) Y[pd(i)] = park[i];
                sync_waves();
                transform<LM>(Y.data(), f.Lw, tab.data(), Nt.data());
                sync_waves();
            }
            for (int s = 0; s < steps; s++) {
                square_step<LM>(X.data(), bnd.data(), prime_of(t / g::TP), f, u, tab.data(), off, mul[s], h, Nt.data(), park.data());
                off = f.mode == TOP ? 0 : f.Lw;
            }
        });
    for (auto &x : th) x.join();
    const int off = f.mode == TOP || !steps ? 0 : f.Lw;
    for (int i = 0; i < f.Lw; i++) dig[i] = X[pd(off + i)];
}
// mul x y R^-1 mod N (y == nullptr: x^2) in base 2^43, all operands as Lw
// balanced digits; np: N' = -N^-1 mod R.
template <int LM>
static void run_gen(int Lw, const double *N, const double *np, const double *x, const double *y, double mul,
                    double *out)
{
    using g = G<LM>;
    std::vector<double> X(lds_words<LM>(), 1e300), bnd(3 * (g::THREADS / 64) + 3), tab(4 * tab_size<LM>());
    std::vector<double> tr[3], park(3 * g::M + 4);
    for (auto &t : tr) t.resize(2 * g::M);
    build_tables(LM, tab.data());
    std::barrier<> blk(g::THREADS);
    std::vector<std::unique_ptr<std::barrier<>>> wv;
    for (int w = 0; w < g::THREADS / 64; w++) wv.emplace_back(new std::barrier<>(64));
    g_block = &blk;
    g_wave = &wv;
    std::vector<std::thread> th;
    for (int t = 0; t < g::THREADS; t++)
        th.emplace_back([&, t] {
            t_id = t;
            auto load = [&](const double *v) {
                for (int i = t; i < Lw; i += g::THREADS) X[pd(i)] = v[i];
                sync_waves();
            };
            const double *src[3] = {N, np, y};
            for (int k = 0; k < (y ? 3 : 2); k++) {
                load(src[k]);
                transform<LM>(X.data(), Lw, tab.data(), tr[k].data());
                sync_waves();
            }
            Twid<LM> h[hoisted<LM>() ? 2 : 1];
            for (int i = 0; i < (hoisted<LM>() ? 2 : 0); i++)
                h[i].load(tab.data() + (2 * (t / g::TP) + i) * tab_size<LM>(), t & (g::TP - 1));
            load(x);
            mont_step<LM>(X.data(), bnd.data(), prime_of(t / g::TP), Lw, tab.data(), 0, mul, h,
                          y ? tr[2].data() : nullptr, tr[1].data(), tr[0].data(), park.data());
        });
    for (auto &x2 : th) x2.join();
    for (int i = 0; i < Lw; i++) out[i] = X[pd(Lw + i)];
}
extern "C" int gen_shape(int L, int *lw, int *sh)
{
    const Gen g = gen_of(L);
    *lw = g.Lw;
    *sh = g.sh;
    return g.lm;
}
extern "C" double gen_digit(const uint32_t *v, int n, int sh, int i) { return gen_limb(v, n, sh, i); }
extern "C" int gen_mont(int lm, int Lw, const double *N, const double *np, const double *x, const double *y,
                        double mul, double *out)
{
    switch (lm) {
    case 7: run_gen<7>(Lw, N, np, x, y, mul, out); break;
    case 8: run_gen<8>(Lw, N, np, x, y, mul, out); break;
    case 9: run_gen<9>(Lw, N, np, x, y, mul, out); break;
    case 10: run_gen<10>(Lw, N, np, x, y, mul, out); break;
    case 11: run_gen<11>(Lw, N, np, x, y, mul, out); break;
    case 12: run_gen<12>(Lw, N, np, x, y, mul, out); break;
    case 13: run_gen<13>(Lw, N, np, x, y, mul, out); break;
    case 14: run_gen<14>(Lw, N, np, x, y, mul, out); break;
    default: return 0;
    }
    return 1;
}
extern "C" int dec_choose(long long D, long long lo, long long hi, int *mode)
{
    const Choice c = choose(D, lo, hi);
    *mode = c.mode;
    return c.lm;
}
// 1 when the digits are m N + add
extern "C" int dec_equals(const long long *terms, int nterm, long long D, int lm, int mode, const double *dig,
                          int m, int add)
{
    Form f;
    std::vector<int64_t> t(terms, terms + 2 * nterm);
    make_form(t.data(), nterm, D, lm, mode, f);
    Share sh[MAX_TERMS];
    for (int k = 1; k < f.nt; k++) sh[k] = share_of(f, k);
    return equals(dig, f, sh, m, add);
}
// terms: nterm (coef, exp) pairs; dig: room for 8192; returns Lw (0: not handled)
extern "C" int dec_square(const long long *terms, int nterm, long long D, int lm, int mode, double *dig,
                          const double *mul, int steps)
{
    Form f;
    std::vector<int64_t> t(terms, terms + 2 * nterm);
    make_form(t.data(), nterm, D, lm, mode, f);
    if (!f.lm) return 0;
    switch (f.lm) {
    case 7: run<7>(f, dig, mul, steps); break;
    case 8: run<8>(f, dig, mul, steps); break;
    case 9: run<9>(f, dig, mul, steps); break;
    case 10: run<10>(f, dig, mul, steps); break;
    case 11: run<11>(f, dig, mul, steps); break;
    case 12: run<12>(f, dig, mul, steps); break;
    case 13: run<13>(f, dig, mul, steps); break;
    case 14: run<14>(f, dig, mul, steps); break;
    default: return 0;
    }
    return f.Lw;
}
// dig (2 Lw): x -> m and (x + m N) / R, limb by limb; returns Lw
extern "C" int dec_solve(const long long *terms, int nterm, long long D, double *dig)
{
    Form f;
    std::vector<int64_t> t(terms, terms + 2 * nterm);
    make_form(t.data(), nterm, D, MAX_LM, DENSE, f);
    std::vector<double> T(pd(2 * f.Lw) + 1);
    for (int i = 0; i < 2 * f.Lw; i++) T[pd(i)] = dig[i];
    solve(T.data(), f, true);
    for (int i = 0; i < 2 * f.Lw; i++) dig[i] = T[pd(i)];
    return f.Lw;
}
