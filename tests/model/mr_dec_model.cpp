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
extern "C" int dec_choose(long long D, long long lo, long long hi, int *mode)
{
    const Choice c = choose(D, lo, hi);
    *mode = c.mode;
    return c.lm;
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
