// Host emulation of the mixed-radix transforms of chapsim1.0_amd/csrc/chs_fftg.h: the threads of
// a block run as threads and meet at a barrier at every __syncthreads.  Each length given is
// checked with both radix orders, both directions and both ends of the line in LDS or in memory
// against a long-double DFT; prints one line per length and exits non-zero on a failure.
#define CHS_HOST_EMU 1
#define __device__
#define __forceinline__ inline
#define __restrict__

#include <barrier>
#include <cmath>
#include <cstdio>
#include <random>
#include <thread>
#include <vector>

static thread_local std::barrier<> *g_bar = nullptr;
static void __syncthreads() { g_bar->arrive_and_wait(); }
static unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((unsigned long long)a * b) >> 32); }
namespace chs {
void wave_lds_sync() {}
}  // namespace chs

#include "../../chapsim1.0_amd/csrc/chs_fftg.h"

template <typename T, int SIGN, bool FL, bool TL> double run(int n, bool desc, unsigned seed)
{
    using C = chs::cpx<T>;
    const chs::GPlan P = chs::gplan(n, desc);
    if (P.np == 0) return 1e9;
    const std::vector<C> tw = chs::gplan_twiddles<T>(P);
    const int nl = 2;   // lines of the block, and a thread without one
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    std::vector<C> x(nl * n), y(nl * n), lds(nl * P.ls);
    for (auto &e : x) e = {(T)U(rng), (T)U(rng)};
    if (FL)
        for (int l = 0; l < nl; ++l)
            for (int i = 0; i < n; ++i) lds[l * P.ls + i + (i >> P.ps)] = x[l * n + i];
    const int nt = nl * P.tpl + 1;
    std::barrier<> bar(nt);
    std::vector<std::thread> th;
    for (int t = 0; t < nt; ++t)
        th.emplace_back([&, t] {
            g_bar = &bar;
            const int l = t / P.tpl, j = t % P.tpl;
            const bool act = l < nl;
            chs::gfft_lines<T, SIGN, FL, TL>(P, lds.data() + (act ? l : 0) * P.ls, j, act, tw.data(),
                                             [&](int i) { return x[l * n + i]; },
                                             [&](int k, const C &v) { y[l * n + k] = v; });
        });
    for (auto &t : th) t.join();
    double err = 0, big = 0;
    for (int l = 0; l < nl; ++l)
        for (int k = 0; k < n; ++k) {
            long double re = 0, im = 0;
            for (int i = 0; i < n; ++i) {
                const long double a = SIGN * 2.0L * 3.141592653589793238462643383279502884L * ((long long)i * k % n) / n;
                re += x[l * n + i].x * cosl(a) - x[l * n + i].y * sinl(a);
                im += x[l * n + i].x * sinl(a) + x[l * n + i].y * cosl(a);
            }
            const C v = TL ? lds[l * P.ls + k + (k >> P.ps)] : y[l * n + k];
            err = std::fmax(err, std::fmax(std::fabs((double)(v.x - re)), std::fabs((double)(v.y - im))));
            big = std::fmax(big, std::sqrt((double)(re * re + im * im)));
        }
    return err / big;
}

int main(int argc, char **argv)
{
    int bad = 0;
    for (int a = 1; a < argc; ++a) {
        const int n = atoi(argv[a]);
        double e = 0, f = 0;
        for (bool d : {false, true}) {
            e = std::fmax(e, std::fmax(run<double, -1, false, true>(n, d, 1), run<double, 1, true, false>(n, d, 2)));
            e = std::fmax(e, std::fmax(run<double, -1, false, false>(n, d, 3), run<double, 1, true, true>(n, d, 4)));
            f = std::fmax(f, std::fmax(run<float, -1, false, true>(n, d, 5), run<float, 1, true, false>(n, d, 6)));
        }
        const chs::GPlan P = chs::gplan(n, false);
        const bool ok = e < 1e-14 && f < 2e-6;
        bad += !ok;
        std::printf("n %d: %d passes, %d threads, f64 %.2e f32 %.2e %s\n", n, P.np, P.tpl, e, f, ok ? "ok" : "WRONG");
    }
    return bad != 0;
}
