// Complex FFTs of any length 2^a 3^b 5^c for gfx950 whose passes run in registers, radix up to
// 16, with one LDS exchange between passes: most even lengths up to 256 take two passes (150 =
// 10 x 15), longer ones three.  A block owns whole lines; a thread runs at most one butterfly
// per pass: thread j of a line's tpl takes x[j + r n / R], r = 0..R-1 (times the pass's
// twiddles), and stores to (j / Ns) Ns R + j % Ns + r Ns (Stockham order, Ns = product of the
// radices before).  The first pass can take its inputs from memory and the last hand its outputs
// to memory, so a two-pass line crosses LDS once, where the radix 2..5 passes of chs_fft.h cross
// it once per pass with index divisions per element.
#pragma once
#include <vector>

#include "chs_fft.h"
#include "chs_fftr.h"

namespace chs {

// DFT of length R = R1 R2, R1 and R2 coprime, without twiddles (Good-Thomas): input index
// (R2 n1 + R1 n2) mod R, output index by the Chinese remainder theorem.
constexpr int modinv(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if (a * x % m == 1) return x;
    return 1;
}
template <typename T, int R1, int R2> __device__ __forceinline__ void dft_coprime(cpx<T> *v, int sign)
{
    constexpr int R = R1 * R2, c1 = R2 * modinv(R2 % R1, R1), c2 = R1 * modinv(R1 % R2, R2);
    cpx<T> a[R2][R1];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < R1; ++n1) a[n2][n1] = v[(R2 * n1 + R1 * n2) % R];
        bfly<T, R1>(a[n2], sign);
    }
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
        cpx<T> b[R2];
#pragma unroll
        for (int n2 = 0; n2 < R2; ++n2) b[n2] = a[n2][k1];
        bfly<T, R2>(b, sign);
#pragma unroll
        for (int k2 = 0; k2 < R2; ++k2) v[(k1 * c1 + k2 * c2) % R] = b[k2];
    }
}

// In-register DFT of length R, natural order in and out.
template <typename T, int R> __device__ __forceinline__ void gdft(cpx<T> *v, int sign)
{
    if constexpr (R <= 5) bfly<T, R>(v, sign);
    else if constexpr (R == 8 || R == 16) rdft<T, R>(v, sign);
    else if constexpr (R == 6) dft_coprime<T, 2, 3>(v, sign);
    else if constexpr (R == 10) dft_coprime<T, 2, 5>(v, sign);
    else if constexpr (R == 12) dft_coprime<T, 4, 3>(v, sign);
    else if constexpr (R == 15) dft_coprime<T, 3, 5>(v, sign);
    else {
        static_assert(R == 9, "radix");
        // 3 x 3 with the twiddles w9^(n2 k1)
        constexpr T c1 = T(0.76604444311897803520239265055542), s1 = T(0.64278760968653932632264340990726);
        constexpr T c2 = T(0.17364817766693034885171662676931), s2 = T(0.98480775301220805936674302458952);
        constexpr T c4 = T(-0.93969262078590838405410927732473), s4 = T(0.34202014332566873304409961468226);
        const T s = T(sign);
        cpx<T> a[3][3];
#pragma unroll
        for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < 3; ++n1) a[n2][n1] = v[3 * n1 + n2];
            bfly<T, 3>(a[n2], sign);
        }
        a[1][1] = crot(a[1][1], c1, s * s1);
        a[1][2] = crot(a[1][2], c2, s * s2);
        a[2][1] = crot(a[2][1], c2, s * s2);
        a[2][2] = crot(a[2][2], c4, s * s4);
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            cpx<T> b[3] = {a[0][k1], a[1][k1], a[2][k1]};
            bfly<T, 3>(b, sign);
#pragma unroll
            for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = b[k2];
        }
    }
}

// A plan: radices in pass order, and for pass p the twiddles' offset in the table, the product
// of the radices before it and the reciprocal that divides a thread index by that.
struct GPlan {
    int n, np, tpl;       // length, passes, threads per line (n / smallest radix)
    int ps, ls;           // LDS index o is kept at o + (o >> ps); padded line stride
    int R[5], Ns[5], off[5];
    unsigned rcp[5];      // ceil(2^32 / Ns): j / Ns = mulhi(j, rcp) for j < 2^16 (Ns >= 2)
};

template <int R> struct Radix { static constexpr int value = R; };

// f(Radix<R>) for the plan's radix (uniform over the block).
template <typename F> __device__ __forceinline__ void by_radix(int R, F &&f)
{
    switch (R) {
    case 2: f(Radix<2>{}); break;
    case 3: f(Radix<3>{}); break;
    case 4: f(Radix<4>{}); break;
    case 5: f(Radix<5>{}); break;
    case 6: f(Radix<6>{}); break;
    case 8: f(Radix<8>{}); break;
    case 9: f(Radix<9>{}); break;
    case 10: f(Radix<10>{}); break;
    case 12: f(Radix<12>{}); break;
    case 15: f(Radix<15>{}); break;
    default: f(Radix<16>{}); break;
    }
}

// Pass p of the block's lines (see gfft_lines): First / Last: it takes its inputs from in, gives its
// outputs to out; otherwise the line's LDS.  A function of its own per position, not a loop over
// the passes: a loop's invariants of all radices' cases would be kept in registers.
template <typename T, int SIGN, bool First, bool FromLds, bool Last, bool ToLds, typename In, typename Out>
__device__ __forceinline__ void gfft_pass(const GPlan &P, int p, cpx<T> *line, int j, bool act,
                                          const cpx<T> *__restrict__ tw, In &&in, Out &&out)
{
    const int Ns = First ? 1 : P.Ns[p];
    by_radix(P.R[p], [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        const int nb = P.n / R;
        const bool mine = act && j < nb;
        const int jd = First ? j : (Last ? 0 : (int)__umulhi((unsigned)j, P.rcp[p])), k = First ? 0 : j - jd * Ns;
        cpx<T> v[R];
        if (mine) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int i = j + r * nb;
                if constexpr (First && !FromLds) v[r] = in(i);
                else v[r] = line[i + (i >> P.ps)];
            }
            if constexpr (!First) {
                const cpx<T> *w = tw + P.off[p] + k;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    cpx<T> f = w[(r - 1) * Ns];
                    if (SIGN > 0) f.y = -f.y;
                    v[r] = cmul(v[r], f);
                }
            }
            gdft<T, R>(v, SIGN);
        }
        if ((FromLds || !First) && (ToLds || !Last)) __syncthreads();   // this pass's inputs are read
        if (mine) {
            const int o = jd * Ns * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int d = o + r * Ns;
                if constexpr (Last && !ToLds) out(d, v[r]);
                else line[d + (d >> P.ps)] = v[r];
            }
        }
    });
    if (ToLds || !Last) __syncthreads();
}

// The transform of the block's lines (plans of two or three passes), SIGN the exponent's.  Every
// thread of the block calls: line is its line's LDS, j its index in the line, act whether it has
// a line.  in(i) gives input i of the line, out(k, value) takes output k; FromLds / ToLds: the
// inputs are in, or the outputs go to, the line's LDS instead (natural order, padded index).
template <typename T, int SIGN, bool FromLds, bool ToLds, typename In, typename Out>
__device__ __forceinline__ void gfft_lines(const GPlan &P, cpx<T> *line, int j, bool act,
                                           const cpx<T> *__restrict__ tw, In &&in, Out &&out)
{
    auto none = [](int, const cpx<T> &) {};
    auto nil = [](int) { return cpx<T>{}; };
    gfft_pass<T, SIGN, true, FromLds, false, true>(P, 0, line, j, act, tw, in, none);
    if (P.np == 3) gfft_pass<T, SIGN, false, true, false, true>(P, 1, line, j, act, tw, nil, none);
    gfft_pass<T, SIGN, false, true, true, ToLds>(P, P.np - 1, line, j, act, tw, nil, out);
}

// Host side: the plan of n with the fewest passes and, of these, the largest smallest radix
// (fewest threads per line); radices ascending, or descending where the last pass writes
// to memory and a small last radix makes its runs long.  np = 0 if n has another prime factor.
inline GPlan gplan(int n, bool descending)
{
    static const int rs[11] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};
    int best[5], nb = 0, cur[5];
    auto rec = [&](auto &&self, int m, int from, int d) -> void {
        if (m == 1) {
            if (d > 0 && (nb == 0 || d < nb || (d == nb && cur[d - 1] > best[nb - 1]))) {
                nb = d;
                for (int i = 0; i < d; ++i) best[i] = cur[i];
            }
            return;
        }
        if (d == 5 || (nb && d >= nb)) return;
        for (int i = from; i < 11; ++i)
            if (m % rs[i] == 0) {
                cur[d] = rs[i];
                self(self, m / rs[i], i, d + 1);
            }
    };
    rec(rec, n, 0, 0);
    GPlan P = {};
    P.n = n;
    P.np = nb;
    if (nb == 0) return P;
    int Ns = 1, off = 0;
    for (int p = 0; p < nb; ++p) {
        P.R[p] = descending ? best[p] : best[nb - 1 - p];
        P.Ns[p] = Ns;
        P.off[p] = off;
        P.rcp[p] = Ns > 1 ? (unsigned)((0x100000000ULL + Ns - 1) / Ns) : 0u;
        if (p > 0) off += (P.R[p] - 1) * Ns;
        Ns *= P.R[p];
    }
    P.tpl = n / best[nb - 1];
    // the first pass stores with stride R[0]: a slot of padding every 8 (16 for radix 16) elements
    // spreads an even stride over the banks
    P.ps = P.R[0] == 16 ? 4 : (P.R[0] % 2 == 0 ? 3 : 30);
    P.ls = (n + ((n - 1) >> P.ps)) | 1;
    return P;
}

template <typename T> std::vector<cpx<T>> gplan_twiddles(const GPlan &P)
{
    std::vector<cpx<T>> tw;
    const long double pi = 3.141592653589793238462643383279502884L;
    for (int p = 1; p < P.np; ++p)
        for (int r = 1; r < P.R[p]; ++r)
            for (int k = 0; k < P.Ns[p]; ++k) {
                const long double a = -2.0L * pi * (long double)((long long)r * k) / (long double)(P.Ns[p] * P.R[p]);
                tw.push_back({(T)std::cos(a), (T)std::sin(a)});
            }
    return tw;
}

}  // namespace chs
