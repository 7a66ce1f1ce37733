// Batched tridiagonal solvers of the reference (TDMAIJI_CYC, TDMAIJJ_nonCYC, TDMAIJI_nonCYC,
// TDMAIJJ_CYC) on device arrays in the reference's Fortran 2-D layout A, B, C, R(isz, jsz),
// I fastest.  One lane per line; each line follows the reference's recurrence in the same
// operation order with FMA contraction off, so results equal the reference's bit for bit.
// The channel substep does not call these (its line solves are exact-inverse stencils); they
// are the entry points for hosts that solve general systems, e.g. the inflow/outflow x-solves
// (MOMFA_io.f90:147-153) and the triply periodic box Poisson (possion3d_FFT99.f90:355-375).
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/chapsim_hip.h"
#include "chs_tdma_rule.h"

namespace {

thread_local std::string g_tdma_err;

// k_tdma_lines_ck: lines of at most 16 NCH points without a work array.  A block is one wavefront with
// 64 lines.  The forward sweep keeps the recurrence's state (h, g1, g2) at the start of every chunk
// of 16 points in LDS and nothing else; a backward sweep takes the chunks in reverse, repeats a
// chunk's forward steps from its state (the same operations, so the same bits) into registers and
// runs the backward recurrence on them.  The cyclic solver needs its backward sweep's end values for
// the last unknown before it can write any, so it sweeps back twice.  A chunk's four input arrays
// go through LDS, 64 lines by 16 points, while the next chunk's are on their way into registers;
// ALONG_I (lines contiguous in memory) is the layout where that transposes them, so that a wavefront
// reads 128-byte runs where one thread per line read 8 bytes of 64 lines.  Bound by the serial
// division per row and sweep (two wavefronts per CU at 256 points); its traffic is the inputs two
// (three) times, 9 (13) passes, where the rows of the recurrence written out
// and read back made 9 (15) and the work array was allocated on every call (256-point cyclic lines
// along x, 32768 of them: 1030 us, 200 of them allocation, -> 205 us).
constexpr int kCk = 16;
template <bool CYC, bool ALONG_I, int NCH>
__global__ __launch_bounds__(64, 1) void k_tdma_lines_ck(int n, int nl, const double *__restrict__ A,
                                                         const double *__restrict__ B, const double *__restrict__ C,
                                                         double *R, const double *__restrict__ bc)
{
#pragma clang fp contract(off)
    constexpr int TS = ALONG_I ? 64 * (kCk + 1) : 64 * kCk;   // one array's tile
    __shared__ double tile[4][TS];
    __shared__ double ck[NCH][CYC ? 3 : 2][64];
    const int lane = threadIdx.x, l0 = blockIdx.x * 64, l = min(l0 + lane, nl - 1);
    const int nch = (n + kCk - 1) / kCk, last = CYC ? n - 2 : n - 1;   // last: the forward sweep's last row
    struct Raw { double v[4][kCk]; };
    auto fetch = [&](int ch, Raw &r) {
        const double *src[4] = {A, B, C, R};
#pragma unroll
        for (int q = 0; q < kCk; ++q) {
            const int line = ALONG_I ? min(l0 + 4 * q + (lane >> 4), nl - 1) : l;
            const int i = min(ch * kCk + (ALONG_I ? lane & 15 : q), n - 1);
            const size_t o = ALONG_I ? (size_t)line * n + i : (size_t)i * nl + line;
#pragma unroll
            for (int f = 0; f < 4; ++f) r.v[f][q] = src[f][o];
        }
    };
    auto slot = [&](int e) { return ALONG_I ? lane * (kCk + 1) + e : e * 64 + lane; };   // this line's point e
    auto raw_slot = [&](int q) { return ALONG_I ? (4 * q + (lane >> 4)) * (kCk + 1) + (lane & 15) : q * 64 + lane; };
    auto place = [&](const Raw &r) {
        __syncthreads();   // the last chunk's reads are done
#pragma unroll
        for (int q = 0; q < kCk; ++q)
#pragma unroll
            for (int f = 0; f < 4; ++f) tile[f][raw_slot(q)] = r.v[f][q];
        __syncthreads();
    };
    const double bc1 = CYC ? 0.0 : bc[l], bc2 = CYC ? 0.0 : bc[nl + l];
    double h = 0.0, g1 = 0.0, g2 = 0.0;
    // forward step of row i (TDMAIJI_CYC.f90:88-125, TDMAIJJ_nonCYC.f90:88-112 and their twins)
    // inner: a row of a chunk that holds neither row 0 nor the last one, without the branches for them
    auto step = [&](int i, int e, bool inner) {
        const int s = slot(e);
        const double a = tile[0][s], b = tile[1][s], c = tile[2][s], r = tile[3][s];
        if (inner) {
            const double pp = 1.0 / (b - h * a);
            if constexpr (CYC) {
                const double qq1 = g1 * a, qq2 = g2 * a;
                h = c * pp;
                g1 = (r - qq1) * pp;
                g2 = -qq2 * pp;
            } else {
                h = c * pp;
                g1 = (r - a * g1) * pp;
            }
            return;
        }
        if (i == 0) {
            h = c / b;
            if constexpr (CYC) {
                g1 = r / b;
                g2 = -a / b;
            } else {
                g1 = (r - a * bc1) / b;
            }
            return;
        }
        const double pp = 1.0 / (b - h * a);
        if constexpr (CYC) {
            const double qq1 = g1 * a, qq2 = g2 * a;
            g1 = (r - qq1) * pp;
            if (i < n - 2) {
                h = c * pp;
                g2 = -qq2 * pp;
            } else {
                g2 = (-c - qq2) * pp;
            }
        } else if (i < n - 1) {
            h = c * pp;
            g1 = (r - a * g1) * pp;
        } else {
            g1 = (r - c * bc2 - a * g1) * pp;
        }
    };
    auto inner = [&](int ch) { return ch > 0 && ch * kCk + kCk - 1 < last; };
    Raw nx;
    fetch(0, nx);
    for (int ch = 0; ch < nch; ++ch) {
        place(nx);
        fetch(ch + 1 < nch ? ch + 1 : ch, nx);
        ck[ch][0][lane] = h;
        ck[ch][1][lane] = g1;
        if constexpr (CYC) ck[ch][2][lane] = g2;
        if (inner(ch)) {
#pragma unroll
            for (int e = 0; e < kCk; ++e) step(0, e, true);
        } else {
            for (int e = 0; e < kCk && ch * kCk + e <= last; ++e) step(ch * kCk + e, e, false);
        }
    }
    const double ge1 = g1, ge2 = g2;   // row `last`, final
    // a backward sweep over rows last .. 0: f(row, e, h, g1, g2, inner) of the row's forward values
    auto back = [&](auto &&f, auto &&chunk_done) {
        fetch(nch - 1, nx);
        for (int ch = nch - 1; ch >= 0; --ch) {
            place(nx);
            fetch(ch > 0 ? ch - 1 : 0, nx);
            h = ck[ch][0][lane];
            g1 = ck[ch][1][lane];
            if constexpr (CYC) g2 = ck[ch][2][lane];
            double H[kCk], G1[kCk], G2[kCk];
            if (inner(ch)) {
#pragma unroll
                for (int e = 0; e < kCk; ++e) {
                    step(0, e, true);
                    H[e] = h;
                    G1[e] = g1;
                    G2[e] = g2;
                }
#pragma unroll
                for (int e = kCk - 1; e >= 0; --e) f(0, e, H[e], G1[e], G2[e], true);
            } else {
#pragma unroll
                for (int e = 0; e < kCk; ++e) {
                    if (ch * kCk + e <= last) step(ch * kCk + e, e, false);
                    H[e] = h;
                    G1[e] = g1;
                    G2[e] = g2;
                }
#pragma unroll
                for (int e = kCk - 1; e >= 0; --e)
                    if (ch * kCk + e <= last) f(ch * kCk + e, e, H[e], G1[e], G2[e], false);
            }
            chunk_done(ch);
        }
    };
    // a chunk's solution, left in tile[3], to R
    auto store = [&](int ch) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kCk; ++q) {
            const int i = ch * kCk + (ALONG_I ? lane & 15 : q), line = l0 + (ALONG_I ? 4 * q + (lane >> 4) : lane);
            if (i < n && line < nl) R[ALONG_I ? (size_t)line * n + i : (size_t)i * nl + line] = tile[3][raw_slot(q)];
        }
    };
    if constexpr (CYC) {
        double b1 = ge1, b2 = ge2;
        auto sweep = [&](int i, double hh, double f1, double f2, bool in) {
            if (!in && i == last) {
                b1 = ge1;
                b2 = ge2;
            } else {
                b1 = -hh * b1 + f1;
                b2 = -hh * b2 + f2;
            }
        };
        back([&](int i, int, double hh, double f1, double f2, bool in) { sweep(i, hh, f1, f2, in); }, [](int) {});
        const size_t oe = ALONG_I ? (size_t)l * n + n - 1 : (size_t)(n - 1) * nl + l;
        const double pp = R[oe] - C[oe] * b1 - A[oe] * ge1;
        const double qq1 = B[oe] + C[oe] * b2 + A[oe] * ge2;
        const double xe = pp / qq1;
        back(
            [&](int i, int e, double hh, double f1, double f2, bool in) {
                sweep(i, hh, f1, f2, in);
                tile[3][slot(e)] = b1 + b2 * xe;
            },
            [&](int ch) {
                if (ch == nch - 1) tile[3][slot((n - 1) - ch * kCk)] = xe;
                store(ch);
            });
    } else {
        double x = 0.0;
        back(
            [&](int i, int e, double hh, double f1, double, bool in) {
                x = !in && i == last ? f1 : f1 - hh * x;
                tile[3][slot(e)] = x;
            },
            store);
    }
}

// The launch for lines of n points (at most 1280: 157 KB of LDS); false: longer lines, and the batches
// that chs_tdma_rule.h leaves to k_tdma_lines (alloc: its work array would be allocated).
template <int NCH>
void launch_ck(int kind, int n, int nl, const double *a, const double *b, const double *c, double *r, const double *bc)
{
    const dim3 g((nl + 63) / 64), t(64);
    if (kind == 0) hipLaunchKernelGGL((k_tdma_lines_ck<true, true, NCH>), g, t, 0, 0, n, nl, a, b, c, r, bc);
    else if (kind == 1) hipLaunchKernelGGL((k_tdma_lines_ck<false, false, NCH>), g, t, 0, 0, n, nl, a, b, c, r, bc);
    else if (kind == 2) hipLaunchKernelGGL((k_tdma_lines_ck<false, true, NCH>), g, t, 0, 0, n, nl, a, b, c, r, bc);
    else hipLaunchKernelGGL((k_tdma_lines_ck<true, false, NCH>), g, t, 0, 0, n, nl, a, b, c, r, bc);
}
bool tdma_ck(int kind, int n, int nl, const double *a, const double *b, const double *c, double *r, const double *bc,
             bool alloc)
{
    if (chs::tdma_thread_per_line(kind, n, nl, alloc)) return false;
    if (n <= 20 * kCk) launch_ck<20>(kind, n, nl, a, b, c, r, bc);        // 65 KB: two blocks on a CU
    else if (n <= 80 * kCk) launch_ck<80>(kind, n, nl, a, b, c, r, bc);
    else return false;
    return true;
}

// The other batches (lines longer than k_tdma_lines_ck's, and short ones), one thread per line.  work:
// 3 n doubles per line, element-major ([i][line]) so that consecutive lines coalesce.
__global__ __launch_bounds__(256) void k_tdma_lines(int kind, int isz, int jsz, const double *__restrict__ A,
                                                    const double *__restrict__ B, const double *__restrict__ C,
                                                    double *__restrict__ R, const double *__restrict__ bc,
                                                    double *__restrict__ work)
{
#pragma clang fp contract(off)
    const bool alongI = (kind == 0 || kind == 2), cyc = (kind == 0 || kind == 3);
    const int n = alongI ? isz : jsz, nl = alongI ? jsz : isz;
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= nl) return;
    const long es = alongI ? 1 : isz, lstr = alongI ? isz : 1;
    const double *a = A + l * lstr, *b = B + l * lstr, *c = C + l * lstr;
    double *r = R + l * lstr;
    double *H = work, *G1 = work + (size_t)n * nl, *G2 = work + (size_t)2 * n * nl;
    auto E = [&](const double *p, int i) { return p[(long)i * es]; };
    auto W = [&](double *p, int i) -> double & { return p[(size_t)i * nl + l]; };
    if (cyc) {
        // TDMAIJI_CYC.f90:88-157 / TDMAIJJ_CYC.f90:88-157
        W(H, 0) = E(c, 0) / E(b, 0);
        W(G1, 0) = E(r, 0) / E(b, 0);
        W(G2, 0) = -E(a, 0) / E(b, 0);
        for (int i = 1; i <= n - 3; ++i) {
            const double pp = 1.0 / (E(b, i) - W(H, i - 1) * E(a, i));
            const double qq1 = W(G1, i - 1) * E(a, i), qq2 = W(G2, i - 1) * E(a, i);
            W(H, i) = E(c, i) * pp;
            W(G1, i) = (E(r, i) - qq1) * pp;
            W(G2, i) = -qq2 * pp;
        }
        {
            const int i = n - 2;
            const double pp = 1.0 / (E(b, i) - W(H, i - 1) * E(a, i));
            const double qq1 = W(G1, i - 1) * E(a, i), qq2 = W(G2, i - 1) * E(a, i);
            W(G1, i) = (E(r, i) - qq1) * pp;
            W(G2, i) = (-E(c, i) - qq2) * pp;
        }
        for (int i = n - 3; i >= 0; --i) {
            W(G1, i) = -W(H, i) * W(G1, i + 1) + W(G1, i);
            W(G2, i) = -W(H, i) * W(G2, i + 1) + W(G2, i);
        }
        const int e = n - 1;
        const double pp = E(r, e) - E(c, e) * W(G1, 0) - E(a, e) * W(G1, e - 1);
        const double qq1 = E(b, e) + E(c, e) * W(G2, 0) + E(a, e) * W(G2, e - 1);
        const double xe = pp / qq1;
        r[(long)e * es] = xe;
        for (int i = n - 2; i >= 0; --i) r[(long)i * es] = W(G1, i) + W(G2, i) * xe;
    } else {
        // TDMAIJJ_nonCYC.f90:88-123 / TDMAIJI_nonCYC.f90:88-123
        const double bc1 = bc[l], bc2 = bc[nl + l];
        W(H, 0) = E(c, 0) / E(b, 0);
        W(G1, 0) = (E(r, 0) - E(a, 0) * bc1) / E(b, 0);
        for (int i = 1; i <= n - 2; ++i) {
            const double pp = 1.0 / (E(b, i) - W(H, i - 1) * E(a, i));
            W(H, i) = E(c, i) * pp;
            W(G1, i) = (E(r, i) - E(a, i) * W(G1, i - 1)) * pp;
        }
        const int e = n - 1;
        const double pp = 1.0 / (E(b, e) - W(H, e - 1) * E(a, e));
        double x = (E(r, e) - E(c, e) * bc2 - E(a, e) * W(G1, e - 1)) * pp;
        r[(long)e * es] = x;
        for (int i = n - 2; i >= 0; --i) {
            x = W(G1, i) - W(H, i) * x;
            r[(long)i * es] = x;
        }
    }
}

// Work buffer of chs_tdma_lines_noalloc, one per GPU for the life of the process (16 MiB).
// Host code never uses this name as an address: each device's address comes from
// hipGetSymbolAddress (scratch_ptr).
constexpr size_t kScratchDoubles = size_t(1) << 21;
__device__ __align__(256) double scratch[kScratchDoubles];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch`, looked up once per device with it current.
hipError_t scratch_ptr(double **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

}  // namespace

extern "C" {

int chs_tdma_lines(int kind, int isz, int jsz, const double *a, const double *b, const double *c, double *r,
                   const double *bc)
{
    if (kind < 0 || kind > 3) {
        g_tdma_err = "chs_tdma_lines: kind must be 0..3";
        return CHS_E_ARG;
    }
    const bool alongI = (kind == 0 || kind == 2), cyc = (kind == 0 || kind == 3);
    const int n = alongI ? isz : jsz, nl = alongI ? jsz : isz;
    if (isz < 1 || jsz < 1 || n < (cyc ? 3 : 2) || !a || !b || !c || !r || (!cyc && !bc)) {
        g_tdma_err = "chs_tdma_lines: bad size or null array (lines need 3 points cyclic, 2 otherwise)";
        return CHS_E_ARG;
    }
    double *work = nullptr;
    hipError_t e = hipSuccess;
    if (tdma_ck(kind, n, nl, a, b, c, r, bc, true)) {
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(0);
    } else if ((e = hipMalloc(&work, sizeof(double) * 3 * (size_t)n * nl)) == hipSuccess) {
        hipLaunchKernelGGL(k_tdma_lines, dim3((nl + 255) / 256), dim3(256), 0, 0, kind, isz, jsz, a, b, c, r,
                           cyc ? nullptr : bc, work);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(0);
        (void)hipFree(work);
    }
    if (e != hipSuccess) {
        g_tdma_err = std::string("chs_tdma_lines: ") + hipGetErrorString(e);
        return CHS_E_HIP;
    }
    return CHS_OK;
}

int chs_tdma_lines_noalloc(int kind, int isz, int jsz, const double *a, const double *b, const double *c, double *r,
                           const double *bc)
{
    if (kind < 0 || kind > 3) {
        g_tdma_err = "chs_tdma_lines_noalloc: kind must be 0..3";
        return CHS_E_ARG;
    }
    const bool alongI = (kind == 0 || kind == 2), cyc = (kind == 0 || kind == 3);
    const int n = alongI ? isz : jsz, nl = alongI ? jsz : isz;
    if (isz < 1 || jsz < 1 || n < (cyc ? 3 : 2) || !a || !b || !c || !r || (!cyc && !bc)) {
        g_tdma_err = "chs_tdma_lines_noalloc: bad size or null array (lines need 3 points cyclic, 2 otherwise)";
        return CHS_E_ARG;
    }
    if (3 * (size_t)n * (size_t)nl > kScratchDoubles) {
        g_tdma_err = "chs_tdma_lines_noalloc: 3 * points per line * lines exceeds the " +
                     std::to_string(kScratchDoubles) + "-double work buffer";
        return CHS_E_ARG;
    }
    // every work entry a line reads was written earlier by the same line: nothing to clear
    double *work = nullptr;
    hipError_t e = hipSuccess;
    if (tdma_ck(kind, n, nl, a, b, c, r, bc, false)) {
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(0);
    } else if ((e = scratch_ptr(&work)) == hipSuccess) {
        hipLaunchKernelGGL(k_tdma_lines, dim3((nl + 255) / 256), dim3(256), 0, 0, kind, isz, jsz, a, b, c, r,
                           cyc ? nullptr : bc, work);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(0);
    }
    if (e != hipSuccess) {
        g_tdma_err = std::string("chs_tdma_lines_noalloc: ") + hipGetErrorString(e);
        return CHS_E_HIP;
    }
    return CHS_OK;
}

const char *chs_tdma_last_error(void) { return g_tdma_err.c_str(); }

}  // extern "C"
