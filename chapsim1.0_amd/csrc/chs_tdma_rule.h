// Which kernel solves a batch of lines: k_tdma_lines (true, one thread per line, three work values a
// point) or k_tdma_lines_ck (false, checkpoints in LDS).  Host code without HIP.
#pragma once
#include <cstddef>

namespace chs {

// k_tdma_lines_ck sweeps three times through chunks of 16 points whatever a line's length, and its
// LDS leaves two wavefronts on a CU; k_tdma_lines' time goes with the points, with the wavefronts (of
// up to four) that its first CUs hold, and, for lines along I, with the 64 cache lines of each load.
// So short lines are its own, the shorter the more wavefronts.  us, k_tdma_lines / k_tdma_lines_ck, by
// kind, points x lines: 0: 4x4096 16 / 22, 17x64 24 / 32, 49x64 45 / 49, 64x64 59 / 51, 16x512 32 / 28;
// 2: 8x4096 18 / 19, 16x512 27 / 21, 24x64 25 / 26; 1: 17x512 21 / 24, 24x1000 24 / 25, 40x512 31 / 30;
// 3: 17x512 25 / 29, 33x512 37 / 38, 49x64 43 / 45, 64x512 58 / 47.
// With a work array to allocate (alloc; about 20 us from 2 MB on, 300 from 64 MB on) it pays only where
// k_tdma_lines_ck takes several rounds of blocks: 3: 18x131072 82 / 97, 10x98304 61 / 50; 0: 4x131072
// 46 / 62, 8x16384 37 / 24.
inline bool tdma_thread_per_line(int kind, int n, int nl, bool alloc)
{
    const bool along_i = kind == 0 || kind == 2, cyc = kind == 0 || kind == 3;
    const size_t work = sizeof(double) * 3 * (size_t)n * (size_t)nl;
    if (alloc && work > (size_t(2) << 20))
        return work <= (size_t(64) << 20) && nl > 98304 && cyc && n <= (along_i ? 6 : 20);
    if (nl == 1) return n <= (cyc ? 84 : 128);   // 64 x 1: 31 / 35 (kind 1)
    const int waves = nl <= 64 ? 1 : nl <= 128 ? 2 : nl <= 192 ? 3 : 4;
    if (along_i) {
        const int lim[2][4] = {{30, 20, 10, 8}, {52, 34, 18, 12}};
        return n <= lim[cyc][waves - 1];
    }
    return n <= (nl > 8192 ? 24 : cyc && waves < 4 ? 52 : 34);
}

}  // namespace chs
