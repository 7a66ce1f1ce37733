"""The reference's batched Thomas solvers (TDMAIJI_CYC, TDMAIJJ_nonCYC, TDMAIJI_nonCYC,
TDMAIJJ_CYC).  The oracle restatement (or_tdma_lines) is pinned bit for bit against vectors the
compiled reference wrote (tests/golden/tdma.npz, make_golden.py make_tdma) and against a dense
solve; the GPU entry point chs_tdma_lines is compared with both, bit for bit."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import oracle

KINDS = range(4)


def _cases(golden):
    g = golden("tdma.npz")
    tags = sorted({k.rsplit("_", 1)[0] for k in g})
    return g, tags


def test_oracle_matches_reference_bitwise(golden):
    g, tags = _cases(golden)
    assert len(tags) == 20
    for t in tags:
        X = oracle.tdma_lines(int(t[1]), g[t + "_A"], g[t + "_B"], g[t + "_C"], g[t + "_R"], g[t + "_bc"])
        assert np.array_equal(X, g[t + "_X"]), t


@pytest.mark.parametrize("kind", KINDS)
def test_oracle_solves_the_system(kind):
    """Dense check of the restatement: the residual of the assembled (cyclic) tridiagonal
    system, boundary values moved to the right-hand side."""
    rng = np.random.default_rng(kind)
    isz, jsz = 9, 6
    A, C_ = rng.uniform(-1, 1, (2, jsz, isz))
    B = 2.5 + rng.uniform(0, 1, (jsz, isz))
    R = rng.standard_normal((jsz, isz))
    alongI, cyc = kind in (0, 2), kind in (0, 3)
    nl = jsz if alongI else isz
    bc = rng.standard_normal((2, nl)) if not cyc else np.zeros((2, nl))
    X = oracle.tdma_lines(kind, A, B, C_, R, bc)
    for line in range(nl):
        sl = (line, slice(None)) if alongI else (slice(None), line)
        a, b, c, r, x = A[sl], B[sl], C_[sl], R[sl].copy(), X[sl]
        Mx = np.diag(b) + np.diag(a[1:], -1) + np.diag(c[:-1], 1)
        if cyc:
            Mx[0, -1], Mx[-1, 0] = a[0], c[-1]
        else:
            r[0] -= a[0] * bc[0, line]
            r[-1] -= c[-1] * bc[1, line]
        assert np.abs(Mx @ x - r).max() < 1e-14


@pytest.mark.gpu
def test_gpu_matches_reference_bitwise(pkg, golden):
    g, tags = _cases(golden)
    for t in tags:
        print(f"tdma {t}", flush=True)
        X = pkg.tdma_lines(int(t[1]), g[t + "_A"], g[t + "_B"], g[t + "_C"], g[t + "_R"], g[t + "_bc"])
        assert np.array_equal(X, g[t + "_X"]), (t, np.abs(X - g[t + "_X"]).max())


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_gpu_matches_oracle_many_lines(pkg, kind):
    """Wide batches (more lines than a block) and long lines, bit for bit against the oracle."""
    rng = np.random.default_rng(10 + kind)
    isz, jsz = (300, 517) if kind in (0, 2) else (517, 300)
    A, C_ = rng.uniform(-1, 1, (2, jsz, isz))
    B = 2.5 + rng.uniform(0, 1, (jsz, isz))
    R = rng.standard_normal((jsz, isz))
    nl = jsz if kind in (0, 2) else isz
    bc = rng.standard_normal((2, nl))
    X = pkg.tdma_lines(kind, A, B, C_, R, bc)
    assert np.array_equal(X, oracle.tdma_lines(kind, A, B, C_, R, bc))


@pytest.mark.gpu
def test_gpu_rejects_bad_arguments(pkg):
    z = np.zeros((4, 2))
    with pytest.raises(pkg.ChsError):
        pkg.tdma_lines(0, z, z + 1, z, z)          # cyclic line of 2 points
    with pytest.raises(pkg.ChsError):
        pkg.tdma_lines(7, z, z + 1, z, z)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [2, 3, 4, 15, 16, 17, 18, 32, 33, 34, 320, 321, 1280, 1281])
def test_gpu_chunk_and_wavefront_edges(pkg, kind, n):
    """Chunks of 16 points with the last one short or holding the cyclic solver's last unknown alone,
    the longest lines of each LDS size and the first beyond them, and wavefronts with one line, all
    but one and one more than 64: bit for bit against the oracle, on both entry points."""
    if n < 3 and kind in (0, 3):
        pytest.skip("a cyclic line needs 3 points")
    for nl in (1, 63, 65):
        rng = np.random.default_rng(1000 * kind + n + nl)
        isz, jsz = (n, nl) if kind in (0, 2) else (nl, n)
        A, C_ = rng.uniform(-1, 1, (2, jsz, isz))
        B = 2.5 + rng.uniform(0, 1, (jsz, isz))
        R = rng.standard_normal((jsz, isz))
        bc = rng.standard_normal((2, nl))
        ref = oracle.tdma_lines(kind, A, B, C_, R, bc)
        assert np.array_equal(pkg.tdma_lines(kind, A, B, C_, R, bc), ref), (n, nl)
        assert np.array_equal(pkg.tdma_lines(kind, A, B, C_, R, bc, noalloc=True), ref), (n, nl)


# us of a call on MI355X, one thread per line / checkpoints in LDS: kind, points, lines, work array allocated
ROUTES = [(0, 4, 4096, 1, 16, 22), (0, 4, 64, 1, 15, 22), (0, 8, 512, 1, 20, 24), (0, 17, 64, 1, 24, 32), (0, 49, 64, 1, 45, 49),
          (0, 16, 512, 1, 32, 28), (0, 64, 64, 1, 59, 51), (0, 128, 8, 1, 91, 77), (0, 33, 65, 1, 36, 43), (0, 33, 256, 1, 50, 43),
          (0, 256, 32768, 1, 1029, 205), (0, 8, 16384, 1, 37, 24), (0, 4, 131072, 1, 46, 62), (0, 16, 131072, 1, 219, 86),
          (0, 4, 131072, 0, 18, 62), (0, 8, 65536, 0, 23, 42), (0, 24, 16384, 0, 42, 35),
          (1, 4, 4096, 1, 15, 17), (1, 17, 512, 1, 21, 24), (1, 64, 64, 1, 41, 36), (1, 64, 1, 1, 31, 35), (1, 128, 8, 1, 66, 53),
          (1, 24, 4096, 1, 53, 25), (1, 8, 65536, 0, 17, 26), (1, 40, 16384, 0, 40, 31),
          (2, 8, 64, 1, 16, 18), (2, 16, 512, 1, 27, 21), (2, 17, 64, 1, 21, 24), (2, 48, 4096, 1, 89, 33), (2, 4, 65536, 0, 16, 28),
          (2, 16, 16384, 0, 28, 21), (2, 18, 65, 1, 21, 24), (2, 49, 1, 1, 28, 31),
          (3, 4, 4096, 1, 16, 21), (3, 17, 512, 1, 25, 29), (3, 33, 64, 1, 33, 39), (3, 49, 64, 1, 43, 46), (3, 64, 512, 1, 58, 47),
          (3, 17, 16384, 1, 54, 30), (3, 18, 131072, 1, 82, 97), (3, 10, 98304, 1, 61, 50), (3, 18, 262144, 1, 1244, 172), (3, 8, 65536, 0, 20, 36)]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ absent")
def test_short_lines_take_the_faster_kernel(tmp_path):
    """The rule between the two kernels against their measured times: the faster one wherever they
    differ by 5 % and more."""
    exe = tmp_path / "tdma_rule"
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "tdma_rule.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", src, "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="".join("%d %d %d %d\n" % r[:4] for r in ROUTES), capture_output=True,
                         text=True, check=True).stdout.split()
    assert len(out) == len(ROUTES)
    for r, o in zip(ROUTES, out):
        assert abs(r[4] / r[5] - 1.0) > 0.05
        assert (o == "1") == (r[4] < r[5]), r


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_gpu_lines_each_side_of_the_rule(pkg, kind):
    """Batches on each side of the rule's limits (by wavefronts for lines along I, by points along J, a
    single line, many lines), on both entry points: bit for bit against the oracle."""
    along_i = kind in (0, 2)
    sizes = [(84, 1), (129, 1), (8, 300), (9, 300), (12, 257), (13, 257), (16, 300), (17, 300), (18, 193), (33, 300), (48, 129)]
    if along_i:
        sizes += [(30, 64), (52, 64), (53, 64), (20, 128), (35, 128), (10, 192), (19, 192)]
    else:
        sizes += [(34, 65), (35, 300), (49, 300), (64, 300), (24, 8200), (25, 8200), (33, 8200)]
    for n, nl in sizes:
        rng = np.random.default_rng(1000 * kind + n + nl)
        isz, jsz = (n, nl) if along_i else (nl, n)
        A, C_ = rng.uniform(-1, 1, (2, jsz, isz))
        B = 2.5 + rng.uniform(0, 1, (jsz, isz))
        R = rng.standard_normal((jsz, isz))
        bc = rng.standard_normal((2, nl))
        ref = oracle.tdma_lines(kind, A, B, C_, R, bc)
        for noalloc in (False, True):
            assert np.array_equal(pkg.tdma_lines(kind, A, B, C_, R, bc, noalloc=noalloc), ref), (n, nl, noalloc)
