"""GPU parity of the plain FP64 substep against the oracle (and the reference's golden
vectors).  Tolerances: velocity and pressure 1e-10 relative (max-norm) per substep,
divergence after projection < 1e-10.  Each test prints the largest errors it saw."""
import numpy as np
import pytest

from oracle import oracle, setup

pytestmark = pytest.mark.gpu

MESHES = [  # L, M, N, STR2, REN, dt
    (16, 16, 16, 1.8, 2800.0, 1.0e-3),
    (20, 18, 30, 2.2, 6875.0, 5.0e-4),
    (64, 64, 64, 1.8, 2800.0, 1.0e-3),
    (48, 36, 40, 2.0, 4000.0, 8.0e-4),
    (256, 24, 256, 2.0, 6875.0, 5.0e-4),
]


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def make(pkg, L, M, N, STR2, REN, seed=3):
    mesh = setup.Mesh(L, M, N, STR2=STR2)
    q, pr = oracle.initial_field(mesh, seed)
    ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=STR2), pkg.PLAIN_FP64)
    ch.upload(q, pr)
    o = oracle.OracleTG(mesh, REN)
    o.set_fields(q, pr)
    return mesh, ch, o


@pytest.mark.parametrize("L,M,N,STR2,REN,dt", MESHES)
def test_projection_and_steps_match_oracle(pkg, L, M, N, STR2, REN, dt):
    print(f"case {L}x{M}x{N}", flush=True)
    mesh, ch, o = make(pkg, L, M, N, STR2, REN)
    cv = 1.0 / REN
    ch.SOLVERRK3_MOM_tg(0, dt, cv)
    o.substep(0, dt)
    gq, gp = ch.download()
    eq = max(rel(gq[c], o.q[c]) for c in range(3))
    ep = rel(gp, o.pr)
    assert eq < 1e-10, ("ns0", eq)
    assert ep < 1e-10, ("ns0", ep)
    assert ch.max_div() < 1e-10
    for step in range(3):
        for ns in (1, 2, 3):
            ch.SOLVERRK3_MOM_tg(ns, dt, cv)
            o.substep(ns, dt)
            gq, gp, gh = ch.download(with_history=True)
            e = max(rel(gq[c], o.q[c]) for c in range(3))
            e_p = rel(gp, o.pr)
            eq, ep = max(eq, e), max(ep, e_p)
            assert e < 1e-10, (step, ns, e)
            assert e_p < 1e-10, (step, ns, e_p)
            assert rel(gh[0], o.convh0[0]) < 1e-10
    div = ch.max_div()
    print(f"  {L}x{M}x{N}: max rel error velocity {eq:.2e}, pressure {ep:.2e}; max div {div:.2e}")
    assert div < 1e-10
    ch.close()


@pytest.mark.parametrize("name", ["tg_16x16x16.npz", "tg_20x18x30.npz"])
def test_matches_reference_golden(pkg, golden, name):
    g = golden(name)
    L, M, N, STR2, REN, dt = (g["params"][i] for i in range(6))
    L, M, N = int(L), int(M), int(N)
    ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=STR2), pkg.PLAIN_FP64)
    ch.upload(g["q_init"], g["pr_init"])
    ch.SOLVERRK3_MOM_tg(0, dt, 1.0 / REN)
    gq, gp = ch.download()
    e0 = [max(rel(gq[c], g["q_ns0"][c]) for c in range(3)), rel(gp, g["pr_ns0"])]
    ch.rk3_step(dt, 1.0 / REN)
    gq, gp = ch.download()
    e1 = [max(rel(gq[c], g["q_step1"][c]) for c in range(3)), rel(gp, g["pr_step1"])]
    phi = ch.poisson(g["poisson_rhs"])
    e2 = rel(phi, g["poisson_phi"])
    print(f"  {name}: projection velocity {e0[0]:.2e} pressure {e0[1]:.2e}; RK3 step velocity "
          f"{e1[0]:.2e} pressure {e1[1]:.2e}; Poisson {e2:.2e}")
    assert e0[0] < 1e-10 and e1[0] < 1e-10
    assert e0[1] < 1e-10 and e1[1] < 1e-10
    assert e2 < 1e-10
    ch.close()


# line lengths 64 ... 1024 run the register FFTs (chs_fftr.h), the others the LDS Stockham
# transforms; fft_reg=0 forces the latter on planned lengths too
# transforms; fft_reg=0 forces the latter on planned lengths too.  ytc: rows per chunk of the
# chunked y-Thomas (-1 automatic, 0 the one-thread-per-line kernel; 4 and 8 give many chunks)
POISSON_MESHES = [(16, 16, 16, 1, -1), (16, 16, 16, 1, 0), (30, 20, 24, 1, 4), (128, 96, 128, 1, -1),
                  (128, 96, 128, 0, 8), (128, 96, 128, 1, 0), (64, 20, 96, 1, 4), (256, 12, 256, 1, -1),
                  (512, 8, 512, 1, -1), (1024, 6, 64, 1, -1), (96, 10, 1024, 1, 4), (64, 256, 64, 1, -1),
                  (64, 300, 32, 1, -1), (32, 61, 48, 1, 4)]


@pytest.mark.parametrize("L,M,N,reg,ytc", POISSON_MESHES)
def test_poisson_matches_oracle(pkg, L, M, N, reg, ytc):
    print(f"poisson {L}x{M}x{N} fft_reg={reg} ytdma_c={ytc}", flush=True)
    mesh = setup.Mesh(L, M, N, STR2=2.2)
    rng = np.random.default_rng(5)
    r = rng.standard_normal((N, M, L))
    w = (1.0 / mesh.DYFI)[None, :, None]
    r -= np.sum(r * w) / (np.sum(w) * L * N)
    o = oracle.OracleTG(mesh, 2800.0)
    ref = o.poisson(r)
    for mode, tol in ((pkg.PLAIN_FP64, 1e-10), (pkg.MIXED, 1e-5)):
        ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=2.2), mode)
        ch.set_tuning(fft_reg=reg, ytdma_c=ytc)
        phi = ch.poisson(r)
        e = rel(phi, ref)
        print(f"  {'plain' if mode == pkg.PLAIN_FP64 else 'mixed'}: rel error {e:.2e}")
        assert e < tol, (mode, e)
        ch.close()


def test_mass_flux_and_walls(pkg):
    L, M, N, REN, dt = 32, 32, 32, 2800.0, 1e-3
    mesh, ch, _ = make(pkg, L, M, N, 1.8, REN)
    ch.SOLVERRK3_MOM_tg(0, dt, 1.0 / REN)
    q0, _ = ch.download()
    bulk0 = np.sum(q0[0][:, 1:M + 1] / mesh.DYFI[None, :, None])
    for _ in range(3):
        ch.rk3_step(dt, 1.0 / REN)
    q, p = ch.download()
    bulk = np.sum(q[0][:, 1:M + 1] / mesh.DYFI[None, :, None])
    # constant mass flux (iFlowDriven = 1): the explicit increment has zero volume mean
    # (RHS_CvLpGpS_tg.f90:165-201); the wall-bounded CN y-solve then moves the bulk by O(beta)
    assert abs(bulk - bulk0) / abs(bulk0) < 1e-9
    assert np.all(q[:, :, 0, :] == 0) and np.all(q[:, :, M + 1, :] == 0)
    assert np.all(q[1, :, 1, :] == 0)                    # v on the bottom wall
    np.testing.assert_array_equal(p[:, 0, :], p[:, 1, :])
    np.testing.assert_array_equal(p[:, M + 1, :], p[:, M, :])
    ch.close()


@pytest.mark.parametrize("L,M,N", [(64, 48, 32), (30, 20, 24)])
def test_poisson_device_refinement(pkg, L, M, N):
    """Device Poisson: FP64 form matches the oracle; the mixed form (FP32 transforms) reaches
    FP64 accuracy with residual-driven FP64 refinement sweeps."""
    mesh = setup.Mesh(L, M, N, STR2=2.2)
    rng = np.random.default_rng(8)
    r = rng.standard_normal((N, M, L))
    w = (1.0 / mesh.DYFI)[None, :, None]
    r -= np.sum(r * w) / (np.sum(w) * L * N)
    ref = oracle.OracleTG(mesh, 2800.0).poisson(r)
    d_r = pkg.DeviceArray.from_host(r)
    d_phi = pkg.DeviceArray(r.shape)
    co = pkg.channel_setup(L, M, N, STR2=2.2)
    plain = pkg.ChannelTG(co, pkg.PLAIN_FP64)
    res = plain.poisson_device(d_r.ptr, d_phi.ptr, 0)
    assert rel(d_phi.to_host(), ref) < 1e-10
    assert res < 1e-9 * np.max(np.abs(r))
    mixed = pkg.ChannelTG(co, pkg.MIXED)
    errs, gauge = [], []
    for nref in (0, 1, 2):
        mixed.poisson_device(d_r.ptr, d_phi.ptr, nref)
        phi = d_phi.to_host()
        errs.append(rel(phi, ref))
        gauge.append(abs(phi[:, 0, :].mean()) / np.max(np.abs(ref)))
    print(f"mixed Poisson {L}x{M}x{N} error vs FP64 after 0/1/2 sweeps: {errs}; "
          f"J=1 plane mean: {gauge}")
    assert errs[0] < 1e-3
    # the sweeps restore the reference's gauge (zero mean over J = 1) in FP64
    assert gauge[1] < 1e-14 and gauge[2] < 1e-14
    assert errs[1] < 1e-8 and errs[2] < 1e-10
    plain.close()
    mixed.close()
    d_r.free()
    d_phi.free()


SHAPES = [
    dict(conv_by=16, conv_kc=3, cnx_nlx=3, cnz_kz=5, cny_ky=7, fftx_tk=2, fftz_nl=1, nxcd=3, cn_xz=1,
         cnxz_by=2),
    dict(conv_by=1, conv_kc=1, cnx_nlx=1, cnz_kz=40, cny_ky=36, fftx_tk=8, fftz_nl=5, cn_xz=1),
    dict(conv_by=4, conv_bx=4, conv_kc=7, nxcd=8, cnxz_by=4, cnz_kz=9, cn_xz=1),
]


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_launch_shapes_keep_results(pkg, shape):
    """chs_set_tuning: other tilings of every kernel (ragged chunks included) give the
    oracle's result to the same tolerance as the default shapes."""
    L, M, N, STR2, REN, dt = 48, 36, 40, 2.0, 4000.0, 8.0e-4
    print(f"shape {SHAPES[shape]}", flush=True)
    mesh, ch, o = make(pkg, L, M, N, STR2, REN)
    ch.set_tuning(**SHAPES[shape])
    cv = 1.0 / REN
    ch.SOLVERRK3_MOM_tg(0, dt, cv)
    o.substep(0, dt)
    for _ in range(2):
        ch.rk3_step(dt, cv)
        for ns in (1, 2, 3):
            o.substep(ns, dt)
    gq, gp = ch.download()
    e, ep = max(rel(gq[c], o.q[c]) for c in range(3)), rel(gp, o.pr)
    print(f"  velocity {e:.2e} pressure {ep:.2e}")
    assert e < 1e-10 and ep < 1e-10
    ch.close()


@pytest.mark.parametrize("L,M,N,fx", [(192, 24, 32, 1), (192, 24, 32, 2), (128, 32, 48, 2), (128, 32, 48, 0),
                                       (64, 48, 32, 2)])
def test_fused_x_solve_matches_oracle(pkg, L, M, N, fx):
    """The x-solve inside k_conv_rhs (conv_fx rows per block; 0: the separate x kernel) on
    whole-line tiles of one to three wavefronts (a 3-wave tile folds its mass-flux partials
    first), with the mass-flux correction applied after the z-solve."""
    STR2, REN, dt = 2.0, 4000.0, 8.0e-4
    print(f"fused x {L}x{M}x{N} conv_fx {fx}", flush=True)
    mesh, ch, o = make(pkg, L, M, N, STR2, REN)
    ch.set_tuning(conv_fx=fx)
    cv = 1.0 / REN
    ch.SOLVERRK3_MOM_tg(0, dt, cv)
    o.substep(0, dt)
    for _ in range(2):
        ch.rk3_step(dt, cv)
        for ns in (1, 2, 3):
            o.substep(ns, dt)
    gq, gp = ch.download()
    e, ep = max(rel(gq[c], o.q[c]) for c in range(3)), rel(gp, o.pr)
    print(f"  velocity {e:.2e} pressure {ep:.2e}")
    assert e < 1e-10 and ep < 1e-10
    assert ch.max_div() < 1e-10
    ch.close()


@pytest.mark.parametrize("L,M,N,REN,dt,ky", [(64, 48, 32, 4000.0, 8.0e-4, 0), (64, 48, 32, 4000.0, 8.0e-4, 16),
                                              (128, 40, 48, 6875.0, 5.0e-4, 7), (64, 24, 16, 2800.0, 2.0e-3, 20),
                                              (192, 36, 64, 2800.0, 1.0e-3, 11), (96, 36, 40, 4000.0, 8.0e-4, 16),
                                              (20, 18, 30, 6875.0, 5.0e-4, 0)])
def test_fused_zy_solve_matches_two_kernels_and_oracle(pkg, L, M, N, REN, dt, ky):
    """k_cn_zy_march (the z and y Crank-Nicolson inverses in one pass, chunks of ky rows, 0 =
    whole lines, ragged last chunks; ragged x and z tiles where L is not a multiple of 64 or N
    of 16) gives the separate z and y kernels' result to rounding and
    the oracle's to 1e-10, in FP64 and in the mixed form (against the mixed two-kernel path)."""
    STR2 = 2.0
    print(f"fused zy {L}x{M}x{N} ky {ky}", flush=True)
    mesh, ch, o = make(pkg, L, M, N, STR2, REN)
    two = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=STR2), pkg.PLAIN_FP64)
    q0, p0 = oracle.initial_field(mesh, 3)
    two.upload(q0, p0)
    ch.set_tuning(cnzy=2, cnzy_ky=ky)
    two.set_tuning(cnzy=0)
    cv = 1.0 / REN
    for c in (ch, two):
        c.SOLVERRK3_MOM_tg(0, dt, cv)
        for _ in range(2):
            c.rk3_step(dt, cv)
    o.substep(0, dt)
    for _ in range(2):
        for ns in (1, 2, 3):
            o.substep(ns, dt)
    gq, gp = ch.download()
    tq, tp = two.download()
    dq, dp = max(rel(gq[c], tq[c]) for c in range(3)), rel(gp, tp)
    e, ep = max(rel(gq[c], o.q[c]) for c in range(3)), rel(gp, o.pr)
    print(f"  fused vs two kernels velocity {dq:.2e} pressure {dp:.2e}; vs oracle velocity {e:.2e} "
          f"pressure {ep:.2e}")
    # rounding only (contractions differ between the kernels); the pressure carries the
    # Poisson solve's amplification of it
    assert dq < 1e-13 and dp < 1e-10
    assert e < 1e-10 and ep < 1e-10
    assert ch.max_div() < 1e-10
    ch.close()
    two.close()
    mixed = [pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=STR2), pkg.MIXED) for _ in range(2)]
    for m, on in zip(mixed, (1, 0)):
        m.upload(q0, p0)
        m.set_tuning(cnzy=2 * on, cnzy_ky=ky)
        m.SOLVERRK3_MOM_tg(0, dt, cv)
        for _ in range(2):
            m.rk3_step(dt, cv)
    (aq, ap), (bq, bp) = mixed[0].download(), mixed[1].download()
    # the mixed form's error against FP64, fused and with two kernels: FP32 rounding of the
    # same size
    ea, eb = max(rel(aq[c], gq[c]) for c in range(3)), max(rel(bq[c], gq[c]) for c in range(3))
    pa, pb = rel(ap, gp), rel(bp, gp)
    print(f"  mixed vs FP64: fused velocity {ea:.2e} pressure {pa:.2e}; two kernels velocity {eb:.2e} "
          f"pressure {pb:.2e}")
    assert ea < 1e-5 and ea < 3 * eb + 1e-7
    assert pa < 3 * pb + 1e-6
    for m in mixed:
        m.close()


@pytest.mark.parametrize("L,M,N,mode", [(128, 40, 48, "plain"), (256, 24, 32, "plain"), (128, 20, 24, "mixed")])
def test_update_two_points_per_lane_bit_identical(pkg, L, M, N, mode):
    """k_update2 (two points per lane, neighbours across lanes and the stretch's edges loaded)
    gives k_update's fields and CFL bit for bit, with and without the CFL reduction."""
    print(f"update2 {L}x{M}x{N} {mode}", flush=True)
    mesh = setup.Mesh(L, M, N, STR2=2.0)
    q, pr = oracle.initial_field(mesh, 5)
    m = pkg.PLAIN_FP64 if mode == "plain" else pkg.MIXED
    out = []
    for w2 in (1, 0):
        ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=2.0), m)
        ch.set_tuning(upd_w2=w2)
        ch.upload(q, pr)
        ch.SOLVERRK3_MOM_tg(0, 5e-4, 1 / 4000.0)
        for _ in range(2):
            ch.rk3_step(5e-4, 1 / 4000.0)
        out.append((*ch.download(), ch.step_state()["cflmm"]))
        ch.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    assert out[0][2] == out[1][2] and np.isfinite(out[0][2])


def test_tuning_rejects_bad_shapes(pkg):
    ch = pkg.ChannelTG(pkg.channel_setup(48, 36, 40, STR2=2.0), pkg.PLAIN_FP64)
    for bad in (dict(conv_by=3), dict(conv_bx=2), dict(conv_kc=0), dict(fft_reg=2), dict(nxcd=0), dict(cn_xz=2), dict(cnxz_by=3), dict(conv_kc=41), dict(fftx_tk=3),
                dict(fftx_tk=6), dict(fftz_nl=100), dict(cny_ky=37), dict(cnx_nlx=10**6), dict(conv_fx=3),
                dict(cnzy=3), dict(cnzy_ky=37), dict(cnzy_nxcd=0), dict(upd_w2=2),
                dict(ytdma_c=12), dict(ytdma_c=-2), dict(no_such_key=1)):
        with pytest.raises(pkg.ChsError):
            ch.set_tuning(**bad)
    ch.close()


def test_autotune_restores_state(pkg):
    """The autotuner leaves the fields as they were and picks valid shapes."""
    import importlib
    tune = importlib.import_module(pkg.__name__ + ".tune")
    L, M, N, STR2, REN, dt = 48, 36, 40, 2.0, 4000.0, 8.0e-4
    mesh, ch, o = make(pkg, L, M, N, STR2, REN)
    cv = 1.0 / REN
    ch.SOLVERRK3_MOM_tg(0, dt, cv)
    before = ch.download(with_history=True)
    res = tune.autotune(ch, dt, cv, steps=1)
    after = ch.download(with_history=True)
    for a, b in zip(before, after):
        assert np.array_equal(a, b)
    cands = tune.candidates(L, M, N)
    for k, v in res["best"].items():
        assert v in cands[k]
    o.substep(0, dt)
    ch.rk3_step(dt, cv)
    for ns in (1, 2, 3):
        o.substep(ns, dt)
    gq, _ = ch.download()
    for c in range(3):
        assert rel(gq[c], o.q[c]) < 1e-10
    ch.close()


def test_config1_100_steps_match_oracle(pkg):
    """The CPU-runnable configuration as configured: 64^3, Re_tau 180 (REN 2800), tanh beta 1.8,
    laminar profile + 10 % seeded perturbations projected by NS = 0, dt 1e-3, 100 RK3 steps,
    plain FP64, against the oracle after every 10 steps (velocity, pressure, x-z mean u,
    maximum divergence)."""
    L, M, N, STR2, REN, dt = 64, 64, 64, 1.8, 2800.0, 1.0e-3
    print(f"config 1 {L}x{M}x{N}, 100 steps", flush=True)
    mesh, ch, o = make(pkg, L, M, N, STR2, REN, seed=180)
    cv = 1.0 / REN
    ch.SOLVERRK3_MOM_tg(0, dt, cv)
    o.substep(0, dt)
    worst = dict(u=0.0, p=0.0, mean=0.0)
    for step in range(1, 101):
        ch.rk3_step(dt, cv)
        for ns in (1, 2, 3):
            o.substep(ns, dt)
        if step % 10 == 0:
            gq, gp = ch.download()
            e = max(rel(gq[c], o.q[c]) for c in range(3))
            e_p = rel(gp, o.pr)
            um_g = gq[0][:, 1:M + 1].mean(axis=(0, 2))
            um_o = o.q[0][:, 1:M + 1].mean(axis=(0, 2))
            e_m = float(np.max(np.abs(um_g - um_o)) / np.max(np.abs(um_o)))
            worst = dict(u=max(worst["u"], e), p=max(worst["p"], e_p), mean=max(worst["mean"], e_m))
            print(f"  step {step}: velocity {e:.2e}, pressure {e_p:.2e}, mean u {e_m:.2e}", flush=True)
    div = ch.max_div()
    print(f"  worst {worst}; max div {div:.2e}", flush=True)
    # measured on MI355X: velocity 7.6e-15, pressure 3.4e-12, mean u 4.4e-16, div 1.6e-15
    assert worst["u"] < 1e-13 and worst["mean"] < 1e-14, worst
    assert worst["p"] < 1e-10, worst
    assert div < 1e-12
    ch.close()


# Mixed-radix transforms (chs_fftg.h): two- and three-pass plans in x and z, plane blocks cut short
# (N = 18, 50, 90), lines of 256 threads, FP64 plans that replace the register ones (128, 512), and
# a length with no plan of three passes (1250, LDS transforms).
MIXED_RADIX_MESHES = [(18, 5, 18), (150, 6, 120), (162, 4, 250), (200, 5, 50), (128, 7, 90), (512, 5, 30),
                      (30, 4, 2048), (2048, 4, 6), (1250, 4, 20), (54, 9, 486)]


@pytest.mark.parametrize("L,M,N", MIXED_RADIX_MESHES)
def test_mixed_radix_poisson_matches_oracle_and_device_output(pkg, L, M, N):
    """The solve against the oracle (bounds as test_poisson_matches_oracle), and the device entry
    point's cell output equal to the host one's, which goes through the halo field."""
    print(f"mixed-radix poisson {L}x{M}x{N}", flush=True)
    mesh = setup.Mesh(L, M, N, STR2=1.9)
    r = np.random.default_rng(L + N).standard_normal((N, M, L))
    w = (1.0 / mesh.DYFI)[None, :, None]
    r -= np.sum(r * w) / (np.sum(w) * L * N)
    ref = oracle.OracleTG(mesh, 2800.0).poisson(r)
    for mode, tol in ((pkg.PLAIN_FP64, 1e-10), (pkg.MIXED, 1e-5)):
        ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.9), mode)
        phi = ch.poisson(r)
        assert rel(phi, ref) < tol, (mode, rel(phi, ref))
        d_r, d_p = pkg.DeviceArray.from_host(r), pkg.DeviceArray(r.shape)
        ch.poisson_device(d_r.ptr, d_p.ptr, 0, False)
        ch.sync()
        assert np.array_equal(d_p.to_host(), phi)
        for d in (d_r, d_p):
            d.free()
        ch.close()


@pytest.mark.parametrize("M", [129, 131, 192, 256, 257, 320, 321, 512, 513, 769, 1024, 1025])
def test_wide_ytdma_matches_serial_lines(pkg, M):
    """The y-Thomas with 16-line runs (M > 128; chunks of 8, 12 and 16 rows, the last one short)
    against one thread per line (ytdma_c = 0), both gauges.  The split sweeps differ from the serial
    one by rounding only; the (0, 0) mode's Neumann sweep amplifies it by at most the condition
    M^2 / 4 of that line (1e-16 * 2.6e5 = 3e-11 at M = 1024)."""
    L, N = 36, 30
    r = np.random.default_rng(M).standard_normal((N, M, L))
    co = pkg.channel_setup(L, M, N, STR2=1.9)
    w = (1.0 / co["dyfi"])[None, :, None]
    r -= np.sum(r * w) / (np.sum(w) * L * N)
    for mode, tol in ((pkg.PLAIN_FP64, 1e-10), (pkg.MIXED, 1e-5)):
        ch = pkg.ChannelTG(co, mode)
        got = [ch.poisson(r), ch.FISHPACK_POIS3D_SIMPLE(r)]
        ch.set_tuning(ytdma_c=0)
        ref = [ch.poisson(r), ch.FISHPACK_POIS3D_SIMPLE(r)]
        for a, b in zip(got, ref):
            assert rel(a, b) < tol, (mode, rel(a, b))
        ch.close()


@pytest.mark.parametrize("L,M,N,REN,dt", [(32, 5, 10, 2000.0, 1.0e-3), (36, 4, 6, 4000.0, 5.0e-4), (60, 7, 50, 4000.0, 5.0e-4),
                                          (64, 9, 20, 4000.0, 5.0e-4), (96, 6, 16, 4000.0, 5.0e-4), (128, 13, 18, 4000.0, 5.0e-4),
                                          (150, 10, 36, 4000.0, 5.0e-4), (192, 11, 12, 4000.0, 5.0e-4), (250, 5, 24, 4000.0, 5.0e-4),
                                          (256, 6, 100, 4000.0, 5.0e-4)])
def test_ragged_convection_tiles_match_oracle(pkg, L, M, N, REN, dt):
    """The direct-to-LDS convection kernel on ragged tiles (each width class, rows past M, a single
    row left, marches cut short) over two RK3 steps against the oracle, and against the
    per-column kernel (conv_dma = 0, conv_fx = 0) to rounding.  Bounds as
    test_projection_and_steps_match_oracle; the two routes differ by the order of the mass-flux
    sum and the banded x-solve's last bits: 1e-13 of the velocity."""
    print(f"ragged convection {L}x{M}x{N}", flush=True)
    mesh, ch, o = make(pkg, L, M, N, 1.8, REN)
    _, ch2, _ = make(pkg, L, M, N, 1.8, REN)
    ch2.set_tuning(conv_dma=0, conv_lds=0, conv_fx=0)
    for c in (ch, ch2):
        c.SOLVERRK3_MOM_tg(0, dt, 1.0 / REN)
        for _ in range(2):
            c.rk3_step(dt, 1.0 / REN)
    o.substep(0, dt)
    for _ in range(2):
        o.step(dt)
    q, p = ch.download()
    q2, p2 = ch2.download()
    assert max(rel(q[c], o.q[c]) for c in range(3)) < 1e-10
    assert rel(p, o.pr) < 1e-9
    assert max(rel(q[c], q2[c]) for c in range(3)) < 1e-13
    ch.close()
    ch2.close()


@pytest.mark.parametrize("L,M,N,mode", [(64, 64, 64, "plain"), (64, 30, 32, "mixed"), (72, 33, 40, "plain"), (72, 33, 40, "mixed")])
def test_y_chunks_by_mesh_change_no_bit(pkg, L, M, N, mode):
    """The rows per chunk of the marching y-solves, chosen by the mesh, change no result: equal to
    48-row chunks bit for bit."""
    q, p = oracle.initial_field(setup.Mesh(L, M, N, STR2=1.8), 3)
    out = []
    for kv in ({}, dict(cnzy_ky=min(48, M), cny3_ky=min(48, M))):
        ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.8), pkg.MIXED if mode == "mixed" else pkg.PLAIN_FP64)
        ch.set_tuning(**kv)
        ch.upload(q, p)
        ch.rk3_step(1.0e-3, 1.0 / 2800.0)
        out.append(ch.download())
        ch.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("L,M,N", [(16, 4, 18), (64, 64, 64), (18, 80, 96), (12, 71, 120), (10, 35, 256), (30, 100, 36),
                                   (20, 97, 90), (6, 18, 162), (8, 16, 512), (24, 12, 30)])
def test_spectral_plane_in_one_block_matches_oracle(pkg, L, M, N):
    """The z-transforms and the y-Thomas of a kx in one block (planes up to 160 KB of LDS: chunks of 4, 8
    and 12 rows, the last short or empty, two- and three-pass z-plans) against the oracle (bound as
    test_poisson_matches_oracle), and both gauges against the separate kernels (ytdma_c = 16),
    which differ by rounding (bound as test_wide_ytdma_matches_serial_lines)."""
    mesh = setup.Mesh(L, M, N, STR2=1.9)
    r = np.random.default_rng(M + N).standard_normal((N, M, L))
    w = (1.0 / mesh.DYFI)[None, :, None]
    r -= np.sum(r * w) / (np.sum(w) * L * N)
    ref = oracle.OracleTG(mesh, 2800.0).poisson(r)
    ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.9), pkg.PLAIN_FP64)
    got = [ch.poisson(r), ch.FISHPACK_POIS3D_SIMPLE(r)]
    assert rel(got[0], ref) < 1e-10
    ch.set_tuning(ytdma_c=16)
    for a, b in zip(got, [ch.poisson(r), ch.FISHPACK_POIS3D_SIMPLE(r)]):
        assert rel(a, b) < 1e-10, rel(a, b)
    ch.close()


@pytest.mark.parametrize("L,M,N", [(64, 132, 64), (128, 192, 64), (64, 256, 50), (48, 161, 128)])
def test_fp32_wide_ytdma_changes_no_bit(pkg, L, M, N):
    """The mixed form's chunked y-solve keeps its 16-row chunks (M = 129 .. 256) in the kernel with 16
    lines per wavefront: the same sums in the same order as with 64 lines (ytdma_c = 16), bit for bit."""
    q, p = oracle.initial_field(setup.Mesh(L, M, N, STR2=1.8), 3)
    out = []
    for kv in ({}, dict(ytdma_c=16)):
        ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.8), pkg.MIXED)
        ch.set_tuning(**kv)
        ch.upload(q, p)
        for _ in range(2):
            ch.rk3_step(1.0e-3, 1.0 / 2800.0)
        out.append(ch.download())
        ch.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("L,M,N,mode", [(64, 192, 256, "mixed"), (64, 160, 256, "mixed"), (64, 64, 64, "plain")])
def test_convection_march_by_mesh_is_near_the_best(pkg, L, M, N, mode):
    """The planes per march that the mesh chooses: within 12 % of the fastest of a few set by hand
    (kernel times; a march too long for the blocks a CU holds cost 23 % at 64x192x256)."""
    ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.8), pkg.MIXED if mode == "mixed" else pkg.PLAIN_FP64)
    ch.upload(*oracle.initial_field(setup.Mesh(L, M, N, STR2=1.8), 3))

    def kernel_ms():
        for _ in range(3):
            ch.rk3_step(5.0e-4, 1.0 / 2800.0)
        ch.profile_reset("conv_rhs")
        for _ in range(20):
            ch.rk3_step(5.0e-4, 1.0 / 2800.0)
        return ch.profile_get("conv_rhs")[0]

    auto, by_hand = kernel_ms(), {}
    for kc in (4, 8, 16, 26):
        ch.set_tuning(conv_kc=kc)
        by_hand[kc] = kernel_ms()
    print(f"  by the mesh {auto:.4f} ms, by hand {by_hand}")
    assert auto < 1.12 * min(by_hand.values())
    ch.close()


def test_default_shapes_can_be_set_again(pkg):
    """None (CHS_TUNE_DEFAULT) puts back what a context was made with, the choices by the mesh among
    them: after other values for every key and None again, a step gives a fresh channel's bits
    (conv_kc, conv_by and conv_fx change the mass flux's last bits, ytdma_c and fft_reg the solve's)."""
    L, M, N = 48, 36, 40
    q, p = oracle.initial_field(setup.Mesh(L, M, N, STR2=2.0), 3)
    other = dict(conv_by=16, conv_kc=3, conv_fence=1, conv_fx=0, conv_lds=1, conv_dma=0, cnx_nlx=3, cnz_kz=5, cny_ky=7,
                 cn_xz=1, cnxz_by=2, fftx_tk=2, fftz_nl=1, nxcd=3, fft_reg=0, ytdma_bs=128, ytdma_rb=8, ytdma_c=0,
                 divg_nxcd=1, cny3_ky=-1, upd_kz=7, upd_by=2, upd_nxcd=3, upd_w2=0, cnzy=2, cnzy_ky=20, cnzy_nxcd=1)
    for mode in (pkg.PLAIN_FP64, pkg.MIXED):
        out = []
        for reset in (False, True):
            ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=2.0), mode)
            ch.upload(q, p)
            if reset:
                ch.set_tuning(**other)
                ch.rk3_step(8.0e-4, 1.0 / 4000.0)
                ch.upload(q, p, np.zeros((3, N, M, L)))
                ch.set_tuning(**{k: None for k in other}, conv_bx=None)
            for _ in range(2):
                ch.rk3_step(8.0e-4, 1.0 / 4000.0)
            ch.profile_reset(None)
            ch.rk3_step(8.0e-4, 1.0 / 4000.0)
            out.append((*ch.download(), [ch.profile_get(k)[1] for k in ("conv_rhs", "cn_x", "cn_xz", "cn_z", "cn_y", "cn_zy",
                                                                         "spec_plane", "ytdma")]))
            with pytest.raises(pkg.ChsError):
                ch.set_tuning(no_such_key=None)
            ch.close()
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
        assert out[0][2] == out[1][2]


@pytest.mark.parametrize("L,M,N", [(48, 9, 90), (90, 6, 48), (120, 5, 150), (150, 7, 120), (250, 4, 54), (12, 5, 486), (96, 80, 96)])
def test_lds_transforms_match_oracle(pkg, L, M, N):
    """The LDS transforms (fft_reg = 0; what batched ensembles launch, and lengths without a plan)
    at lengths with factors 3 and 5 that the mixed-radix plans otherwise take, bounds as
    test_poisson_matches_oracle."""
    print(f"lds poisson {L}x{M}x{N}", flush=True)
    mesh = setup.Mesh(L, M, N, STR2=1.9)
    r = np.random.default_rng(L + N).standard_normal((N, M, L))
    w = (1.0 / mesh.DYFI)[None, :, None]
    r -= np.sum(r * w) / (np.sum(w) * L * N)
    ref = oracle.OracleTG(mesh, 2800.0).poisson(r)
    for mode, tol in ((pkg.PLAIN_FP64, 1e-10), (pkg.MIXED, 1e-5)):
        ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.9), mode)
        ch.set_tuning(fft_reg=0)
        phi = ch.poisson(r)
        assert rel(phi, ref) < tol, (mode, rel(phi, ref))
        ch.close()


@pytest.mark.parametrize("kv", [dict(fftx_tk=2, fftz_nl=1), dict(fftx_tk=8, fftz_nl=5), dict(fftx_tk=4, fftz_nl=51)])
def test_lds_transform_tilings_match_oracle(pkg, kv):
    """fftx_tk and fftz_nl shape the LDS transforms alone (fft_reg = 0): other tilings give the oracle's
    step to test_launch_shapes_keep_results' bounds."""
    L, M, N, STR2, REN, dt = 48, 36, 40, 2.0, 4000.0, 8.0e-4
    print(f"lds tilings {kv}", flush=True)
    mesh, ch, o = make(pkg, L, M, N, STR2, REN)
    ch.set_tuning(fft_reg=0, **kv)
    ch.SOLVERRK3_MOM_tg(0, dt, 1.0 / REN)
    o.substep(0, dt)
    for _ in range(2):
        ch.rk3_step(dt, 1.0 / REN)
        for ns in (1, 2, 3):
            o.substep(ns, dt)
    gq, gp = ch.download()
    assert max(rel(gq[c], o.q[c]) for c in range(3)) < 1e-10 and rel(gp, o.pr) < 1e-10
    ch.close()


@pytest.mark.parametrize("L,M,N", [(128, 20, 16), (192, 12, 18), (64, 24, 32)])
def test_lds_convection_matches_oracle(pkg, L, M, N):
    """The convection kernel that stages its rows through registers (conv_lds rows), which the
    direct-to-LDS one stands in for unless conv_dma = 0."""
    STR2, REN, dt = 2.0, 4000.0, 8.0e-4
    for rows in (1, 2, 4):
        print(f"lds convection {L}x{M}x{N} rows {rows}", flush=True)
        mesh, ch, o = make(pkg, L, M, N, STR2, REN)
        ch.set_tuning(conv_dma=0, conv_lds=rows)
        ch.SOLVERRK3_MOM_tg(0, dt, 1.0 / REN)
        o.substep(0, dt)
        ch.rk3_step(dt, 1.0 / REN)
        for ns in (1, 2, 3):
            o.substep(ns, dt)
        gq, gp = ch.download()
        assert max(rel(gq[c], o.q[c]) for c in range(3)) < 1e-10 and rel(gp, o.pr) < 1e-10
        ch.close()


@pytest.mark.parametrize("L,M,N", [(64, 64, 64), (64, 20, 96), (128, 12, 64), (256, 12, 256), (512, 8, 512), (1024, 6, 64),
                                   (96, 80, 96), (256, 192, 64), (16, 16, 16)])
def test_poisson_entry_points_agree_to_the_bit(pkg, L, M, N):
    """The host entry point's solution (through the halo field) and the device one's (cells) are the same
    bits for each kind of x-transform, in both forms."""
    co = pkg.channel_setup(L, M, N, STR2=1.9)
    r = np.random.default_rng(L + N).standard_normal((N, M, L))
    for mode in (pkg.PLAIN_FP64, pkg.MIXED):
        ch = pkg.ChannelTG(co, mode)
        phi = ch.poisson(r)
        d_r, d_p = pkg.DeviceArray.from_host(r), pkg.DeviceArray(r.shape)
        ch.poisson_device(d_r.ptr, d_p.ptr, 0, False)
        ch.sync()
        assert np.array_equal(d_p.to_host(), phi), mode
        for d in (d_r, d_p):
            d.free()
        ch.close()


@pytest.mark.parametrize("L,M,N", [(512, 20, 512), (512, 84, 250), (1024, 22, 200), (512, 16, 500)])
def test_long_x_lines_each_side_of_the_rule(pkg, L, M, N):
    """L >= 512 takes the register plan's x-transforms on small meshes and the mixed-radix ones on large, the
    forward and the inverse each from a size of its own: both mixes against the oracle, bounds as
    test_poisson_matches_oracle."""
    print(f"long x lines {L}x{M}x{N}", flush=True)
    test_mixed_radix_poisson_matches_oracle_and_device_output(pkg, L, M, N)


@pytest.mark.parametrize("L,M,N,mode", [(1280, 64, 128, "mixed"), (1280, 64, 128, "plain"), (1024, 96, 128, "mixed")])
def test_forward_transform_tile_order_is_the_faster(pkg, L, M, N, mode):
    """Rows grouped by XCD or in dispatch order, whichever the mesh chose: within 8 % of the faster of the
    two (short runs of the spectrum grouped cost 28 to 38 % at 1280x64x128)."""
    ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.8), pkg.MIXED if mode == "mixed" else pkg.PLAIN_FP64)
    rng = np.random.default_rng(1)
    ch.upload(1e-3 * rng.standard_normal((3, N, M + 2, L)), np.zeros((N, M + 2, L)))

    def kernel_ms():
        for _ in range(2):
            ch.rk3_step(1.0e-6, 1.0 / 2800.0)
        ch.profile_reset("divg_fftx")
        for _ in range(10):
            ch.rk3_step(1.0e-6, 1.0 / 2800.0)
        return ch.profile_get("divg_fftx")[0]

    auto, by_hand = kernel_ms(), []
    for nx in (1, 8):
        ch.set_tuning(divg_nxcd=nx)
        by_hand.append(kernel_ms())
    print(f"  by the mesh {auto:.4f} ms, dispatch order and grouped {by_hand}")
    assert auto < 1.08 * min(by_hand)
    ch.close()


@pytest.mark.parametrize("L,M,N", [(128, 256, 128), (128, 224, 128), (128, 144, 128), (64, 250, 64)])
def test_wide_ytdma_is_no_slower_than_the_chunks_it_replaces(pkg, L, M, N):
    """The y-Thomas that the mesh chooses against 16-row chunks of 64 lines (ytdma_c = 16), kernel times
    within 8 % (12-row chunks at M = 256, six wavefronts a block, took 23 % longer)."""
    ch = pkg.ChannelTG(pkg.channel_setup(L, M, N, STR2=1.9), pkg.PLAIN_FP64)
    d_r = pkg.DeviceArray.from_host(np.random.default_rng(1).standard_normal((N, M, L)))
    d_p = pkg.DeviceArray((N, M, L))

    def kernel_ms():
        for _ in range(3):
            ch.poisson_device(d_r.ptr, d_p.ptr, 0, False)
        ch.profile_reset("ytdma")
        for _ in range(20):
            ch.poisson_device(d_r.ptr, d_p.ptr, 0, False)
        return ch.profile_get("ytdma")[0]

    auto = kernel_ms()
    ch.set_tuning(ytdma_c=16)
    chunks = kernel_ms()
    print(f"  {L}x{M}x{N}: by the mesh {auto:.4f} ms, 16-row chunks {chunks:.4f} ms")
    assert auto < 1.08 * chunks
    for d in (d_r, d_p):
        d.free()
    ch.close()
