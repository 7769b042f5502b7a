"""Sweeps, products, assembly, coarse inverse and Arnoldi vectors at the sizes
where their kernels change: levels of 3^3 .. 33^3 nodes (one workgroup, a
workgroup per plane, a launch per line group), lines longer than a wavefront,
single panels of the coarse inverse and its size limit, one workgroup against
many in the norms.

Tolerances: FP64 sweeps, products and entries agree with the oracle within
1e-12 of the largest value (some hundred roundings of 1.1e-16 per row and
sweep); variants of one sweep agree bit for bit."""
import numpy as np
import pytest

import orc
import parmoon_amd as pa
from parmoon_amd import prm as P
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("order,nref0,nlev", [(1, 1, 5), (2, 1, 4)])
def test_sweeps_match_the_oracle(ctx, order, nref0, nlev):
    S, O = pa.System(ctx, nref0, nlev, order), orc.System(nref0, nlev, order)
    blk = P.config1b() if order == 1 else P.config2(nref=nref0 + nlev - 1)
    S.assemble(blk)
    O.assemble(blk)
    rng = np.random.default_rng(3)
    for lev in range(nlev):
        sp, E = O.levels[lev], O.entries(lev)
        x, b = rng.standard_normal(sp.N), rng.standard_normal(sp.N)
        rows = np.argsort(S.colours(lev)[:sp.active], kind="stable").astype(np.int32)
        for kind, omega, sweeps in [(2, 1.0, 1), (2, 0.7, 2), (3, 1.0, 1), (3, 0.7, 2), (3, 1.0, 3)]:
            print(f"[case] order {order} level {lev} ({sp.N} nodes) kind {kind} omega {omega} x {sweeps}", flush=True)
            ref = x
            for _ in range(sweeps):
                ref = sp.smooth_ordered(E, kind, omega, ref, b, rows)
            assert rel(S.smooth(kind, omega, sweeps, x, b, level=lev), ref) < 1e-12
    S.close()


@pytest.mark.parametrize("order,nref0,nlev,precision", [(1, 1, 5, 0), (1, 1, 5, 1), (2, 1, 4, 0), (2, 1, 4, 1)])
def test_plane_sweeps_equal_line_sweeps(ctx, order, nref0, nlev, precision):
    print(f"[case] planes against line groups, order {order} precision {precision}", flush=True)
    S = pa.System(ctx, nref0, nlev, order)
    S.assemble(P.config1b() if order == 1 else P.config2(nref=nref0 + nlev - 1))
    rhs = S.rhs()
    n, na = int(S.dims()[0]), int(S.dims()[1])
    sol0 = np.zeros(n)
    sol0[na:] = rhs[na:] + 0.25  # (Dirichlet values that are not zero)
    for pre, post, smoother in [(3, 1, 3), (1, 2, 3), (2, 2, 2)]:
        base = dict(solver=16, restart=20, maxit=6, res_norm_min=0.0, red_factor=0.0, smoother=smoother, omega=1.0,
                    pre=pre, post=post, precision=precision)
        a, ia, _ = S.solve(P.solver_opt(wg_sweep_rows=-1, **base), rhs, sol0, check=False)
        b, ib, _ = S.solve(P.solver_opt(wg_sweep_rows=0, **base), rhs, sol0, check=False)
        assert ia[0] == ib[0] and np.array_equal(a, b), (pre, post, smoother)
    S.close()


def test_lines_longer_than_a_wavefront(ctx):
    """257^3 Q1: 128 row pairs per line.  The sweep against its definition,
    colour by colour with residuals; the products against each other."""
    S = pa.System(ctx, 7, 2, 1)
    S.assemble(P.config1b())
    d = S.dims()
    n, na = int(d[0]), int(d[1])
    col = S.colours()[:na]
    rng = np.random.default_rng(5)
    x, b = rng.standard_normal(n), rng.standard_normal(n)
    diag, ref = np.zeros(na), x.copy()
    ref[na:] = b[na:]
    for c in range(8):
        e = np.zeros(n)
        e[:na][col == c] = 1.0
        diag += np.where(col == c, S.matvec(e)[:na], 0.0)
        print(f"[case] diagonal of colour {c}", flush=True)
    for c in [0, 1, 2, 3, 4, 5, 6, 7, 7, 6, 5, 4, 3, 2, 1, 0]:
        r, _ = S.defect(ref, b)
        ref[:na] += np.where(col == c, r[:na] / diag, 0.0)
        print(f"[case] residual before colour {c}", flush=True)
    assert rel(S.smooth(3, 1.0, 1, x, b), ref) < 1e-12
    assert rel(S.matvec(x, precision=1), S.matvec(x)) < 1e-5
    S.close()


@pytest.mark.parametrize("order,nref,example,linear", [(1, 1, "sine", True), (1, 2, "lognormal", False),
                                                       (1, 3, "sine", False), (1, 4, "curl", True),
                                                       (2, 1, "sine", True), (2, 1, "curl", False),
                                                       (2, 2, "lognormal", False), (2, 3, "sine", False)])
def test_entries_match_the_oracle(ctx, order, nref, example, linear):
    print(f"[case] assembly order {order} nref {nref} {example} linear {linear}", flush=True)
    if example == "curl":
        blk = P.config2(nref=nref, linear=linear)
    elif example == "lognormal":
        blk = P.lognormal(seed=2, nref=nref)
    else:
        blk = P.config1b()
    blk[P.LINEAR] = 1.0 if linear else 0.0
    S, O = pa.System(ctx, nref, 1, order), orc.System(nref, 1, order)
    S.assemble(blk)
    O.assemble(blk)
    assert rel(S.entries(), O.entries()) < 1e-12
    assert rel(S.rhs(), O.rhs()) < 1e-12
    S.close()


@pytest.mark.parametrize("nref", [1, 3, 5])
@pytest.mark.parametrize("example,linear", [("laplace", True), ("laplace", False), ("sine", True), ("sine", False),
                                            ("heat", False)])
def test_q1_rows_of_constant_coefficients(ctx, nref, example, linear):
    """Rows and right-hand sides with a reaction and a time, 8 and 27 points."""
    print(f"[case] Q1 rows nref {nref} {example} linear {linear}", flush=True)
    if example == "heat":
        blk = P.heat_amc(0.3)
    elif example == "laplace":
        blk = P.base(P.EX_LAPLACE, eps=0.7)
    else:
        blk = P.base(P.EX_SINE_CD, eps=1e-2, form=P.FORM_SDFEM, b=(0.3, -1.0, 0.5), c=0.7)
    blk[P.LINEAR] = 1.0 if linear else 0.0
    S, O = pa.System(ctx, nref, 1, 1), orc.System(nref, 1, 1)
    S.assemble(blk)
    O.assemble(blk)
    assert rel(S.entries(), O.entries()) < 1e-12
    assert rel(S.rhs(), O.rhs()) < 1e-12
    S.close()


def test_two_matrices_of_constant_coefficients(ctx):
    """A step of the SUPG time form with the sine coefficients: solution against
    the oracle's, both solved to 1e-10 of the residual or better."""
    print("[case] TCD SUPG step, sine coefficients, 8^3 Q1", flush=True)
    from test_gpu_tcd_supg import supg_opt
    prm = P.base(P.EX_SINE_CD, eps=1e-2, form=P.FORM_TCD_SUPG_AK, b=(0.3, -1.0, 0.5))
    S, O = pa.System(ctx, 1, 3, 1), orc.System(1, 3, 1)
    u0 = orc.Space(3, 1).interpolate(prm)
    S.tcd_init(prm, u0)
    p = prm.copy()
    p[P.TIME] = 1e-2
    S.tcd_step(p, [1e-2, .5, .5, .5, .5], supg_opt(0))
    O.set_multicolour()
    ref, _ = O.tcd3d(prm, [1e-2, 1.5e-2, .5, .5, .5, .5], supg_opt(), u0, max_steps=1)
    assert rel(S.solution(), ref) < 1e-9
    S.close()


@pytest.mark.parametrize("order,alpha", [(1, 0.02), (1, 19.0), (1, 20.0 - 1e-9), (1, 20.0 + 1e-9), (2, 22.0),
                                         (1, 1e9)])
def test_streamline_parameter_around_its_limit(ctx, order, alpha):
    """delta = (coth a - 1/a) hK / (2 |b|) with the local Peclet number a on both
    sides of the value from which coth a is 1 in FP64."""
    print(f"[case] streamline parameter, order {order} alpha {alpha}", flush=True)
    blk = P.config1b()
    nu = 1.0 / (blk[P.POLYDEG] if blk[P.POLYDEG] > 0 else 1.0)
    blk[P.EPS] = nu * np.linalg.norm(blk[P.B0:P.B2 + 1]) * np.sqrt(3.0) / 8 / (2 * alpha)
    S, O = pa.System(ctx, 3, 1, order), orc.System(3, 1, order)
    S.assemble(blk)
    O.assemble(blk)
    assert rel(S.entries(), O.entries()) < 1e-12
    assert rel(S.rhs(), O.rhs()) < 1e-12
    S.close()


@pytest.mark.parametrize("order,nref", [(1, 1), (1, 2), (1, 3), (2, 2), (1, 4)])
def test_exact_coarse_solve(ctx, order, nref):
    """One level: the cycle is the explicit inverse (1, 27, 343, 343 and 3375
    rows), so one step solves to its accuracy, 1e-16 times a condition below 1e5."""
    print(f"[case] one level, order {order} nref {nref}", flush=True)
    S = pa.System(ctx, nref, 1, order)
    S.assemble(P.config1b())
    rhs = S.rhs()
    n, na = int(S.dims()[0]), int(S.dims()[1])
    sol0 = np.zeros(n)
    sol0[na:] = rhs[na:]
    x, info, rc = S.solve(P.solver_opt(solver=16, restart=10, maxit=1, res_norm_min=0.0, red_factor=0.0, smoother=3,
                                       omega=1.0), rhs, sol0, check=False)
    assert info[1] < 1e-10 * info[2]
    S.close()


@pytest.mark.parametrize("order,nref", [(1, 3), (1, 4), (2, 4)])
def test_residual_norm_on_device_vectors(ctx, order, nref):
    """9^3 and 17^3 (one workgroup), 33^3 nodes; r may be b."""
    print(f"[case] residual norm order {order} nref {nref}", flush=True)
    S = pa.System(ctx, nref, 1, order)
    S.assemble(P.config1b())
    M = order * (1 << nref) + 1
    n = M ** 3
    rng = np.random.default_rng(7)
    x, b = rng.standard_normal(n), rng.standard_normal(n)
    hip = Hip()
    xd, bd, rd, res = hip.upload(x), hip.upload(b), hip.upload(np.zeros(n)), hip.upload(np.zeros(1))
    S.defect_noalloc(xd, bd, rd, res)
    ctx.sync()
    r, norm = hip.download(rd, n), hip.download(res, 1)[0]
    i = np.arange(n)
    surface = np.zeros(n, bool)
    for c in (i % M, i // M % M, i // (M * M)):
        surface |= (c == 0) | (c == M - 1)
    assert np.array_equal(r[surface], (b - x)[surface])
    assert abs(norm - np.linalg.norm(r)) < 1e-13 * np.linalg.norm(r)
    S.defect_noalloc(xd, bd, bd, res)
    ctx.sync()
    assert np.array_equal(hip.download(bd, n), r)
    hip.free()
    S.close()


@pytest.mark.parametrize("nref,restart,precision", [(2, 3, 0), (3, 7, 0), (4, 1, 0), (4, 12, 0), (4, 12, 1), (5, 12, 0)])
def test_arnoldi_at_small_sizes(ctx, nref, restart, precision):
    """125 .. 35937 nodes, restarts within and beyond the iterations: the
    solution of the oracle within the solves' tolerance."""
    print(f"[case] FGMRES({restart}) nref {nref} precision {precision}", flush=True)
    blk = P.config1b()
    S, O = pa.System(ctx, nref - 1, 2, 1), orc.System(nref - 1, 2, 1)
    S.assemble(blk)
    O.assemble(blk)
    rhs = O.rhs()
    sol0 = np.zeros_like(rhs)
    sol0[O.levels[-1].active:] = rhs[O.levels[-1].active:]
    base = dict(solver=16, maxit=400, res_norm_min=0.0, red_factor=0.0, rel_target=1e-11, smoother=3, omega=1.0)
    if nref == 5:
        base["coarse"] = 3  # (the 17^3 level by sweeps)
    x, info, rc = S.solve(P.solver_opt(restart=restart, precision=precision, **base), rhs, sol0)
    assert rc == 0 and info[1] <= 1e-11 * info[2] * 1.0001
    r, _ = O.levels[-1].defect(O.entries(), x, rhs)
    assert float(np.linalg.norm(r)) <= 1.1e-11 * info[2]
    S.close()


@pytest.mark.parametrize("nref", [1, 2, 3, 5, 6, 7])
@pytest.mark.parametrize("example", ["sine", "curl"])
def test_q2_rows_match_cell_matrices(ctx, nref, example):
    """The two-matrix form without stabilisation and the form of the right-hand
    side alone (a row per thread) against the one-matrix form (cell matrices):
    lines of 2 to 128 row pairs, several lines or a half of one per workgroup."""
    print(f"[case] Q2 rows against cell matrices nref {nref} {example}", flush=True)
    blk = (P.config2(nref=min(nref, 5)) if example == "curl" else
           P.base(P.EX_SINE_CD, eps=1e-2, b=(0.3, -1.0, 0.5), c=0.7, linear=True))
    blk[P.DELTA0] = 0.0
    S = pa.System(ctx, nref, 1, 2)
    x = np.random.default_rng(8).standard_normal(int(S.dims()[0]))
    out = {}
    for form in (P.FORM_TCD_A, P.FORM_TCD_SUPG_AK, P.FORM_RHS):
        b = blk.copy()
        b[P.FORM] = form
        S.assemble(b)
        out[form] = (S.matvec(x), S.rhs())
    assert rel(out[P.FORM_TCD_SUPG_AK][0], out[P.FORM_TCD_A][0]) < 1e-12
    assert rel(out[P.FORM_TCD_SUPG_AK][1], out[P.FORM_TCD_A][1]) < 1e-12
    assert rel(out[P.FORM_RHS][1], out[P.FORM_TCD_A][1]) < 1e-12
    S.close()


@pytest.mark.parametrize("order,nref", [(1, 1), (1, 2), (1, 3), (1, 4), (2, 1), (2, 2), (2, 3)])
@pytest.mark.parametrize("coarse", [1, 3])
def test_coarse_loop_matches_the_oracle(ctx, order, nref, coarse):
    """One level of 3^3 .. 17^3 nodes: the cycle is the coarse loop, three sweeps
    (reduction 0) or as many as its norms ask for."""
    print(f"[case] coarse loop order {order} nref {nref} coarse {coarse}", flush=True)
    S, O = pa.System(ctx, nref, 1, order), orc.System(nref, 1, order)
    blk = P.config1b() if order == 1 else P.config2(nref=nref)
    S.assemble(blk)
    O.assemble(blk)
    if coarse == 3:
        O.set_multicolour()
    sp = O.levels[-1]
    rng = np.random.default_rng(6)
    rhs, sol0 = rng.standard_normal(sp.N), rng.standard_normal(sp.N)
    sol0[sp.active:] = rhs[sp.active:]
    for sweeps, red in [(3, 0.0), (10, 0.3)]:
        opt = P.solver_opt(solver=11, maxit=2, res_norm_min=0.0, red_factor=0.0, omega=0.6, coarse=coarse,
                           coarse_sweeps=sweeps, coarse_red=red)
        ref, _ = O.solve(opt, rhs, sol0)
        got, _, _ = S.solve(opt, rhs, sol0, check=False)
        assert rel(got, ref) < 1e-12, (sweeps, red)
    S.close()


def test_relaxed_sweeps_of_long_lines(ctx):
    """257^3 Q1, two SSOR sweeps with omega 0.7: the turns within and between the
    sweeps, with the sums kept there, against the definition by residuals."""
    S = pa.System(ctx, 7, 2, 1)
    S.assemble(P.config1b())
    n, na = int(S.dims()[0]), int(S.dims()[1])
    col = S.colours()[:na]
    rng = np.random.default_rng(9)
    x, b = rng.standard_normal(n), rng.standard_normal(n)
    diag, ref = np.zeros(na), x.copy()
    ref[na:] = b[na:]
    for c in range(8):
        e = np.zeros(n)
        e[:na][col == c] = 1.0
        diag += np.where(col == c, S.matvec(e)[:na], 0.0)
    for c in 2 * (list(range(8)) + list(range(7, -1, -1))):
        r, _ = S.defect(ref, b)
        ref[:na] += np.where(col == c, 0.7 * r[:na] / diag, 0.0)
        print(f"[case] residual before colour {c}", flush=True)
    assert rel(S.smooth(3, 0.7, 2, x, b), ref) < 1e-12
    S.close()


def test_solves_on_long_lines(ctx):
    """257^3 Q1, five levels: sweeps from zero, kept sums in the defects and in A z,
    in FP64, FP32 and with FP16 values.  The residual that the solve reports is
    that of its solution, and the FP32 forms, which restart the Krylov space with
    every outer correction, take at most twice the iterations."""
    S = pa.System(ctx, 4, 5, 1)
    S.assemble(P.config1b())
    rhs = S.rhs()
    its = {}
    for prec in (0, 1, 3):
        print(f"[case] 257^3 Q1 solve, precision {prec}", flush=True)
        opt = P.solver_opt(solver=16, restart=30, maxit=200, res_norm_min=0.0, red_factor=0.0, rel_target=1e-8,
                           smoother=3, omega=1.0, precision=prec)
        info, rc = S.solve_resident(opt, check=False)
        assert rc == 0 and info[1] <= 1e-8 * info[2] * 1.0001, (prec, rc, info)
        _, res = S.defect(S.solution(), rhs)
        assert abs(res - info[1]) <= 1e-5 * res, (prec, res, info)
        its[prec] = int(info[0])
    print(f"iterations {its}", flush=True)
    assert max(its[1], its[3]) <= 2 * its[0]
    S.close()
