"""Parity of the HIP library with the CPU oracle on the same seeded inputs.

Integer results (iteration counts, broken flags) must be identical; FP64
fields agree within 1e-10 relative to the field's magnitude, the bar the
plain GPU form has to meet against the reference solver.
"""
import ctypes as C
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from conftest import tail_close
from solver_cpp_amd.capi import ptr
from solver_cpp_amd.geometry import CONFIGS, EXAMPLE_NUMERICS, polycrystal, uniform_orientations
from solver_cpp_amd.rve import Rve, tension_x

pytestmark = pytest.mark.gpu
IP = C.POINTER(C.c_int)
REL = 1e-10  # per-point tolerance of the plain FP64 form


def close(a, b, rel=REL, what=""):
    a, b = np.asarray(a), np.asarray(b)
    scale = max(np.abs(b).max(), 1e-300)
    err = np.abs(a - b).max() / scale
    assert err <= rel, f"{what}: max |diff| / max |ref| = {err:.3e} > {rel:.1e}"


def test_backend(product):
    assert product.backend == "hip-gfx950"


# ---- spectral stages ---------------------------------------------------------------
# generic lengths, and the compile-time pencil lengths (2^a from 8, 3 * 2^a from
# 12, 9 * 2^a from 18, and 27) in every axis, with odd and even numbers of x rows
FFT_CELLS = [(2, 1, 1), (4, 3, 5), (8, 8, 8), (6, 10, 7), (16, 12, 9), (32, 32, 32), (20, 14, 22), (8, 3, 3),
             (12, 24, 16), (128, 8, 6), (24, 48, 12), (96, 2, 64), (256, 2, 3), (512, 1, 1), (384, 3, 1),
             (192, 2, 12), (18, 36, 27), (72, 27, 18), (144, 3, 36), (288, 2, 1), (27, 8, 72), (54, 18, 9)]


@pytest.mark.parametrize("cells", FFT_CELLS)
def test_fft_r2c_c2r(product, oracle, cells):
    rng = np.random.default_rng(sum(cells))
    c = np.array(cells, dtype=np.int32)
    N = int(np.prod(cells))
    K = (cells[0] // 2 + 1) * cells[1] * cells[2]
    howmany = 9
    f = rng.standard_normal(howmany * N)
    a, b = np.zeros(2 * howmany * K), np.zeros(2 * howmany * K)
    product.check(product.sc_fft_r2c(ptr(c, IP), howmany, ptr(f), ptr(a)), "fft_r2c")
    oracle.sc_fft_r2c(ptr(c, IP), howmany, ptr(f), ptr(b))
    close(a, b, 1e-13, "r2c")
    back = np.zeros_like(f)
    product.check(product.sc_fft_c2r(ptr(c, IP), howmany, ptr(a), 1.0 / N, ptr(back)), "fft_c2r")
    close(back, f, 1e-13, "c2r(r2c(f)) / N")


def _xi(lib, cells, size, derivative=0):
    c = np.array(cells, dtype=np.int32)
    K = (cells[0] // 2 + 1) * cells[1] * cells[2]
    x1, x2 = np.zeros(6 * K), np.zeros(6 * K)
    lib.sc_spectral_xi(ptr(c, IP), ptr(np.array(size, dtype=float)), derivative, ptr(x1), ptr(x2))
    return x1, x2


@pytest.mark.parametrize("derivative", [0, 1, 2])
def test_xi_tables(product, oracle, derivative):
    cells, size = (6, 5, 4), (6e-5, 5e-5, 4e-5)
    for a, b in zip(_xi(product, cells, size, derivative), _xi(oracle, cells, size, derivative)):
        close(a, b, 1e-15, "xi")


@pytest.mark.parametrize("cells", [(4, 4, 4), (6, 5, 8), (16, 16, 16)])
def test_divergence_and_gamma(product, oracle, cells):
    rng = np.random.default_rng(3)
    c = np.array(cells, dtype=np.int32)
    size = np.array(cells, dtype=float) * 1e-6
    N = int(np.prod(cells))
    xi1, _ = _xi(oracle, cells, size)
    field = rng.standard_normal(9 * N) * 1e7
    scaled = np.zeros(3)
    oracle.sc_scaled_geom_size(ptr(c, IP), ptr(size), 2, ptr(scaled))
    r1, r2 = np.zeros(1), np.zeros(1)
    product.check(product.sc_divergence_rms(ptr(c, IP), ptr(size), ptr(scaled), ptr(xi1), ptr(field), ptr(r1)), "div")
    oracle.sc_divergence_rms(ptr(c, IP), ptr(size), ptr(scaled), ptr(xi1), ptr(field), ptr(r2))
    close(r1, r2, 1e-13, "divergence rms")
    A = rng.standard_normal((9, 9))
    C_ref = ((A @ A.T + 9 * np.eye(9)) * 1e10 * N).reshape(-1).copy()
    aim = rng.standard_normal(9) * 1e-3
    g1, g2 = field.copy(), field.copy()
    product.check(product.sc_gamma_convolution(ptr(c, IP), ptr(xi1), ptr(C_ref), ptr(aim), ptr(g1)), "gamma")
    oracle.sc_gamma_convolution(ptr(c, IP), ptr(xi1), ptr(C_ref), ptr(aim), ptr(g2))
    close(g1, g2, 1e-12, "Gamma * P")


def test_field_updates(product, oracle):
    rng = np.random.default_rng(5)
    n = 3000
    last, rate, f0 = (rng.standard_normal(9 * n) for _ in range(3))
    aim = rng.standard_normal(9)
    o1, o2 = np.zeros(9 * n), np.zeros(9 * n)
    product.check(product.sc_forward_field(n, 0.3, ptr(last), ptr(rate), ptr(aim), ptr(o1)), "forward_field")
    oracle.sc_forward_field(n, 0.3, ptr(last), ptr(rate), ptr(aim), ptr(o2))
    close(o1, o2, 1e-14, "forward_field")
    av = rng.standard_normal(9)
    for het in (0, 1):
        product.check(product.sc_calculate_rate(n, het, ptr(f0), ptr(last), 0.7, ptr(av), ptr(o1)), "rate")
        oracle.sc_calculate_rate(n, het, ptr(f0), ptr(last), 0.7, ptr(av), ptr(o2))
        close(o1, o2, 1e-15, "calculate_rate")


def test_response_reductions(product, oracle):
    rng = np.random.default_rng(6)
    n = 5000
    P = rng.standard_normal(9 * n) * 1e8
    d = rng.standard_normal(81 * n) * 1e10
    q = uniform_orientations(1, 4)[0]
    outs = []
    for lib in (product, oracle):
        pa, cv, cm = np.zeros(9), np.zeros(81), np.zeros(81)
        lib.check(lib.sc_response_reductions(n, ptr(P), ptr(d), ptr(q), ptr(pa), ptr(cv), ptr(cm)), "reductions")
        outs.append((pa, cv, cm))
    for a, b in zip(*outs):
        close(a, b, 1e-12, "reductions")


# ---- material point ------------------------------------------------------------------
def _mp_batch(lib, F, Fp0, dt, Lp=None, xi0=None, material=None):
    n = F.shape[0]
    m, p, _ = lib.defaults()
    if material:
        material(m)
    I9 = np.tile(np.eye(3).reshape(-1), (n, 1))
    Z9 = np.zeros((n, 9))
    xi0 = np.full((n, 12), m.xi_0_sl) if xi0 is None else xi0
    g0 = np.zeros((n, 12))
    Lp = np.zeros((n, 9)) if Lp is None else Lp.copy()
    out = {k: np.zeros((n, 9)) for k in ["P", "Fp", "S", "Fe"]}
    xi, ga = np.zeros((n, 12)), np.zeros((n, 12))
    d = np.zeros((n, 81))
    br = np.zeros(n, dtype=np.int32)
    it = np.zeros(2 * n, dtype=np.int32)
    rc = lib.sc_mp_update(n, dt, C.byref(m), C.byref(p), ptr(F), ptr(I9), ptr(Fp0), ptr(Z9), ptr(Z9), ptr(xi0),
                          ptr(g0), ptr(Lp), ptr(out["P"]), ptr(out["Fp"]), ptr(out["S"]), ptr(out["Fe"]), ptr(xi),
                          ptr(ga), ptr(d), ptr(br, IP), ptr(it, IP))
    lib.check(rc, "sc_mp_update")
    out.update(Lp=Lp, xi=xi, gamma=ga, dPdF=d, broken=br, iterations=it.reshape(n, 2))
    return out


def _random_batch(oracle, strain, n=4096):
    rng = np.random.default_rng(int(strain * 1e5))
    q = uniform_orientations(n, 11)
    Fp0 = np.zeros((n, 9))
    for c in range(n):
        oracle.sc_qu2om(ptr(q[c]), ptr(Fp0[c]))
    F = np.tile(np.eye(3).reshape(-1), (n, 1)) + strain * rng.uniform(-1, 1, (n, 9))
    return np.ascontiguousarray(F), Fp0


@pytest.mark.parametrize("strain", [5e-4, 1e-3, 2e-3])
def test_mp_update(product, oracle, strain):
    """Random grains and random deformation increments over dt = 0.5 s, from
    the load case's own step (5e-4) to four times it (fully plastic, ~24
    Newton iterations per point): identical iteration counts per point and
    every output within 1e-10."""
    F, Fp0 = _random_batch(oracle, strain)
    a = _mp_batch(product, F, Fp0, 0.5)
    b = _mp_batch(oracle, F, Fp0, 0.5)
    np.testing.assert_array_equal(a["broken"], b["broken"])
    np.testing.assert_array_equal(a["iterations"], b["iterations"])
    for k in ["P", "Fp", "Lp", "S", "Fe", "xi", "gamma", "dPdF"]:
        close(a[k], b[k], REL, k)
    # warm start from the returned Lp (the Newton guess of the next evaluation)
    a2 = _mp_batch(product, F, Fp0, 0.5, Lp=b["Lp"])
    b2 = _mp_batch(oracle, F, Fp0, 0.5, Lp=b["Lp"])
    np.testing.assert_array_equal(a2["iterations"], b2["iterations"])
    close(a2["P"], b2["P"], REL, "P (warm start)")


@pytest.mark.parametrize("n_sl,a_sl", [(10.0, 2.0), (17.3, 1.7)])
def test_mp_update_other_exponents(product, oracle, n_sl, a_sl):
    """Materials other than the example's n_sl = 20, a_sl = 2.25 run the
    runtime-exponent kernels: quarter exponents by binary powering, others
    by pow(); the oracle takes pow() throughout.  Same broken flags, the
    same iteration counts for at least 99 % of the points (a rounding-level
    difference of the powers may move a stopping decision) and every output
    of those within 1e-10, the consistent tangent included."""
    F, Fp0 = _random_batch(oracle, 1e-3)

    def material(m):
        m.n_sl, m.a_sl = n_sl, a_sl

    a = _mp_batch(product, F, Fp0, 0.5, material=material)
    b = _mp_batch(oracle, F, Fp0, 0.5, material=material)
    np.testing.assert_array_equal(a["broken"], b["broken"])
    assert not b["broken"].any()
    same = (a["iterations"] == b["iterations"]).all(axis=1)
    assert same.mean() >= 0.99, same.mean()
    for k in ["P", "Fp", "Lp", "S", "Fe", "xi", "gamma", "dPdF"]:
        close(a[k][same], b[k][same], REL, k)
    # points whose counts differ: within the stopping tests' own spread
    if (~same).any():
        for k in ("P", "Fp", "xi"):
            v = float(np.abs(a[k][~same] - b[k][~same]).max() / np.abs(b[k]).max())
            print(f"exponents {n_sl}/{a_sl}: {(~same).sum()} points with other counts, {k} spread {v:.2e}",
                  flush=True)
            assert v <= 5e-5, (k, v)


@pytest.mark.parametrize("n", [1, 63, 64, 65])
@pytest.mark.parametrize("kind", ["example", "powers", "pow", "no C44", "no C11 - C12"])
def test_mp_update_edges(product, oracle, n, kind):
    """Callers' point updates around one wave's width, for the example's
    exponents, quarter exponents and general ones, and for the two stiffnesses
    whose Newton system is scaled instead of divided by the stiffness.  Every
    output of the points with the oracle's counts within 1e-10 (the two solve
    the same equations to a stopping test that both meet or miss alike); a
    stopping decision at its threshold may move for 1 point in 100, so at most
    two points here have other counts (none where there is one point), and they
    agree within the stopping tests' spread.  No point is broken."""
    F, Fp0 = _random_batch(oracle, 1e-3, n=65)
    F, Fp0 = F[:n].copy(), Fp0[:n].copy()

    def material(m):
        if kind in ("powers", "pow"):
            m.n_sl, m.a_sl = (10.0, 2.0) if kind == "powers" else (17.3, 1.7)
        if kind == "no C44":
            m.C_44 = 0.0
        if kind == "no C11 - C12":
            m.C_11 = m.C_12

    a = _mp_batch(product, F, Fp0, 0.5, material=material)
    b = _mp_batch(oracle, F, Fp0, 0.5, material=material)
    assert not a["broken"].any() and not b["broken"].any()
    same = (a["iterations"] == b["iterations"]).all(axis=1)
    assert (~same).sum() <= (0 if n == 1 else 2)
    for k in ["P", "Fp", "Lp", "S", "Fe", "xi", "gamma", "dPdF"]:
        close(a[k][same], b[k][same], REL, k)
    for k in ("P", "Fp", "xi"):
        close(a[k], b[k], 5e-5, k)


def test_mp_update_substepping(product, oracle):
    """Steps of 2 % strain in 0.5 s force cutbacks and substeps.  The
    integration's stopping tests (Newton, state fixed point) then sit close
    to their thresholds for some points, so rounding decides between two
    valid results: two CPU builds of the oracle (with and without fused
    multiply-add) already disagree on 201 of these 4096 points.  Required:
    the same broken flags, at most 300 points with other iteration counts,
    the rest within 1e-10, and the points with other counts within twice the
    spread of those two oracle builds (measured on the same batch: P 1.41e-3,
    Fp 1.40e-4, xi 6.66e-4 of each field's maximum): a flipped stopping
    decision changes the substep sequence, and with it the time
    discretisation of the step, by that much and no more."""
    F, Fp0 = _random_batch(oracle, 2e-2)
    a = _mp_batch(product, F, Fp0, 0.5)
    b = _mp_batch(oracle, F, Fp0, 0.5)
    np.testing.assert_array_equal(a["broken"], b["broken"])
    same = (a["iterations"] == b["iterations"]).all(axis=1)
    assert (~same).sum() <= 300, (~same).sum()
    assert (b["iterations"][:, 1] > 12).any()  # substepping happened
    for k in ["P", "Fp", "Lp", "xi", "gamma"]:
        close(a[k][same], b[k][same], REL, k)
    diff = ~same & (b["broken"] == 0)
    spread = {k: float(np.abs(a[k][diff] - b[k][diff]).max() / np.abs(b[k]).max()) if diff.any() else 0.0
              for k in ("P", "Fp", "xi")}
    print(f"substepping: {diff.sum()} of {len(same)} points with other counts, spread {spread}", flush=True)
    bound = {"P": 2 * 1.41e-3, "Fp": 2 * 1.40e-4, "xi": 2 * 6.66e-4}
    for k, v in spread.items():
        assert v <= bound[k], (k, v)


# The grid solver updates its cells with kernels of its own (csrc/constitutive.hip);
# sc_mp_update runs the callers' (csrc/points.hip).  The tests above reach the
# latter, the ones below the former.
EXPONENTS = {"example": (20.0, 2.25), "powers": (10.0, 2.0), "pow": (17.3, 1.7)}


def _context_update(lib, F, ori, kind):
    """One residual evaluation of a 16^3 context with an orientation for every
    cell, at the given F, over 0.5 s from the undeformed state."""
    m, _, _ = lib.defaults()
    m.n_sl, m.a_sl = EXPONENTS[kind]
    r = Rve(lib, (16, 16, 16), (1e-5,) * 3, np.arange(4096), ori, material=m, **EXAMPLE_NUMERICS)
    try:
        r.init()
        r.forward(False, False, 0.5, 1.0, 10.0, tension_x(t=10.0, N=20))
        r.form_residual(F)
        out = {k: r.field(k).reshape(4096, -1) for k in ("P", "Fp", "Lp", "S", "Fe", "xi", "gamma")}
        out["iterations"] = r.field("iterations").reshape(4096, 2).astype(int)
        return out
    finally:
        r.close()


@pytest.mark.parametrize("kind", list(EXPONENTS))
def test_solver_update(product, oracle, kind):
    """The inputs of test_mp_update (1e-3) and test_mp_update_other_exponents
    through the solver's kernels, with those tests' requirements against the
    oracle, and against the callers' update of the same points."""
    F, Fp0 = _random_batch(oracle, 1e-3)
    ori = uniform_orientations(4096, 11)
    print(f"solver update: {kind}", flush=True)
    a, b = _context_update(product, F, ori, kind), _context_update(oracle, F, ori, kind)

    def material(m):
        m.n_sl, m.a_sl = EXPONENTS[kind]

    c = _mp_batch(product, F, Fp0, 0.5, material=material)
    assert not c["broken"].any()
    for other, what in ((b, "oracle"), (c, "callers' update")):
        same = (a["iterations"] == other["iterations"]).all(axis=1)
        assert same.mean() >= (1.0 if kind == "example" else 0.99), (what, same.mean())
        for k in ["P", "Fp", "Lp", "S", "Fe", "xi", "gamma"]:
            close(a[k][same], other[k][same], REL, f"{k} ({what})")
        for k in ("P", "Fp", "xi"):
            close(a[k], other[k], 5e-5, f"{k} ({what})")


def test_solver_update_substepping(product, oracle):
    """The inputs of test_mp_update_substepping through the solver's kernels: at
    most 300 of 4096 points with other counts than the oracle, the rest within
    1e-10.  Points with other counts are not compared here: on this path (Fp of
    the start state as init leaves it) two CPU builds of the oracle differ from
    each other on 215 points, by up to 1.5e-3 of P and 2.8e-4 of Fp."""
    F, _ = _random_batch(oracle, 2e-2)
    ori = uniform_orientations(4096, 11)
    a, b = _context_update(product, F, ori, "example"), _context_update(oracle, F, ori, "example")
    same = (a["iterations"] == b["iterations"]).all(axis=1)
    print(f"solver substepping: {(~same).sum()} points with other counts", flush=True)
    assert (~same).sum() <= 300, (~same).sum()
    assert (b["iterations"][:, 1] > 12).any()  # substepping happened
    for k in ["P", "Fp", "Lp", "xi", "gamma"]:
        close(a[k][same], b[k][same], REL, k)


# ---- outer solver ----------------------------------------------------------------------
def test_ngmres_replays_fortran_trace(product, trace):
    F, r, inc = trace["F"], trace["r"], trace["increment"]
    for i in range(1, 11):
        idx = np.where(inc == i)[0]
        x0 = np.ascontiguousarray(F[idx[0]])
        rr = np.ascontiguousarray(r[idx])
        xe = np.zeros_like(rr)
        product.check(product.sc_ngmres_replay(243, 30, ptr(x0), len(idx), ptr(rr), ptr(xe)), "replay")
        np.testing.assert_allclose(xe, F[idx], atol=1e-14, rtol=0)


# ---- full solver ------------------------------------------------------------------------
def _pair(product, oracle, cells, grains, seed=1, ori_seed=None, **kw):
    mat, ori, size = polycrystal(cells, grains, seed=seed, ori_seed=ori_seed)
    return Rve(product, cells, size, mat, ori, **kw), Rve(oracle, cells, size, mat, ori, **kw)


def test_first_increment_homogeneous_forward(product, oracle):
    """The first increment forwards a homogeneous field, whose average the
    reference takes with one add chain per component (its rounding error,
    all of one sign, is 8.1e-13 at 32^3 for F_xx = 1.0005).  The forwarded F
    must be the reference's to the last bits (not only to 1e-10): that
    offset stays in the average of F through the increment, and <P> of the
    first increment, small against the stiffness, moves by about 1e-8 of
    itself with it.  Checked: F after forward within 1e-15, then the whole
    first increment with identical counts and <P> within 1e-10."""
    cells = (32, 32, 32)
    a, b = _pair(product, oracle, cells, 24, seed=7, ori_seed=8, **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    load = tension_x(t=10.0, N=20)
    a.forward(False, False, 0.5, 1.0, 10.0, load)
    b.forward(False, False, 0.5, 1.0, 10.0, load)
    np.testing.assert_allclose(a.field("F"), b.field("F"), rtol=0, atol=1e-15)
    sa, sb = a.calculate_solution(), b.calculate_solution()
    assert (sa.required_iterations, sa.residual_evaluations) == (sb.required_iterations, sb.residual_evaluations)
    close(np.array(a.scalars().P_av), np.array(b.scalars().P_av), REL, "<P>")
    close(a.field("P"), b.field("P"), REL, "P")


@pytest.mark.parametrize("cells", [(16, 12, 8), (10, 6, 7), (80, 80, 80)])
def test_state_read_between_forward_and_solve(product, cells):
    """f_materialpoint_forward (phase_mechanical.f90:992-1007) copies the
    state into its start values.  A context instead exchanges the current and
    start buffers of Fp, S, xi and gamma, and a read that comes before the next
    material-point update takes the start ones.  Read right after the forward
    step, the fields are the previous increment's converged values, as after
    the copy, and the next increment is bitwise the one of a context whose
    fields were not read in between."""
    mat, ori, size = polycrystal(cells, 4, seed=11, ori_seed=12)
    load = tension_x(t=10.0, N=20)
    names = ["Fp", "S", "xi", "gamma"]
    rs = [Rve(product, cells, size, mat, ori, **EXAMPLE_NUMERICS) for _ in range(2)]
    try:
        for r in rs:
            r.init()
            r.forward(False, False, 0.5, 1.0, 10.0, load)
            r.calculate_solution()
        before = {k: rs[0].field(k) for k in names}
        assert not np.array_equal(before["gamma"], np.zeros_like(before["gamma"]))  # plastic
        for r in rs:
            r.forward(False, True, 0.5, 0.5, 9.5, load)
        for k in names:  # only the first context reads
            np.testing.assert_array_equal(rs[0].field(k), before[k], err_msg=k)
        sa, sb = rs[0].calculate_solution(), rs[1].calculate_solution()
        assert (sa.required_iterations, sa.residual_evaluations) == (sb.required_iterations, sb.residual_evaluations)
        for k in ["F", "P", "Fp", "S", "xi", "gamma"]:
            np.testing.assert_array_equal(rs[0].field(k), rs[1].field(k), err_msg=k)
    finally:
        for r in rs:
            r.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_field_reads_beside_each_other_and_a_solve(product, precision):
    """sc_rve_get_field writes nothing of the context.  Four threads read four
    fields of one context at once, each the same values every time; then two
    threads read P and the slip resistances while a third solves an increment:
    counts, scalars and fields are bitwise those of a context left alone."""
    cells = (24, 18, 16)
    print(f"concurrent reads: cells {cells} precision {precision}", flush=True)
    mat, ori, size = polycrystal(cells, 6, seed=15, ori_seed=16)
    load = tension_x(t=10.0, N=20)
    rs = [Rve(product, cells, size, mat, ori, precision=precision, **EXAMPLE_NUMERICS) for _ in range(2)]
    try:
        for r in rs:
            r.init()
            r.forward(False, False, 0.5, 1.0, 10.0, load)
            r.calculate_solution()
        names = ["P", "xi", "Fe", "gamma"]
        want = {k: rs[0].field(k) for k in names}
        with ThreadPoolExecutor(4) as ex:
            for k, got in ex.map(lambda k: (k, [rs[0].field(k) for _ in range(25)]), names):
                for g in got:
                    np.testing.assert_array_equal(g, want[k], err_msg=k)
        for r in rs:
            r.forward(False, True, 0.5, 0.5, 9.5, load)
        with ThreadPoolExecutor(3) as ex:
            solve = ex.submit(rs[0].calculate_solution)

            def watch(k):
                reads = 0
                while reads < 500 and not (solve.done() and reads):
                    rs[0].field(k)
                    reads += 1
                return reads

            reads = [ex.submit(watch, k) for k in ("P", "xi")]
            sa = solve.result()
            assert all(f.result() > 0 for f in reads)
        sb = rs[1].calculate_solution()
        assert (sa.required_iterations, sa.residual_evaluations) == (sb.required_iterations, sb.residual_evaluations)
        assert (sa.err_div, sa.err_BC) == (sb.err_div, sb.err_BC)
        for k in ["F", "P", "Fp", "S", "xi", "gamma"]:
            np.testing.assert_array_equal(rs[0].field(k), rs[1].field(k), err_msg=k)
    finally:
        for r in rs:
            r.close()


@pytest.mark.parametrize("derivative", [0, 1])
@pytest.mark.parametrize("cells", [(8, 8, 8), (16, 8, 16), (8, 16, 32), (16, 16, 64), (8, 8, 128), (64, 64, 64)])
def test_divergence_of_an_evaluation_equals_the_separate_launches(product, cells, derivative):
    """The divergence decides convergence, and a context alone (its convolution in
    one kernel with the z transforms) has to stop where a batch of it does (separate
    launches, the kernels of sc_divergence_rms).  err_div of a solution's last
    evaluation is bitwise the divergence of its P.  (A power-of-two cell count:
    the two scale the root by N in different ways, which are then the same.)"""
    assert np.log2(np.prod(cells)) % 1 == 0
    mat, ori, size = polycrystal(cells, 5, seed=17, ori_seed=18)
    r = Rve(product, cells, size, mat, ori, derivative=derivative, **EXAMPLE_NUMERICS)
    try:
        r.init()
        r.forward(False, False, 0.5, 1.0, 10.0, tension_x(t=10.0, N=20))
        sol = r.calculate_solution()
        c, size = np.array(cells, dtype=np.int32), np.array(size, dtype=float)
        scaled, rms = np.zeros(3), np.zeros(1)
        product.check(product.sc_scaled_geom_size(ptr(c, IP), ptr(size), r.desc.grid_num.divergence_correction,
                                                  ptr(scaled)), "scaled size")
        xi1, _ = _xi(product, cells, size, derivative)
        product.check(product.sc_divergence_rms(ptr(c, IP), ptr(size), ptr(scaled), ptr(xi1), ptr(r.field("P")),
                                                ptr(rms)), "divergence")
        assert sol.err_div == rms[0], (float(sol.err_div).hex(), float(rms[0]).hex())
    finally:
        r.close()


@pytest.mark.parametrize("cells", [(27, 18, 24), (20, 14, 22)])
def test_fft_plan_modes_give_the_same_bits(product, cells):
    """fft_plan_mode 1 (launch shapes timed per grid, like FFTW_MEASURE) and 0
    (built-in shapes, like FFTW_ESTIMATE) on pencil lengths (27, 18, 24) and
    generic ones (20, 14, 22): the same counts and bitwise the same fields."""
    mat, ori, size = polycrystal(cells, 6, seed=3, ori_seed=4)
    out = []
    for mode in (0, 1):
        r = Rve(product, cells, size, mat, ori, fft_plan_mode=mode, **EXAMPLE_NUMERICS)
        r.init()
        incs = [(d["iterations"], d["evaluations"]) for d, _ in zip(r.increments([tension_x(t=1.0, N=2)]), range(2))]
        out.append((incs, r.field("F"), r.field("P")))
        r.close()
    assert out[0][0] == out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("cells", [(8, 6, 4), (8, 6, 16), (7, 5, 12), (9, 8, 32), (6, 4, 64)])
def test_init_and_single_residual(product, oracle, cells):
    """Init, a solution and one residual at a perturbed F, over grids with odd
    and even x lengths and z lengths that take the pencil FFT (12, 16, 32,
    64) or the generic passes (4)."""
    print(f"single residual: cells {cells}", flush=True)
    a, b = _pair(product, oracle, cells, 5)
    a.init()
    b.init()
    sa, sb = a.scalars(), b.scalars()
    close(sa.C_minMaxAvg, sb.C_minMaxAvg, 1e-13, "C_minMaxAvg")
    close(sa.C_volAvg, sb.C_volAvg, 1e-13, "C_volAvg")
    close(a.field("x_p"), b.field("x_p"), 1e-14, "x_p")
    close(a.field("x_n"), b.field("x_n"), 1e-14, "x_n")
    load = tension_x(t=10.0, N=20)
    for R in (a, b):
        R.forward(False, False, 0.5, 1.0, 10.0, load)
    close(a.field("F"), b.field("F"), 1e-13, "forward F")
    # a solution then one more residual at a perturbed F
    sol_a, sol_b = a.calculate_solution(), b.calculate_solution()
    assert sol_a.required_iterations == sol_b.required_iterations
    assert sol_a.residual_evaluations == sol_b.residual_evaluations
    F = b.field("F") + 1e-5 * np.random.default_rng(2).standard_normal(9 * b.N)
    ra, rb = a.form_residual(F), b.form_residual(F)
    close(ra, rb, REL, "residual")
    close(a.field("P"), b.field("P"), REL, "P")


def test_loadcase_16cubed_20grains(product, oracle):
    """Plain FP64 on the CPU-runnable configuration: 16^3 grid, 20 Voronoi
    grains, uniaxial tension dot_F_xx = 1e-3/s to 1 % strain in 20 increments,
    N_iter_min/max = 4/40.  Per-point P and F within 1e-10, identical
    iteration and evaluation counts per increment."""
    cfg = CONFIGS["C1"]
    e = cfg["edge"]
    a, b = _pair(product, oracle, (e, e, e), cfg["grains"], cfg["seed"], cfg["ori_seed"], **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    load = [tension_x(t=cfg["t"], N=cfg["N"])]
    ia, ea = a.loop_over_loadcase(load)
    ib, eb = b.loop_over_loadcase(load)
    np.testing.assert_array_equal(ia, ib)
    np.testing.assert_array_equal(ea, eb)
    close(a.field("F"), b.field("F"), REL, "F")
    close(a.field("P"), b.field("P"), REL, "P")
    close(a.field("Fp"), b.field("Fp"), REL, "Fp")
    close(a.field("xi"), b.field("xi"), REL, "xi")
    close(a.scalars().P_av, b.scalars().P_av, REL, "P_av")
    close(a.field("x_p"), b.field("x_p"), 1e-12, "x_p")


@pytest.mark.parametrize("kind", ["powers", "pow"])
def test_loadcase_other_exponents(product, oracle, kind):
    """Five increments of tension (to 0.25 % strain, past the yield point) with
    exponents that are not compiled in: the solver's run-time instantiations of
    the update and of the tangent.  Same counts; a stopping decision that the
    powers' rounding moves is worth up to 5e-5 of a point's P (see
    test_mp_update_other_exponents) and n_sl = 20 times that in its tangent."""
    cells = (8, 6, 12)
    mat, ori, size = polycrystal(cells, 5, seed=23, ori_seed=24)
    print(f"load case: exponents {kind}", flush=True)
    rs = []
    for lib in (product, oracle):
        m, _, _ = lib.defaults()
        m.n_sl, m.a_sl = EXPONENTS[kind]
        r = Rve(lib, cells, size, mat, ori, material=m, **EXAMPLE_NUMERICS)
        r.init()
        rs.append((r, *r.loop_over_loadcase([tension_x(t=2.5, N=5)])))
    (a, ia, ea), (b, ib, eb) = rs
    np.testing.assert_array_equal(ia, ib)
    np.testing.assert_array_equal(ea, eb)
    assert b.field("gamma").max() > 1e-4  # plastic
    for k in ("F", "P", "Fp", "xi"):
        close(a.field(k), b.field(k), 5e-5, k)
    close(a.scalars().C_volAvg, b.scalars().C_volAvg, 1e-3, "C_volAvg")
    close(a.scalars().C_minMaxAvg, b.scalars().C_minMaxAvg, 1e-3, "C_minMaxAvg")


def test_loadcase_update_gamma(product, oracle):
    """update_gamma = 1 (MechSolverBasic::calculate_solution,
    mech_solver_basic.cpp:127 -> MechBase::update_gamma, mech_base.cpp:156-211):
    the reference stiffness of the Gamma operator is taken again from
    C_minMaxAvg before every solve instead of once at init.  12^3 grid, 8
    grains, 6 tension increments: identical iterations and evaluations, F,
    P and the final C_ref within 1e-10 of the oracle's."""
    cells = (12, 12, 12)
    a, b = _pair(product, oracle, cells, 8, seed=13, ori_seed=14, update_gamma=1, **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    load = [tension_x(t=3.0, N=6)]
    ia, ea = a.loop_over_loadcase(load)
    ib, eb = b.loop_over_loadcase(load)
    np.testing.assert_array_equal(ia, ib)
    np.testing.assert_array_equal(ea, eb)
    close(a.field("F"), b.field("F"), REL, "F")
    close(a.field("P"), b.field("P"), REL, "P")
    sa, sb = a.scalars(), b.scalars()
    close(sa.C_ref, sb.C_ref, 1e-12, "C_ref")


def test_loadcase_64cubed_200grains_first_increments(product, oracle):
    """The drop-in configuration (64^3 grid, 200 Voronoi grains, tension to
    2 % in 40 increments), its first two increments: identical iterations
    and evaluations, per-point F, P, Fp and xi within 1e-10 of the oracle.
    (Two increments keep the oracle's share to about half a minute.)"""
    cfg = CONFIGS["C2"]
    e = cfg["edge"]
    a, b = _pair(product, oracle, (e, e, e), cfg["grains"], cfg["seed"], cfg["ori_seed"], **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    load = [tension_x(t=cfg["t"], N=cfg["N"])]
    for ra, rb in zip(a.increments(load), b.increments(load)):
        print(f"64^3 increment {ra['increment']}: iterations {ra['iterations']} / {rb['iterations']}", flush=True)
        assert (ra["iterations"], ra["evaluations"]) == (rb["iterations"], rb["evaluations"])
        if ra["increment"] == 2:
            break
    close(a.field("F"), b.field("F"), REL, "F")
    close(a.field("P"), b.field("P"), REL, "P")
    close(a.field("Fp"), b.field("Fp"), REL, "Fp")
    close(a.field("xi"), b.field("xi"), REL, "xi")


@pytest.mark.parametrize("cells", [(32, 32, 32), (32, 24, 64)])
def test_mixed_precision_larger_pencils(product, oracle, cells):
    """Mixed form on grids whose FP32 pencils hold 16 points per thread (x, z
    lengths 32 and 64; y 24 with 12): first three increments of the tension
    load case against the FP64 oracle, within the bounds of the 16^3 test."""
    print(f"mixed precision: cells {cells}", flush=True)
    mat, ori, size = polycrystal(cells, 24, seed=7, ori_seed=8)
    a = Rve(product, cells, size, mat, ori, precision=1, **EXAMPLE_NUMERICS)
    b = Rve(oracle, cells, size, mat, ori, **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    load = [tension_x(t=10.0, N=20)]
    for ra, rb in zip(a.increments(load), b.increments(load)):
        if ra["increment"] == 3:
            break
    assert a.stats().fp32_evaluations > 0
    close(np.array(a.scalars().P_av), np.array(b.scalars().P_av), 2e-5, "<P>")
    close(a.field("P"), b.field("P"), 1e-4, "P")


@pytest.mark.parametrize("precision", [0, 1])
def test_profiling_changes_no_bits(product, precision):
    """Kernel timing brackets the launches of an evaluation with events and adds
    the sums of the iteration counts, which also make the scalars that the
    evaluation's last kernels send to the host more: counts, <P>, err_div and
    fields are bitwise those without it in every increment."""
    print(f"profiled: precision {precision}", flush=True)
    cells = (16, 12, 8)
    mat, ori, size = polycrystal(cells, 9, seed=21, ori_seed=22)
    runs = []
    for timed in (False, True):
        r = Rve(product, cells, size, mat, ori, precision=precision, **EXAMPLE_NUMERICS)
        r.init()
        r.profile(timed)
        trace = [(d["iterations"], d["evaluations"], r.scalars().P_av[:], r.scalars().err_div)
                 for d in r.increments([tension_x(t=4.0, N=8)])]
        runs.append((trace, r.field("F"), r.field("P"), r.field("xi")))
    (ta, Fa, Pa, xa), (tb, Fb, Pb, xb) = runs
    assert ta == tb
    np.testing.assert_array_equal(Fa, Fb)
    np.testing.assert_array_equal(Pa, Pb)
    np.testing.assert_array_equal(xa, xb)


def test_mixed_precision_16cubed(product, oracle):
    """Mixed form on the CPU-runnable configuration: FP32 transforms and Gamma
    (FP64 material point, FP64 norms) until the convergence criteria hold,
    then an FP64 solve continued from that F, against the FP64 oracle.  Both
    results satisfy the solver tolerances; they differ by a fraction of them:
    <P> within 2e-5 relative and every cell's P within 1e-4 of max |P|."""
    cfg = CONFIGS["C1"]
    e = cfg["edge"]
    mat, ori, size = polycrystal((e, e, e), cfg["grains"], seed=cfg["seed"], ori_seed=cfg["ori_seed"])
    a = Rve(product, (e, e, e), size, mat, ori, precision=1, **EXAMPLE_NUMERICS)
    b = Rve(oracle, (e, e, e), size, mat, ori, **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    load = [tension_x(t=cfg["t"], N=cfg["N"])]
    ia, ea = a.loop_over_loadcase(load)
    ib, eb = b.loop_over_loadcase(load)
    st = a.stats()
    assert st.fp32_evaluations > 0
    assert st.residual_evaluations - st.fp32_evaluations >= len(ia)  # every increment ends in FP64
    pa, pb = np.array(a.scalars().P_av), np.array(b.scalars().P_av)
    close(pa, pb, 2e-5, "<P>")
    close(a.field("P"), b.field("P"), 1e-4, "P")


def test_mixed_precision_128cubed(product, oracle):
    """The mixed-precision configuration (128^3 grid, 1000 Voronoi grains,
    tension to 3 % in 60 increments).  Anchored to the oracle at its own size
    by one residual evaluation after init and forward (P and r within 1e-10;
    the oracle's share is one 128^3 evaluation), then the first six
    increments of the mixed form against the GPU's FP64 form (itself held to
    the oracle by the 16^3 and 64^3 load-case tests): <P> within 2e-5 and
    every cell's P within 1e-4 of max |P| (both forms stop anywhere within
    eps_rel_div 5e-4), and with both at 1000-fold tighter tolerances over
    the first two increments <P> within 1e-6 (the error of precision
    itself)."""
    cfg = CONFIGS["C3"]
    e = cfg["edge"]
    mat, ori, size = polycrystal((e, e, e), cfg["grains"], seed=cfg["seed"], ori_seed=cfg["ori_seed"])
    load = [tension_x(t=cfg["t"], N=cfg["N"])]
    a = Rve(product, (e, e, e), size, mat, ori, **EXAMPLE_NUMERICS)
    b = Rve(oracle, (e, e, e), size, mat, ori, **EXAMPLE_NUMERICS)
    a.init()
    b.init()
    dt = cfg["t"] / cfg["N"]
    a.forward(False, False, dt, 1.0, cfg["t"], load[0])
    b.forward(False, False, dt, 1.0, cfg["t"], load[0])
    F = b.field("F")
    ra, rb = a.form_residual(F), b.form_residual(F)
    close(ra, rb, REL, "r (128^3)")
    close(a.field("P"), b.field("P"), REL, "P (128^3)")
    a.close()
    b.close()
    del b

    def run(precision, n, **num):
        r = Rve(product, (e, e, e), size, mat, ori, precision=precision, **dict(EXAMPLE_NUMERICS, **num))
        r.init()
        for d in r.increments(load):
            if d["increment"] == n:
                break
        out = (np.array(r.scalars().P_av), r.field("P"), r.stats())
        r.close()
        return out

    pm, Pm, st = run(1, 6)
    pf, Pf, _ = run(0, 6)
    assert st.fp32_evaluations > 0
    close(pm, pf, 2e-5, "<P> mixed vs FP64, 6 increments")
    close(Pm, Pf, 1e-4, "P mixed vs FP64, 6 increments")
    tight = dict(itmax=100, eps_rel_div=5e-7, eps_abs_div=1e-12, eps_rel_P=1e-6, eps_abs_P=1e-6)
    pm, _, _ = run(1, 2, **tight)
    pf, _, _ = run(0, 2, **tight)
    close(pm, pf, 1e-6, "<P> mixed vs FP64, tight tolerances")


def test_mixed_precision_tight_tolerances(product, oracle):
    """Precision error apart from the solvers' stopping spread: with the
    divergence and stress tolerances 1000 times tighter (eps_rel_div 5e-7,
    eps_rel_P 1e-6, absolute floors out of the way), both forms converge to
    the equilibrium itself, so what remains between the mixed form and the
    FP64 oracle is the arithmetic.  The FP32 stage stops at its own floor
    (a relative divergence of 1e-5) and the FP64 solve finishes each
    increment.  Required: <P> within 1e-6 relative in every increment and
    every cell's P within 1e-6 of max |P|.  The plain FP64 form is checked
    against the same oracle run: identical counts, and P within 1e-9 (at
    these tolerances N-GMRES works on residuals a thousand times smaller,
    whose least-squares combinations carry rounding further than at the
    default ones)."""
    cfg = CONFIGS["C1"]
    e = cfg["edge"]
    tight = dict(itmin=4, itmax=100, eps_rel_div=5e-7, eps_abs_div=1e-12, eps_rel_P=1e-6, eps_abs_P=1e-6)
    mat, ori, size = polycrystal((e, e, e), cfg["grains"], seed=cfg["seed"], ori_seed=cfg["ori_seed"])
    m = Rve(product, (e, e, e), size, mat, ori, precision=1, **tight)
    p = Rve(product, (e, e, e), size, mat, ori, precision=0, **tight)
    o = Rve(oracle, (e, e, e), size, mat, ori, **tight)
    for r in (m, p, o):
        r.init()
    load = [tension_x(t=cfg["t"], N=cfg["N"])]
    gens = [r.increments(load) for r in (m, p, o)]
    worst = 0.0
    for k in range(6):
        dm, dp, do = (next(g) for g in gens)
        print(f"tight increment {k + 1}: mixed {dm['iterations']}/{dm['evaluations']}, fp64 {dp['iterations']}/"
              f"{dp['evaluations']}, oracle {do['iterations']}/{do['evaluations']}", flush=True)
        assert (dp["iterations"], dp["evaluations"]) == (do["iterations"], do["evaluations"])
        pm, po = np.array(m.scalars().P_av), np.array(o.scalars().P_av)
        err = np.abs(pm - po).max() / np.abs(po).max()
        worst = max(worst, err)
        assert err <= 1e-6, f"increment {k + 1}: <P> {err:.2e}"
        close(p.field("P"), o.field("P"), 1e-9, "P (fp64)")
    print(f"tight: worst <P> error of the mixed form {worst:.2e}", flush=True)
    close(m.field("P"), o.field("P"), 1e-6, "P (mixed)")
    st = m.stats()
    assert st.fp32_evaluations > 0


def test_mixed_precision_reuses_the_last_update(product):
    """The FP64 finish of a mixed increment starts at the F the FP32 stage
    returned; when that was the FP32 stage's last evaluation, its FP64
    material-point update is taken as it is: evaluations outnumber the
    material-point updates, and the FP64 spectral check still runs in every
    increment."""
    cells = (16, 16, 16)
    mat, ori, size = polycrystal(cells, 20, seed=1, ori_seed=2)
    r = Rve(product, cells, size, mat, ori, precision=1, **EXAMPLE_NUMERICS)
    r.init()
    r.reset_stats()
    n_inc = len(list(r.increments([tension_x(t=3.0, N=6)])))
    st = r.stats()
    assert st.residual_evaluations - st.fp32_evaluations >= n_inc
    assert st.material_point_updates < st.residual_evaluations * r.N


C2_FIXTURE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "c2_fixture.npz")


@pytest.mark.skipif(not os.path.exists(C2_FIXTURE), reason="c2 fixture not generated")
def test_loadcase_64cubed_200grains_all_increments():
    """The drop-in configuration through all 40 increments (64^3 grid, 200
    Voronoi grains, tension to 2 %) against the oracle's run of the same
    load case (tests/golden/c2_fixture.npz, made by make_load_fixtures.py):
    identical iterations and evaluations in every increment and <P> within
    1e-10 relative in every increment; at increments 2, 10, 20 and 40, F, P,
    Fp and xi by tail_close on the fixture's cells (a seeded random sample
    and the cells of a cluster where stopping decisions differ)."""
    from solver_cpp_amd.capi import Library
    from conftest import PRODUCT_SO

    fx = np.load(C2_FIXTURE)
    product = Library(PRODUCT_SO)
    cfg = CONFIGS["C2"]
    e = cfg["edge"]
    mat, ori, size = polycrystal((e, e, e), cfg["grains"], seed=cfg["seed"], ori_seed=cfg["ori_seed"])
    a = Rve(product, (e, e, e), size, mat, ori, **EXAMPLE_NUMERICS)
    a.init()
    cells, n_rand = fx["cells"], int(fx["n_random"])
    sampled = set(int(i) for i in fx["sampled"])
    N = e ** 3
    for k, inc in enumerate(a.increments([tension_x(t=cfg["t"], N=cfg["N"])])):
        assert (inc["iterations"], inc["evaluations"]) == (fx["iterations"][k], fx["evaluations"][k]), k + 1
        close(np.array(a.scalars().P_av), fx["P_av"][k], REL, f"<P> increment {k + 1}")
        if inc["increment"] in sampled:
            i = inc["increment"]
            for name in ("F", "P", "Fp", "xi"):
                got = a.field(name).reshape(N, -1)[cells]
                tail_close(got, fx[f"{name}_{i}"], n_rand, f"64^3 increment {i}: {name}")
