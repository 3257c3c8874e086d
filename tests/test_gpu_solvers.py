"""GPU parity of the solvers through the C ABI against the CPU oracle.

Bar (FP64): the GPU solution satisfies the FP64 true residual
||b - M x|| / ||b|| <= tol, agrees with the oracle's solution to 1e-8
relative, and the iteration count is within 2% of the oracle's (which restates
ker_invert_openacc / multishift_invert step for step).  FP32-inner solvers have
no buildable reference (the sp_ sources are generated by a python2 tool absent
here): their bar is the FP64 true residual.
"""
import ctypes as C
import pathlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import openstaple_amd as ost  # noqa: E402
from openstaple_amd import lib  # noqa: E402
from gpu_util import Dev, init_lattice, rel  # noqa: E402
from oracle import Oracle  # noqa: E402

GOLDEN = pathlib.Path(__file__).resolve().parent / "golden"


def iters_close(a, b):
    return abs(a - b) <= max(1, 0.02 * b)


class Sys:
    def __init__(self, shape, seed=1, kind="expH", param=0.3, mass=0.05):
        self.o = Oracle(*shape)
        self.L = init_lattice(shape)
        o = self.o
        self.u = o.gen_expH(param, seed) if kind == "expH" else o.gen_cold(param, seed)
        self.ph = o.phases()
        self.b = o.gen_gauss(seed + 100)
        self.mass = mass
        self.du, self.dph, self.db = Dev(self.u), Dev(self.ph), Dev(self.b)
        self.fp = ost.ferm_param(mass, self.dph.p)
        self.scratch = [Dev(nbytes=self.b.nbytes) for _ in range(4)]

    def cg(self, res, max_cg=10000, shift=0.0, restart=10000):
        x = Dev(nbytes=self.b.nbytes)
        cg = C.c_int(0)
        tr = C.c_double(0)
        r, h, s, p = (d.p for d in self.scratch)
        st = lib.ostp_cg_solve(self.du.p, C.byref(self.fp), x.p, self.db.p, res, r, h, s, p, max_cg, shift, restart,
                               C.byref(cg), C.byref(tr))
        ost.check(0, "ostp_cg_solve")
        return st, cg.value, x.get(self.b), tr.value


@pytest.fixture(scope="module")
def cfg1():
    # configuration 1: 8^4, U = exp(i 0.3 H), seed 1, antiperiodic t, m = 0.05
    return Sys((8, 8, 8, 8), seed=1, kind="expH", param=0.3, mass=0.05)


def test_cg_config1(cfg1):
    s = cfg1
    st, cg, x, tr = s.cg(1e-10)
    ost_, ocg, ox = s.o.cg(s.u, s.ph, s.mass, s.b, 1e-10)
    assert st == 1 and ost_ == 1
    assert tr <= 1e-10
    assert iters_close(cg, ocg), (cg, ocg)
    assert rel(x, ox) < 1e-8
    r = s.b - s.o.mdagm(s.u, x, s.ph, s.mass)
    assert np.linalg.norm(r) / np.linalg.norm(s.b) <= 1e-10


def test_cg_reference_entry_point_with_restarts(cfg1):
    """ker_invert_openacc itself (restart count from inverter_tricks)."""
    s = cfg1
    lib.ostp_set_inverter_tricks(0, 0, 0.1, 40)
    try:
        x = Dev(nbytes=s.b.nbytes)
        cg = C.c_int(0)
        r, h, sc, p = (d.p for d in s.scratch)
        st = lib.ker_invert_openacc(s.du.p, C.byref(s.fp), x.p, s.db.p, 1e-9, r, h, sc, p, 10000, 0.002,
                                    C.byref(cg))
        ost.check(0, "ker_invert_openacc")
        ost_, ocg, ox = s.o.cg(s.u, s.ph, s.mass, s.b, 1e-9, shift=0.002, restart=40)
        assert st == 1 and ost_ == 1
        assert iters_close(cg.value, ocg), (cg.value, ocg)
        assert rel(x.get(s.b), ox) < 1e-7
    finally:
        lib.ostp_set_inverter_tricks(0, 0, 0.1, 10000)


def test_cg_max_cg_failure(cfg1):
    s = cfg1
    st, cg, x, tr = s.cg(1e-12, max_cg=7, restart=7)
    ost_, ocg, ox = s.o.cg(s.u, s.ph, s.mass, s.b, 1e-12, max_cg=7, restart=7)
    assert st == 0 and ost_ == 0 and cg == ocg == 7
    assert rel(x, ox) < 1e-10


def test_mixed_precision_config1(cfg1):
    s = cfg1
    uf = s.o.to_float_gauge(s.u)
    phf = s.ph.astype(np.float32)
    duf, dphf = Dev(uf), Dev(phf)
    fp = ost.ferm_param(s.mass, s.dph.p, dphf.p)
    vb = s.b.nbytes
    d64 = [Dev(nbytes=vb) for _ in range(4)]
    d32 = [Dev(nbytes=vb // 2) for _ in range(5)]
    ip = ost.InverterPackage()
    ip.u, ip.u_f = s.du.p, duf.p
    ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = (d.p for d in d64)
    ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = (d.p for d in d32)
    x = Dev(nbytes=vb)
    cg, ru, tr = C.c_int(0), C.c_int(0), C.c_double(0)
    st = lib.ostp_mixed_solve(ip, C.byref(fp), x.p, s.db.p, 1e-10, 10000, 0.0, 0.1, C.byref(cg), C.byref(ru),
                              C.byref(tr))
    ost.check(0, "ostp_mixed_solve")
    assert st == 1 and tr.value <= 1e-10 and ru.value >= 1
    xs = x.get(s.b)
    r = s.b - s.o.mdagm(s.u, xs, s.ph, s.mass)
    assert np.linalg.norm(r) / np.linalg.norm(s.b) <= 1e-10
    # the oracle's FP32 restatement converges in a comparable number of steps
    ost_, ocg, ox = s.o.mixed(s.u, uf, s.ph, phf, s.mass, s.b, 1e-10)
    assert ost_ == 1 and abs(cg.value - ocg) <= 0.1 * ocg, (cg.value, ocg)
    # the reference entry point
    x2 = Dev(nbytes=vb)
    cg2 = C.c_int(0)
    st2 = lib.inverter_mixed_precision(ip, C.byref(fp), x2.p, s.db.p, 1e-10, 10000, 0.0, C.byref(cg2))
    assert st2 == 1 and cg2.value == cg.value


def remez19(mass, lmax=64.0):
    """Order-19 x^(-1/4) of saved_approxs rescaled exactly from [4e-7, 1] to
    [4e-7*lmax, lmax] (a_k lmax^(3/4), b_k lmax, a0 lmax^(-1/4))."""
    ra = ost.read_remez(str(GOLDEN / "approx_-1_over_4_order_19_mloglm_6.4.REMEZ"))
    power = ra.exponent_num / ra.exponent_den
    eps = lmax ** power
    ra.RA_a0 *= eps
    for k in range(ra.approx_order):
        ra.RA_a[k] *= lmax * eps
        ra.RA_b[k] *= lmax
    ra.lambda_min *= lmax
    ra.lambda_max = lmax
    return ra


def test_multishift_19_shifts_and_recombine(cfg1):
    s = cfg1
    ra = remez19(s.mass)
    order = ra.approx_order
    vb = s.b.nbytes
    out, sf = Dev(nbytes=order * vb), Dev(nbytes=order * vb)
    r, h, sc, p = (d.p for d in s.scratch)
    cg = C.c_int(0)
    before = C.c_int.in_dll(lib, "multishift_invert_iterations").value
    st = lib.multishift_invert(s.du.p, C.byref(s.fp), C.byref(ra), out.p, s.db.p, 1e-10, r, h, sc, p, sf.p, 10000,
                               C.byref(cg))
    ost.check(0, "multishift_invert")
    assert C.c_int.in_dll(lib, "multishift_invert_iterations").value == before + cg.value
    shifts = [ra.RA_b[k] for k in range(order)]
    ost_, ocg, oxs = s.o.multishift(s.u, s.ph, s.mass, shifts, s.b, 1e-10)
    assert st == 1 and ost_ == 1
    assert iters_close(cg.value, ocg), (cg.value, ocg)
    xs = out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))
    for k in range(order):
        assert rel(xs[k], oxs[k]) < 1e-8, k
        rk = s.b - s.o.mdagm(s.u, xs[k], s.ph, s.mass, shifts[k])
        assert np.linalg.norm(rk) / np.linalg.norm(s.b) < 1e-9
    # the per-shift verification after the loop (all shifts' M applications
    # together): its relative residuals against the oracle's operator on the
    # same solutions
    out2, sres, cg2 = Dev(nbytes=order * vb), (C.c_double * 25)(), C.c_int(0)
    st2 = lib.ostp_multishift_solve(s.du.p, C.byref(s.fp), C.byref(ra), out2.p, s.db.p, 1e-10, r, h, sc, p, sf.p,
                                    10000, 0, C.byref(cg2), sres)
    ost.check(0, "ostp_multishift_solve")
    assert st2 == 1 and cg2.value == cg.value
    xs2 = out2.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))
    for k in range(order):
        rk = s.b - s.o.mdagm(s.u, xs2[k], s.ph, s.mass, shifts[k])
        expect = np.linalg.norm(rk) / np.linalg.norm(s.b)
        assert abs(sres[k] - expect) <= 1e-4 * expect + 1e-15, (k, sres[k], expect)
    chi = Dev(nbytes=vb)
    lib.recombine_shifted_vec3_to_vec3(out.p, s.db.p, chi.p, C.byref(ra))
    ost.check(0, "recombine")
    expect = s.o.recombine(xs, s.b, ra.RA_a0, [ra.RA_a[k] for k in range(order)])
    assert rel(chi.get(s.b), expect) < 1e-13


@pytest.mark.parametrize("window", [8, 13, 64])
def test_multishift_window_matches_per_iteration_updates(cfg1, window):
    """The windowed shift updates (residuals kept, x_k and p_k updated once per
    window; 13 leaves partial windows) give the iteration count of the
    per-iteration updates exactly and the same solutions to rounding, in FP64
    and in the FP32 CG-M."""
    s = cfg1
    ra = remez19(s.mass)
    order = ra.approx_order
    vb = s.b.nbytes
    r, h, sc, p = (d.p for d in s.scratch)

    def run(w):
        prev = lib.ostp_set_multishift_window(w)
        try:
            out, sf = Dev(nbytes=order * vb), Dev(nbytes=order * vb)
            cg = C.c_int(0)
            st = lib.multishift_invert(s.du.p, C.byref(s.fp), C.byref(ra), out.p, s.db.p, 1e-10, r, h, sc, p, sf.p,
                                       10000, C.byref(cg))
            ost.check(0, "multishift_invert")
            return st, cg.value, out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))
        finally:
            lib.ostp_set_multishift_window(prev)

    st1, cg1, xs1 = run(1)
    stw, cgw, xsw = run(window)
    assert st1 == 1 and stw == 1
    assert cgw == cg1
    assert cg1 > 2 * window or window == 64, cg1
    for k in range(order):
        assert rel(xsw[k], xs1[k]) < 1e-12, (k, rel(xsw[k], xs1[k]))


def test_multishift_wrappers(cfg1):
    """inverter_multishift_wrapper: DP CG-M, and the SP-accelerated path
    (FP32 CG-M + per-shift DP refinement, inverter_wrappers.c:58-98)."""
    s = cfg1
    ra = remez19(s.mass)
    order = ra.approx_order
    vb = s.b.nbytes
    uf = s.o.to_float_gauge(s.u)
    phf = s.ph.astype(np.float32)
    duf, dphf = Dev(uf), Dev(phf)
    fp = ost.ferm_param(s.mass, s.dph.p, dphf.p)
    d64 = [Dev(nbytes=vb) for _ in range(4)]
    d32 = [Dev(nbytes=vb // 2) for _ in range(5)]
    sf64, sf32 = Dev(nbytes=order * vb), Dev(nbytes=order * vb // 2)
    ip = ost.InverterPackage()
    ip.u, ip.u_f = s.du.p, duf.p
    ip.ferm_shift_temp, ip.ferm_shift_temp_f, ip.nshifts = sf64.p, sf32.p, order
    ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = (d.p for d in d64)
    ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = (d.p for d in d32)
    shifts = [ra.RA_b[k] for k in range(order)]
    for single, mixed in ((0, 0), (1, 0), (1, 1)):
        lib.ostp_set_inverter_tricks(single, mixed, 0.1, 10000)
        out = Dev(nbytes=order * vb)
        it = lib.inverter_multishift_wrapper(ip, C.byref(fp), C.byref(ra), out.p, s.db.p, 1e-10, 10000, 0)
        ost.check(0, "inverter_multishift_wrapper")
        assert it > 0
        xs = out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))
        for k in range(order):
            rk = s.b - s.o.mdagm(s.u, xs[k], s.ph, s.mass, shifts[k])
            assert np.linalg.norm(rk) / np.linalg.norm(s.b) <= 1e-10 * (1.0 if single else 10.0), (single, mixed, k)
    lib.ostp_set_inverter_tricks(0, 0, 0.1, 10000)


@pytest.mark.parametrize("half_inner,graph_its", [(0, 16), (1, 16), (1, 0)])
def test_multishift_mixed_reliable_updates(cfg1, half_inner, graph_its):
    """ostp_multishift_mixed_solve: FP32 CG-M with FP64 reliable updates of the
    base residual, then the shifts still above res refined together by the
    batched solver (FP16 or FP32 inner; its iterations captured 16 per HIP
    graph or, graph_its = 0, launched directly).  The CG-M iteration count stays within
    10% of the FP64 CG-M's (the reliable updates keep the Krylov space).
    Every shift reaches the FP64 true residual with the oracle's operator and
    agrees with the oracle's FP64 CG-M solution (solved to 1e-12) within the
    bound the residual implies."""
    s = cfg1
    ra = remez19(s.mass)
    order = ra.approx_order
    vb = s.b.nbytes
    uf = s.o.to_float_gauge(s.u)
    phf = s.ph.astype(np.float32)
    duf, dphf = Dev(uf), Dev(phf)
    fp = ost.ferm_param(s.mass, s.dph.p, dphf.p)
    d32 = [Dev(nbytes=vb // 2) for _ in range(5)]
    d64 = [Dev(nbytes=vb) for _ in range(4)]
    sf32 = Dev(nbytes=order * vb // 2)
    ip = ost.InverterPackage()
    ip.u, ip.u_f = s.du.p, duf.p
    ip.ferm_shift_temp_f, ip.nshifts = sf32.p, order
    ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = (d.p for d in d32)
    ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = (d.p for d in d64)
    out = Dev(nbytes=order * vb)
    cgm = C.c_int(0)
    cgr, tr = (C.c_int * order)(), (C.c_double * order)()
    prev = lib.ostp_set_batched_graph_iterations(graph_its)
    try:
        conv = lib.ostp_multishift_mixed_solve(ip, C.byref(fp), C.byref(ra), out.p, s.db.p, 1e-10, 10000,
                                               half_inner, C.byref(cgm), cgr, tr)
    finally:
        lib.ostp_set_batched_graph_iterations(prev)
    ost.check(0, "ostp_multishift_mixed_solve")
    shifts = [ra.RA_b[k] for k in range(order)]
    _, ocg, _ = s.o.multishift(s.u, s.ph, s.mass, shifts, s.b, 1e-10)
    _, _, oxs = s.o.multishift(s.u, s.ph, s.mass, shifts, s.b, 1e-12)
    print(f"\nhalf_inner={half_inner}: CG-M {cgm.value} iterations (FP64 CG-M {ocg}), refinement", list(cgr))
    assert conv == order and abs(cgm.value - ocg) <= 0.1 * ocg
    xs = out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))
    for k in range(order):
        rk = s.b - s.o.mdagm(s.u, xs[k], s.ph, s.mass, shifts[k])
        assert np.linalg.norm(rk) / np.linalg.norm(s.b) <= 1e-10, k
        assert tr[k] <= 1e-10
        # ||x - x*|| <= ||A^-1|| ||r||: about cond(A) 1e-10 at worst (cond ~ 6e3 for the smallest shift)
        assert rel(xs[k], oxs[k]) < 1e-6, k


@pytest.mark.parametrize("window", [8, 13])
def test_multishift_mixed_window_matches_per_iteration_updates(cfg1, window):
    """The FP32 CG-M with FP64 reliable updates applies its shift updates once
    per window (windows at fixed iterations, reliable updates inside them): the same CG-M
    iteration count as the per-iteration updates, refinement counts within a
    few iterations of theirs, and every refined shift at the FP64 true
    residual with the oracle's operator."""
    s = cfg1
    ra = remez19(s.mass)
    order = ra.approx_order
    vb = s.b.nbytes
    uf = s.o.to_float_gauge(s.u)
    phf = s.ph.astype(np.float32)
    duf, dphf = Dev(uf), Dev(phf)
    fp = ost.ferm_param(s.mass, s.dph.p, dphf.p)
    d32 = [Dev(nbytes=vb // 2) for _ in range(5)]
    d64 = [Dev(nbytes=vb) for _ in range(4)]
    sf32 = Dev(nbytes=order * vb // 2)
    ip = ost.InverterPackage()
    ip.u, ip.u_f = s.du.p, duf.p
    ip.ferm_shift_temp_f, ip.nshifts = sf32.p, order
    ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = (d.p for d in d32)
    ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = (d.p for d in d64)
    got = []
    for w in (1, window):
        prev = lib.ostp_set_multishift_window(w)
        try:
            out = Dev(nbytes=order * vb)
            cgm = C.c_int(0)
            cgr, tr = (C.c_int * order)(), (C.c_double * order)()
            conv = lib.ostp_multishift_mixed_solve(ip, C.byref(fp), C.byref(ra), out.p, s.db.p, 1e-10, 10000, 0,
                                                   C.byref(cgm), cgr, tr)
            ost.check(0, "ostp_multishift_mixed_solve")
            got.append((conv, cgm.value, list(cgr), [tr[k] for k in range(order)],
                        out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))))
        finally:
            lib.ostp_set_multishift_window(prev)
    (c1, n1, r1, t1, x1), (cw, nw, rw, tw, xw) = got
    assert c1 == cw == order and n1 == nw and n1 > 2 * window
    # the windowed FP32 accumulators round differently: refinement counts within a few iterations
    assert all(abs(a - b) <= max(3, 0.2 * a) for a, b in zip(r1, rw)), (r1, rw)
    shifts = [ra.RA_b[k] for k in range(order)]
    for k in range(order):
        assert tw[k] <= 1e-10
        rk = s.b - s.o.mdagm(s.u, xw[k], s.ph, s.mass, shifts[k])
        assert np.linalg.norm(rk) / np.linalg.norm(s.b) <= 1e-10, k
        assert rel(xw[k], x1[k]) < 1e-6, k


def test_power_method_vs_oracle(cfg1):
    """ker_find_max_eigenvalue_openacc / find_min_max_eigenvalue_soloopenacc /
    ker_find_min_eigenvalue_openacc on the GPU against the oracle restatement
    (pinned by the dense eigen-decomposition) from the same start vector: the
    same iteration count (the norm's reduction order may move the 1e-5 stop by
    one iteration) and the same eigenvalue estimate."""
    s = cfg1
    start = s.o.gen_gauss(7)
    v_o, it_o = s.o.find_max_eigenvalue(s.u, s.ph, s.mass, start)
    r, h, pp = Dev(nbytes=start.nbytes), Dev(nbytes=start.nbytes), Dev(start)
    it = C.c_int(0)
    v = lib.ostp_find_max_eigenvalue(s.du.p, C.byref(s.fp), r.p, h.p, pp.p, C.byref(it))
    ost.check(0, "ostp_find_max_eigenvalue")
    assert abs(it.value - it_o) <= 1, (it.value, it_o)
    if it.value == it_o:
        assert abs(v - v_o) <= 1e-12 * v_o, (v, v_o)
    else:
        assert abs(v - v_o) <= 1e-5 * v_o, (v, v_o)
    pp2, pp3 = Dev(start), Dev(start)
    mm = (C.c_double * 2)()
    lib.find_min_max_eigenvalue_soloopenacc(s.du.p, C.byref(s.fp), r.p, h.p, pp2.p, pp3.p, mm)
    ost.check(0, "find_min_max_eigenvalue_soloopenacc")
    assert mm[0] == s.mass * s.mass and mm[1] == v
    vmin_o, itm_o = s.o.find_min_eigenvalue(s.u, s.ph, s.mass, start, v_o)
    itm = C.c_int(0)
    vmin = lib.ostp_find_min_eigenvalue(s.du.p, C.byref(s.fp), r.p, h.p, pp3.p, v_o, C.byref(itm))
    assert abs(itm.value - itm_o) <= 1 and abs(vmin - vmin_o) <= 1e-5 * abs(vmin_o), (vmin, vmin_o)


def test_multishift_fp32():
    s = Sys((8, 8, 8, 8), seed=5, kind="cold", param=0.5, mass=0.1)
    ra = remez19(s.mass)
    order = ra.approx_order
    uf = s.o.to_float_gauge(s.u)
    phf = s.ph.astype(np.float32)
    bf = s.b.astype(np.complex64)
    duf, dphf, dbf = Dev(uf), Dev(phf), Dev(bf)
    fp = ost.ferm_param(s.mass, s.dph.p, dphf.p)
    vbf = bf.nbytes
    out, sf = Dev(nbytes=order * vbf), Dev(nbytes=order * vbf)
    sc = [Dev(nbytes=vbf) for _ in range(4)]
    cg = C.c_int(0)
    res = (C.c_double * 25)()
    st = lib.ostp_multishift_solve(duf.p, C.byref(fp), C.byref(ra), out.p, dbf.p, 1e-5, *(d.p for d in sc), sf.p,
                                   10000, 1, C.byref(cg), res)
    ost.check(0, "ostp_multishift_solve(single)")
    assert st == 1
    xs = out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex64)).astype(np.complex128)
    for k in range(order):
        rk = s.b - s.o.mdagm(s.u, xs[k], s.ph, s.mass, ra.RA_b[k])
        assert np.linalg.norm(rk) / np.linalg.norm(s.b) < 2e-5


def test_multishift_window_cut_by_max_cg(cfg1):
    """A solve stopped by max_cg in the middle of a window (19 iterations,
    W = 8): the partial window is applied once, and the unconverged solutions,
    the shifted directions and the status are those of the per-iteration
    updates."""
    s = cfg1
    ra = remez19(s.mass)
    order = ra.approx_order
    vb = s.b.nbytes
    r, h, sc, p = (d.p for d in s.scratch)
    got = []
    for w in (1, 8):
        prev = lib.ostp_set_multishift_window(w)
        try:
            out, sf = Dev(nbytes=order * vb), Dev(nbytes=order * vb)
            cg = C.c_int(0)
            st = lib.multishift_invert(s.du.p, C.byref(s.fp), C.byref(ra), out.p, s.db.p, 1e-10, r, h, sc, p, sf.p,
                                       19, C.byref(cg))
            ost.check(0, "multishift_invert")
            got.append((st, cg.value, out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128)),
                        sf.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex128))))
        finally:
            lib.ostp_set_multishift_window(prev)
    # the status is the reference's per-shift check |b - M x_k| <= |b|, the same on both paths
    assert got[0][1] == got[1][1] == 19 and got[0][0] == got[1][0]
    for k in range(order):
        assert rel(got[1][2][k], got[0][2][k]) < 1e-12, k
        assert rel(got[1][3][k], got[0][3][k]) < 1e-12, k


def test_multishift_fp32_window_matches_per_iteration_updates():
    s = Sys((8, 8, 8, 8), seed=5, kind="cold", param=0.5, mass=0.1)
    ra = remez19(s.mass)
    order = ra.approx_order
    duf, dphf, dbf = Dev(s.o.to_float_gauge(s.u)), Dev(s.ph.astype(np.float32)), Dev(s.b.astype(np.complex64))
    fp = ost.ferm_param(s.mass, s.dph.p, dphf.p)
    vbf = s.b.nbytes // 2
    sc = [Dev(nbytes=vbf) for _ in range(4)]
    got = []
    for w in (1, 8):
        prev = lib.ostp_set_multishift_window(w)
        try:
            out, sf = Dev(nbytes=order * vbf), Dev(nbytes=order * vbf)
            cg = C.c_int(0)
            st = lib.ostp_multishift_solve(duf.p, C.byref(fp), C.byref(ra), out.p, dbf.p, 1e-5, *(d.p for d in sc),
                                           sf.p, 10000, 1, C.byref(cg), None)
            ost.check(0, "ostp_multishift_solve(single)")
            assert st == 1
            got.append((cg.value, out.get(np.zeros((order, 3, s.o.sizeh), dtype=np.complex64)).astype(np.complex128)))
        finally:
            lib.ostp_set_multishift_window(prev)
    assert got[0][0] == got[1][0] and got[0][0] > 8
    for k in range(order):
        assert rel(got[1][1][k], got[0][1][k]) < 1e-5, k


def test_zero_source_matches_reference_semantics():
    """b = 0: ker_invert_openacc's omega = 0/0 poisons x; the final true
    residual is NaN so the call reports failure after one iteration."""
    s = Sys((4, 4, 4, 4), seed=9, kind="cold", param=0.5, mass=0.1)
    s.db.put(np.zeros_like(s.b))
    st, cg, x, tr = s.cg(1e-10)
    zero = np.zeros_like(s.b)
    ost_, ocg, ox = s.o.cg(s.u, s.ph, s.mass, zero, 1e-10)
    assert st == ost_ == 0 and cg == ocg == 1


def test_cg_full_size_16_true_residual():
    s = Sys((16, 16, 16, 16), seed=3, kind="cold", param=0.5, mass=0.02)
    st, cg, x, tr = s.cg(1e-10)
    assert st == 1 and tr <= 1e-10
    r = s.b - s.o.mdagm(s.u, x, s.ph, s.mass)
    assert np.linalg.norm(r) / np.linalg.norm(s.b) <= 1e-10


def test_config2_full_shape():
    """Configuration 2 at its full size: 32^4, generate_Conf_cold eps = 0.5
    (seed 1) smeared by 2 stout steps (rho = 0.15), the order-19 x^(-1/4)
    approximation rescaled to [m^2, 64] with m = 0.01, a Gaussian source, 1e-10
    per shift.  FP64 CG-M, the FP32 CG-M with FP64 reliable updates and
    batched refinement (FP16 and FP32 inner) and the reference's
    SP-accelerated wrapper: every shift's FP64 true residual <= 1e-10 (the
    library's FP64 operator, pinned against the oracle at smaller sizes); the
    reduced-precision CG-M takes the FP64 CG-M's iteration count (within 2%); every shift
    agrees with the FP64 CG-M's solution within 1e-6 (cond ~ 1e4 for the
    smallest shift times the 1e-10 residuals)."""
    shape, mass = (32, 32, 32, 32), 0.01
    L = init_lattice(shape)
    sizeh, vb, gb = L.sizeh, L.vec3_bytes, 8 * L.su3_bytes
    lib.ostp_set_stout(0.15, 2, 0.0, 0, 0, 1)
    lib.ostp_set_inverter_tricks(0, 0, 0.1, 10000)
    raw = Dev(nbytes=gb)
    lib.ostp_generate_Conf_cold(raw.p, 0.5, 1)
    levels = Dev(nbytes=lib.ostp_stout_steps() * gb)
    lib.stout_wrapper(raw.p, levels.p, 0)
    u = levels.p + (lib.ostp_stout_steps() - 1) * gb
    ph, phf, uf = Dev(nbytes=64 * sizeh), Dev(nbytes=32 * sizeh), Dev(nbytes=8 * L.su3f_bytes)
    lib.calc_u1_phases(ph.p, ost.BfParam(0, 0, 0, 0, 0, 0), 0.0, 0.0)
    lib.ostp_phases_to_float(ph.p, phf.p)
    lib.ostp_convert_double_to_float_gauge(u, uf.p)
    b = Dev(nbytes=vb)
    lib.ostp_generate_vec3_soa_gauss(b.p, 1, 0)
    ost.check(0, "setup")
    ra = remez19(mass)
    order = ra.approx_order
    fp = ost.ferm_param(mass, ph.p, phf.p)
    d64 = [Dev(nbytes=vb) for _ in range(4)]
    d32 = [Dev(nbytes=vb // 2) for _ in range(5)]
    sf, sf32 = Dev(nbytes=order * vb), Dev(nbytes=order * vb // 2)
    ip = ost.InverterPackage()
    ip.u, ip.u_f = u, uf.p
    ip.ferm_shift_temp, ip.ferm_shift_temp_f, ip.nshifts = sf.p, sf32.p, order
    ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = (d.p for d in d64)
    ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = (d.p for d in d32)
    tmp_s, tmp_h, diff = Dev(nbytes=vb), Dev(nbytes=vb), Dev(nbytes=vb)
    bn = lib.l2norm2_global(b.p)

    def worst_true_residual(out):
        w = 0.0
        for k in range(order):
            lib.fermion_matrix_multiplication_shifted(u, tmp_s.p, out.p + k * vb, tmp_h.p, C.byref(fp), ra.RA_b[k])
            lib.combine_in1_minus_in2(b.p, tmp_s.p, tmp_h.p)
            w = max(w, (lib.l2norm2_global(tmp_h.p) / bn) ** 0.5)
        return w

    def worst_rel_err(out, ref):
        w = 0.0
        for k in range(order):
            lib.combine_in1_minus_in2(out.p + k * vb, ref.p + k * vb, diff.p)
            w = max(w, (lib.l2norm2_global(diff.p) / lib.l2norm2_global(ref.p + k * vb)) ** 0.5)
        return w

    x64 = Dev(nbytes=order * vb)
    cg = C.c_int(0)
    sres = (C.c_double * 25)()
    st = lib.ostp_multishift_solve(u, C.byref(fp), C.byref(ra), x64.p, b.p, 1e-10, *(d.p for d in d64), sf.p, 20000,
                                   0, C.byref(cg), sres)
    ost.check(0, "ostp_multishift_solve")
    assert st == 1 and worst_true_residual(x64) <= 1e-10
    for half_inner in (1, 0):
        out = Dev(nbytes=order * vb)
        cgm = C.c_int(0)
        cgr, tr = (C.c_int * order)(), (C.c_double * order)()
        conv = lib.ostp_multishift_mixed_solve(ip, C.byref(fp), C.byref(ra), out.p, b.p, 1e-10, 20000, half_inner,
                                               C.byref(cgm), cgr, tr)
        ost.check(0, "ostp_multishift_mixed_solve")
        print(f"\n32^4: FP64 CG-M {cg.value} iterations; reduced precision (half_inner={half_inner}) {cgm.value}, "
              f"refinement {list(cgr)}")
        assert conv == order and iters_close(cgm.value, cg.value)
        assert max(tr[k] for k in range(order)) <= 1e-10 and worst_true_residual(out) <= 1e-10
        assert worst_rel_err(out, x64) < 1e-6
    out = Dev(nbytes=order * vb)
    lib.ostp_set_inverter_tricks(1, 1, 0.1, 10000)
    lib.inverter_multishift_wrapper(ip, C.byref(fp), C.byref(ra), out.p, b.p, 1e-10, 20000, 0)
    lib.ostp_set_inverter_tricks(0, 0, 0.1, 10000)
    ost.check(0, "inverter_multishift_wrapper")
    assert worst_true_residual(out) <= 1e-10 and worst_rel_err(out, x64) < 1e-6


# 8 and 480 half-sites (less than a block, a last block that is not full), the
# last lattice whose hops are split over waves (49152 half-sites) and one above it
@pytest.mark.parametrize("shape", [(2, 2, 2, 2), (6, 4, 4, 10), (16, 16, 16, 24), (16, 16, 16, 26)])
def test_solver_iterations_at_block_edges(shape):
    """CG (with restarts) and CG-M (three shifts, windows and per-iteration
    updates) against the oracle: the solutions differ by at most both
    residuals times the condition number (bounded by 1 + 4 * 16 / m^2)."""
    mass = 0.4
    s = Sys(shape, seed=9, kind="cold", param=0.4, mass=mass)
    cond = 1 + 64 / mass ** 2
    st, cg, x, tr = s.cg(1e-10, restart=12)
    ost_, ocg, ox = s.o.cg(s.u, s.ph, mass, s.b, 1e-10, restart=12)
    assert st == 1 and ost_ == 1 and tr <= 1e-10 and iters_close(cg, ocg), (st, ost_, cg, ocg)
    assert rel(x, ox) < 2e-10 * cond
    ra = remez19(mass)
    ra.approx_order = 3
    vb = s.b.nbytes
    b = np.array([ra.RA_b[k] for k in range(3)])
    _, mcg, mx = s.o.multishift(s.u, s.ph, mass, b, s.b, 1e-10)[:3]
    for w in (1, 8):
        prev = lib.ostp_set_multishift_window(w)
        try:
            out, sf = Dev(nbytes=3 * vb), Dev(nbytes=3 * vb)
            cg = C.c_int(0)
            st = lib.multishift_invert(s.du.p, C.byref(s.fp), C.byref(ra), out.p, s.db.p, 1e-10,
                                       *(d.p for d in s.scratch), sf.p, 10000, C.byref(cg))
            ost.check(0, "multishift_invert")
        finally:
            lib.ostp_set_multishift_window(prev)
        assert st == 1 and iters_close(cg.value, mcg), (w, cg.value, mcg)
        got = out.get(np.zeros((3, 3, s.o.sizeh), dtype=np.complex128))
        for k in range(3):
            assert rel(got[k], mx[k]) < 2e-10 * cond, (w, k)


# delta 0.9: nearly every second iteration is a reliable update, also right
# after one another and in the last iteration of a batch
@pytest.mark.parametrize("shape", [(2, 2, 2, 2), (6, 4, 4, 10), (16, 16, 16, 8)])
@pytest.mark.parametrize("delta", [0.1, 0.9])
def test_mixed_iterations_at_block_edges(shape, delta):
    """The FP32 iterations with FP64 reliable updates against the oracle's:
    the true residual (FP64, the oracle's operator), the iterations (FP32
    rounding moves their number by a tenth at most, one on a small count), and
    a solve cut short by max_cg."""
    mass = 0.2
    s = Sys(shape, seed=4, kind="cold", param=0.4, mass=mass)
    uf, phf = s.o.to_float_gauge(s.u), s.ph.astype(np.float32)
    duf, dphf = Dev(uf), Dev(phf)
    fp = ost.ferm_param(mass, s.dph.p, dphf.p)
    vb = s.b.nbytes
    d32 = [Dev(nbytes=vb // 2) for _ in range(5)]
    ip = ost.InverterPackage()
    ip.u, ip.u_f = s.du.p, duf.p
    ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = (d.p for d in s.scratch)
    ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = (d.p for d in d32)
    x = Dev(nbytes=vb)
    cg, ru, tr = C.c_int(0), C.c_int(0), C.c_double(0)
    args = (C.byref(cg), C.byref(ru), C.byref(tr))
    x.put(np.zeros_like(s.b))
    st = lib.ostp_mixed_solve(ip, C.byref(fp), x.p, s.db.p, 1e-10, 10000, 0.0, delta, *args)
    ost.check(0, "ostp_mixed_solve")
    r = s.b - s.o.mdagm(s.u, x.get(s.b), s.ph, mass)
    assert st == 1 and ru.value >= 1 and np.linalg.norm(r) / np.linalg.norm(s.b) <= 1e-10
    ost_, ocg, _ = s.o.mixed(s.u, uf, s.ph, phf, mass, s.b, 1e-10, delta=delta)
    assert ost_ == 1 and abs(cg.value - ocg) <= max(1, 0.1 * ocg), (cg.value, ocg)
    x.put(np.zeros_like(s.b))
    st = lib.ostp_mixed_solve(ip, C.byref(fp), x.p, s.db.p, 1e-10, 5, 0.0, delta, *args)
    ost.check(0, "ostp_mixed_solve")
    assert st == 0 and cg.value == 5
    r = s.b - s.o.mdagm(s.u, x.get(s.b), s.ph, mass)
    # the FP64 residual of what the five FP32 steps added
    assert abs(np.linalg.norm(r) / np.linalg.norm(s.b) - tr.value) <= 1e-6 * tr.value


# ten and twenty shifts are the most that one pass of a window's update takes
@pytest.mark.parametrize("order", [1, 10, 11, 20, 21, 24])
@pytest.mark.parametrize("window", [9, 64])
def test_multishift_window_orders(order, window):
    """Solutions and directions from windowed updates against those of the
    per-iteration updates (the same recurrence, summed in another order)."""
    s = Sys((4, 6, 4, 6), seed=3, kind="cold", param=0.5, mass=0.1)
    ra = remez19(s.mass)
    ra.approx_order = order
    for k in range(order):
        ra.RA_b[k] = 0.003 * 1.4 ** k
    vb = s.b.nbytes
    got = []
    for w in (1, window):
        prev = lib.ostp_set_multishift_window(w)
        try:
            # what the outputs held before is not read
            out, sf = Dev(np.full(order * 3 * s.o.sizeh, np.nan + 0j)), Dev(np.full(order * 3 * s.o.sizeh, np.nan + 0j))
            cg = C.c_int(0)
            st = lib.multishift_invert(s.du.p, C.byref(s.fp), C.byref(ra), out.p, s.db.p, 1e-9,
                                       *(d.p for d in s.scratch), sf.p, 10000, C.byref(cg))
            ost.check(0, "multishift_invert")
        finally:
            lib.ostp_set_multishift_window(prev)
        shape = np.zeros((order, 3, s.o.sizeh), dtype=np.complex128)
        got.append((st, cg.value, out.get(shape), sf.get(shape)))
    assert got[0][0] == got[1][0] == 1 and got[0][1] == got[1][1]
    for k in range(order):
        assert rel(got[1][2][k], got[0][2][k]) < 1e-12, k
        # the directions' terms cancel, by 1e3 to 1e4 at most over these iterations, times 64 roundings
        assert rel(got[1][3][k], got[0][3][k]) < 1e-10, k


# above 49152 half-sites the solver's hops take phases that are +-1 as signs;
# 1e-5 off is not +-1
@pytest.mark.parametrize("phases", [dict(), dict(mu=1e-5), dict(bf=(0, 0, 1, 0, 0, 0), charge=1.0)])
def test_solver_phases_of_large_lattices(phases):
    """CG-M with one shift against the oracle: both residuals times the
    condition number, far below what phases off by 1e-5 change."""
    mass = 0.4
    s = Sys((16, 16, 16, 26), seed=9, kind="cold", param=0.4, mass=mass)
    ph = s.o.phases(**phases)
    dph = Dev(ph)
    fp = ost.ferm_param(mass, dph.p)
    ra = remez19(mass)
    ra.approx_order = 1
    vb = s.b.nbytes
    out, sf = Dev(nbytes=vb), Dev(nbytes=vb)
    cg = C.c_int(0)
    st = lib.multishift_invert(s.du.p, C.byref(fp), C.byref(ra), out.p, s.db.p, 1e-10, *(d.p for d in s.scratch),
                               sf.p, 10000, C.byref(cg))
    ost.check(0, "multishift_invert")
    _, ocg, ox = s.o.multishift(s.u, ph, mass, [ra.RA_b[0]], s.b, 1e-10)
    assert st == 1 and iters_close(cg.value, ocg), (cg.value, ocg)
    assert rel(out.get(s.b), ox[0]) < 2e-10 * (1 + 64 / mass ** 2)
