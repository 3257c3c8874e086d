"""The 2+1-flavour RHMC of the 48^3x12 workload on the GPU.

Workload: tree-level Symanzik gauge action at beta = 3.8, 2 stout steps with
rho = 0.15, staggered light quarks (m_l = 0.0015, two flavours: the action
<phi, (M^+M)^(-1/2) phi>, heat bath with (M^+M)^(1/4)) and a strange quark
(m_s = 0.04: (M^+M)^(-1/4), heat bath (M^+M)^(1/8)), order-19 rational
approximations from the committed .REMEZ files (the x^(-1/2) one generated by
the repository's Remez), 2nd-order Omelyan integrator.

Bar:
  * 4^3x8: a forward MD trajectory followed by the trajectory with the momenta
    flipped returns links and momenta to 1e-9 (relative); the energy
    violation H(end) - H(start), with the fermion action evaluated by the
    library's multishift solver and recombination, falls as the square of the
    step (ratio 4 within 20%);
  * 4^3x8: the full update (heat bath, power-method bounds, rescaled
    approximations, MD, acceptance) has dS falling as the step squared (ratio
    4 within 25%);
  * 48^3x12 (the full lattice, 10 Omelyan steps x 5 gauge sub-steps, tau = 1):
    forward then back restores links and momenta to 1e-9.
"""
import ctypes as C
import pathlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import openstaple_amd as ost  # noqa: E402
from openstaple_amd import lib  # noqa: E402
from gpu_util import Dev, init_lattice, rel  # noqa: E402

GOLDEN = pathlib.Path(__file__).resolve().parent / "golden"
C0_TLSM, C1_TLSM = 5.0 * 0.33333333333333333333333, -0.25 * 0.33333333333333333333333
BETA = 3.8
# (mass, degeneracy, heat-bath mother, MD / acceptance mother)
FLAVOURS = [(0.0015, 2, "approx_1_over_4_order_19_mloglm_7.0.REMEZ", "approx_-1_over_2_order_19_mloglm_7.0.REMEZ"),
            (0.04, 1, "approx_1_over_8_order_19_mloglm_6.4.REMEZ", "approx_-1_over_4_order_19_mloglm_6.4.REMEZ")]


def rescaled(name, lmax):
    """A mother approximation on [lambda_min, 1] rescaled to [lmax lambda_min, lmax]."""
    ra = ost.read_remez(str(GOLDEN / name))
    e = ra.exponent_num / ra.exponent_den
    ra.RA_a0 *= lmax ** e
    for k in range(ra.approx_order):
        ra.RA_a[k] *= lmax ** (1 + e)
        ra.RA_b[k] *= lmax
    ra.lambda_min *= lmax
    ra.lambda_max *= lmax
    return ra


def set_md(no_md, gauge_scale, t):
    ost.ActionParam.in_dll(lib, "act_params").beta = BETA
    p = ost.MdParam(no_md=no_md, gauge_scale=gauge_scale, t=t)
    mp = ost.MdParam.in_dll(lib, "md_parameters")
    C.memmove(C.addressof(mp), C.addressof(p), C.sizeof(p))
    lib.initialize_md_global_variables(p)


class Nf21:
    """Fields and buffers of multistep_2MN_SOLOOPENACC for the two flavours,
    one pseudofermion each, on a generate_Conf_cold field."""

    def __init__(self, shape, eps=0.3, seed=3, lmax=20.0, res=1e-10):
        self.lat = lat = init_lattice(shape)
        lib.ostp_set_stout(0.15, 2, 0.0, 0, 0, 1)
        lib.ostp_set_inverter_tricks(0, 0, 0.1, 10000)
        self.res = res
        sizeh, vb = lat.sizeh, lat.vec3_bytes
        self.gb = 8 * lat.su3_bytes
        self.tb = 8 * 64 * sizeh
        self.u = Dev(nbytes=self.gb)
        lib.ostp_generate_Conf_cold(self.u.p, eps, seed)
        self.u0 = self.u.get(np.zeros(self.gb, np.uint8))
        self.ph = Dev(nbytes=8 * 8 * sizeh)
        lib.calc_u1_phases(self.ph.p, ost.BfParam(0, 0, 0, 0, 0, 0), 0.0, 0.0)
        self.chi = Dev(nbytes=2 * vb)
        for f in range(2):
            lib.ostp_generate_vec3_soa_gauss(self.chi.p + f * vb, 77, 10 + f)
        self.arr, self.gl3, self.taux = Dev(nbytes=2 * self.gb), Dev(nbytes=self.gb), Dev(nbytes=self.gb)
        self.ipd = Dev(nbytes=self.tb)
        self.xs, self.sf = Dev(nbytes=19 * vb), Dev(nbytes=19 * vb)
        self.d64 = [Dev(nbytes=vb) for _ in range(4)]
        self.out = Dev(nbytes=vb)
        self.fps = (ost.FermParam * 2)()
        for f, (mass, deg, _, md) in enumerate(FLAVOURS):
            fp = self.fps[f]
            fp.ferm_mass, fp.degeneracy, fp.number_of_ps, fp.index_of_the_first_ps = mass, deg, 1, f
            fp.phases = self.ph.p
            fp.approx_md = rescaled(md, lmax)
            fp.approx_li = rescaled(md, lmax)
        ost.check(0, "setup")

    def ip(self, conf_p):
        ipk = ost.InverterPackage()
        ipk.u = conf_p
        ipk.ferm_shift_temp, ipk.nshifts = self.sf.p, 19
        ipk.loc_r, ipk.loc_h, ipk.loc_s, ipk.loc_p = (d.p for d in self.d64)
        return ipk

    def trajectory(self, du, dm):
        lib.multistep_2MN_SOLOOPENACC(self.ipd.p, du.p, self.arr.p, self.gl3.p, self.taux.p, self.fps, 2,
                                      self.chi.p, self.xs.p, self.ip(du.p), dm.p, None, self.res, 50000)
        ost.check(0, "multistep_2MN_SOLOOPENACC")

    def fermion_action(self, du):
        lib.stout_wrapper(du.p, self.arr.p, 0)
        v = self.arr.p + self.gb
        tot = 0.0
        vb = self.lat.vec3_bytes
        for f in range(2):
            ra = self.fps[f].approx_li
            chi_f = self.chi.p + f * vb
            lib.inverter_multishift_wrapper(self.ip(v), C.byref(self.fps, f * C.sizeof(ost.FermParam)),
                                            C.byref(ra), self.xs.p, chi_f, 1e-12, 50000, 1)
            lib.recombine_shifted_vec3_to_vec3(self.xs.p, chi_f, self.out.p, C.byref(ra))
            tot += lib.real_scal_prod_global(chi_f, self.out.p)
        ost.check(0, "fermion action")
        return tot

    def hamiltonian(self, du, dm):
        s = C0_TLSM * lib.calc_plaquette_soloopenacc(du.p, None, None) + \
            C1_TLSM * lib.calc_rettangolo_soloopenacc(du.p, None, None)
        kin = sum(lib.calc_momenta_action(dm.p, None, mu) for mu in range(8))
        return kin - BETA / 3.0 * s + self.fermion_action(du)

    def momenta(self, seed):
        dm = Dev(nbytes=self.tb)
        lib.ostp_generate_Momenta_gauss(dm.p, seed, 0)
        return dm


def forward_back(F, no_md, gauge_scale, t, seed):
    set_md(no_md, gauge_scale, t)
    du = Dev(F.u0)
    dm = F.momenta(seed)
    m0 = dm.get(np.zeros(F.tb // 8))
    F.trajectory(du, dm)
    moved = rel(du.get(F.u0).view(np.float64), F.u0.view(np.float64))
    lib.invert_momenta(dm.p)
    F.trajectory(du, dm)
    back_u = rel(du.get(F.u0).view(np.float64), F.u0.view(np.float64))
    back_m = rel(dm.get(m0), -m0)
    return moved, back_u, back_m


def test_nf21_md_reversible_and_second_order():
    F = Nf21((4, 4, 4, 8))
    moved, back_u, back_m = forward_back(F, 3, 3, 0.5, 5)
    assert moved > 1e-3 and back_u < 1e-9 and back_m < 1e-9, (moved, back_u, back_m)
    dh = []
    for no_md in (3, 6):
        set_md(no_md, 3, 0.5)
        du, dm = Dev(F.u0), F.momenta(6)
        h0 = F.hamiltonian(du, dm)
        F.trajectory(du, dm)
        dh.append(F.hamiltonian(du, dm) - h0)
    ratio = dh[0] / dh[1]
    assert abs(ratio - 4.0) < 0.8, (dh, ratio)


@pytest.mark.parametrize("shape", [(4, 4, 4, 8), (8, 8, 8, 8)])  # the second with t-fastest tiles
def test_force_sources_solved_together_match_one_by_one(shape):
    """fermion_force_soloopenacc with the two flavours' rational solves run
    together (one CG-M iteration stream, shared-link hops) gives the force of
    the one-by-one solves bit for bit: phases as one array and as two arrays
    of equal values; with different phases (imaginary mu in one flavour) the
    solves run one by one and the force matches as well."""
    F = Nf21(shape)
    lat = F.lat
    du = Dev(F.u0)

    def force(batch):
        prev = lib.ostp_set_multishift_batching(batch)
        try:
            ipd = Dev(nbytes=F.tb)
            lib.fermion_force_soloopenacc(du.p, F.arr.p, F.gl3.p, ipd.p, F.fps, 2, F.chi.p, F.res, F.taux.p, F.xs.p,
                                          F.ip(du.p), 50000)
            ost.check(0, "fermion_force_soloopenacc")
            return ipd.get(np.zeros(F.tb // 8))
        finally:
            lib.ostp_set_multishift_batching(prev)

    before = C.c_int.in_dll(lib, "multishift_invert_iterations").value
    f1 = force(1)
    its1 = C.c_int.in_dll(lib, "multishift_invert_iterations").value - before
    f0 = force(0)
    its0 = C.c_int.in_dll(lib, "multishift_invert_iterations").value - before - its1
    assert np.abs(f0).max() > 1e-3
    assert np.array_equal(f1, f0) and its1 == its0, (rel(f1, f0), its1, its0)
    # equal values in two arrays
    ph2 = Dev(nbytes=8 * 8 * lat.sizeh)
    lib.calc_u1_phases(ph2.p, ost.BfParam(0, 0, 0, 0, 0, 0), 0.0, 0.0)
    F.fps[1].phases = ph2.p
    assert np.array_equal(force(1), f0)
    # different phases: one by one, same force as the unbatched call
    lib.calc_u1_phases(ph2.p, ost.BfParam(0, 0, 0, 0, 0, 0), 0.1, 1.0)
    g1, g0 = force(1), force(0)
    assert np.array_equal(g1, g0) and not np.array_equal(g1, f0)
    F.fps[1].phases = F.ph.p
    # a heavy second flavour stops many iterations before the first
    m_s = F.fps[1].ferm_mass
    F.fps[1].ferm_mass = 0.5
    try:
        b0 = C.c_int.in_dll(lib, "multishift_invert_iterations").value
        h1 = force(1)
        n1 = C.c_int.in_dll(lib, "multishift_invert_iterations").value - b0
        h0 = force(0)
        n0 = C.c_int.in_dll(lib, "multishift_invert_iterations").value - b0 - n1
        assert np.array_equal(h1, h0) and n1 == n0
    finally:
        F.fps[1].ferm_mass = m_s


def test_force_with_an_earlier_error_left_recorded():
    """An error that an earlier call left recorded (non-aborting mode, not
    yet read by the host) does not stop fermion_force_soloopenacc: with the
    flavours' solves together, the force equals the one computed with no
    error pending, and the earlier message is still there afterwards."""
    F = Nf21((4, 4, 4, 8))
    du = Dev(F.u0)

    def force():
        ipd = Dev(nbytes=F.tb)
        lib.fermion_force_soloopenacc(du.p, F.arr.p, F.gl3.p, ipd.p, F.fps, 2, F.chi.p, F.res, F.taux.p, F.xs.p,
                                      F.ip(du.p), 50000)
        return ipd

    clean = force()
    ost.check(0, "fermion_force_soloopenacc")
    clean = clean.get(np.zeros(F.tb // 8))
    assert np.abs(clean).max() > 1e-3
    assert lib.ostp_set_multishift_precision(7, 0) == -1  # a bad mode: an error recorded, nothing changed
    msg = lib.ostp_last_error()
    assert msg
    try:
        pending = force()
        assert lib.ostp_last_error() == msg
    finally:
        lib.ostp_clear_error()
    assert np.array_equal(pending.get(np.zeros(F.tb // 8)), clean)


def set_ptr(name, value):
    C.c_void_p.in_dll(lib, name).value = value


GLOBALS = ("conf_acc_bkp", "aux_conf_acc", "auxbis_conf_acc", "gstout_conf_acc_arr", "momenta", "ipdot_acc",
           "ferm_phi_acc", "ferm_chi_acc", "ferm_shiftmulti_acc", "k_p_shiftferm", "kloc_r", "kloc_h", "kloc_s",
           "kloc_p", "fermions_parameters")


def test_nf21_rhmc_update_second_order():
    shape = (4, 4, 4, 8)
    lat = init_lattice(shape)
    lib.ostp_set_stout(0.15, 2, 0.0, 0, 0, 1)
    lib.ostp_set_inverter_tricks(0, 0, 0.1, 10000)
    sizeh, vb = lat.sizeh, lat.vec3_bytes
    gb, tb = 8 * lat.su3_bytes, 8 * 64 * sizeh
    conf = Dev(nbytes=gb)
    lib.ostp_generate_Conf_cold(conf.p, 0.3, 4)
    u0 = conf.get(np.zeros(gb, np.uint8))
    sizes = {"conf_acc_bkp": gb, "aux_conf_acc": gb, "auxbis_conf_acc": gb, "gstout_conf_acc_arr": 2 * gb,
             "momenta": tb, "ipdot_acc": tb, "ferm_phi_acc": 2 * vb, "ferm_chi_acc": 2 * vb,
             "ferm_shiftmulti_acc": 19 * vb, "k_p_shiftferm": 19 * vb, "kloc_r": vb, "kloc_h": vb, "kloc_s": vb,
             "kloc_p": vb}
    bufs = {k: Dev(nbytes=n) for k, n in sizes.items()}
    for k, d in bufs.items():
        set_ptr(k, d.p)
    ph = Dev(nbytes=8 * 8 * sizeh)
    lib.calc_u1_phases(ph.p, ost.BfParam(0, 0, 0, 0, 0, 0), 0.0, 0.0)
    fps = (ost.FermParam * 2)()
    for f, (mass, deg, fi, md) in enumerate(FLAVOURS):
        fp = fps[f]
        fp.ferm_mass, fp.degeneracy, fp.number_of_ps, fp.index_of_the_first_ps = mass, deg, 1, f
        fp.phases = ph.p
        fp.approx_fi_mother = ost.read_remez(str(GOLDEN / fi))
        fp.approx_md_mother = ost.read_remez(str(GOLDEN / md))
        fp.approx_li_mother = ost.read_remez(str(GOLDEN / md))
    set_ptr("fermions_parameters", C.addressof(fps))
    ai = ost.AllocSettings.in_dll(lib, "alloc_info")
    ai.NDiffFlavs, ai.NPS_tot, ai.maxApproxOrder, ai.maxNeededShifts = 2, 2, 19, 19
    try:
        ds = []
        for no_md in (4, 8):
            set_md(no_md, 3, 0.5)
            conf.put(u0)
            lib.ostp_set_rng_seed(11, 0)
            lib.UPDATE_SOLOACC_UNOSTEP_VERSATILE(conf.p, 1e-12, 1e-12, 0, 0, 1, 50000)
            ost.check(0, "UPDATE_SOLOACC_UNOSTEP_VERSATILE")
            info = ost.RhmcInfo()
            assert lib.ostp_rhmc_last_info(C.byref(info)) == 0
            assert info.md_multishift_iterations > 0
            ds.append(info.delta_S)
        ratio = ds[0] / ds[1]
        assert abs(ratio - 4.0) < 1.0, (ds, ratio)
        # the flavours' rational solves (heat bath, MD force, acceptance) run
        # together or one by one: the same update bit for bit; and the same
        # again with an error an earlier call left recorded (non-aborting
        # mode, not yet read), which the update leaves in place
        runs = []
        for batch, pending in ((1, False), (0, False), (1, True)):
            prev = lib.ostp_set_multishift_batching(batch)
            try:
                conf.put(u0)
                lib.ostp_set_rng_seed(11, 0)
                if pending:
                    assert lib.ostp_set_multishift_precision(7, 0) == -1  # a bad mode: recorded, nothing changed
                    msg = lib.ostp_last_error()
                    assert msg
                lib.UPDATE_SOLOACC_UNOSTEP_VERSATILE(conf.p, 1e-12, 1e-12, 0, 0, 1, 50000)
                if pending:
                    assert lib.ostp_last_error() == msg
                    lib.ostp_clear_error()
                ost.check(0, "UPDATE_SOLOACC_UNOSTEP_VERSATILE")
            finally:
                lib.ostp_set_multishift_batching(prev)
            info = ost.RhmcInfo()
            lib.ostp_rhmc_last_info(C.byref(info))
            runs.append((info.delta_S, info.md_multishift_iterations, conf.get(np.zeros(gb, np.uint8))))
        for r in runs[1:]:
            assert r[0] == runs[0][0] and r[1] == runs[0][1]
            assert np.array_equal(r[2], runs[0][2])
    finally:
        for name in GLOBALS:
            set_ptr(name, None)



@pytest.mark.parametrize("shape, ps", [((2, 2, 2, 2), (1, 1)), ((6, 4, 4, 10), (2, 1)), ((4, 4, 4, 8), (2, 2)),
                                       ((16, 16, 16, 26), (2, 1))])
def test_systems_iterated_together_match_one_by_one(shape, ps):
    """Two, three and four systems in one CG-M iteration stream, on lattices
    with blocks that are not full and on one too large for split hops: the
    force is that of the one-by-one solves bit for bit."""
    F = Nf21(shape)
    vb = F.lat.vec3_bytes
    F.chi = Dev(nbytes=sum(ps) * vb)
    for k in range(sum(ps)):
        lib.ostp_generate_vec3_soa_gauss(F.chi.p + k * vb, 77, 10 + k)
    for f in range(2):
        F.fps[f].ferm_mass = 0.1 + 0.1 * f
        F.fps[f].number_of_ps, F.fps[f].index_of_the_first_ps = ps[f], f * ps[0]
    du = Dev(F.u0)
    forces = []
    for batch in (1, 0):
        prev = lib.ostp_set_multishift_batching(batch)
        try:
            ipd = Dev(nbytes=F.tb)
            lib.fermion_force_soloopenacc(du.p, F.arr.p, F.gl3.p, ipd.p, F.fps, 2, F.chi.p, F.res, F.taux.p, F.xs.p,
                                          F.ip(du.p), 50000)
            ost.check(0, "fermion_force_soloopenacc")
        finally:
            lib.ostp_set_multishift_batching(prev)
        forces.append(ipd.get(np.zeros(F.tb // 8)))
    assert np.abs(forces[0]).max() > 1e-3 and np.array_equal(forces[0], forces[1]), rel(forces[0], forces[1])


@pytest.mark.parametrize("batch", [1, 0])
@pytest.mark.parametrize("bad", [0, 1])
def test_failed_force_leaves_no_old_force(batch, bad):
    """A force that fails on the way (a flavour without phases, recorded as an
    error) leaves a zero force, and the flavours' sum as far as it came."""
    F = Nf21((4, 4, 4, 4))
    du = Dev(F.u0)
    F.ipd.put(np.ones(F.tb // 8))
    F.gl3.put(np.ones(F.gb // 8))
    F.fps[bad].phases = None
    prev = lib.ostp_set_multishift_batching(batch)
    lib.fermion_force_soloopenacc(du.p, F.arr.p, F.gl3.p, F.ipd.p, F.fps, 2, F.chi.p, F.res, F.taux.p, F.xs.p,
                                  F.ip(du.p), 50000)
    lib.ostp_set_multishift_batching(prev)
    msg = lib.ostp_last_error()
    lib.ostp_clear_error()
    assert b"null pointer" in msg
    assert not F.ipd.get(np.zeros(F.tb // 8)).any()
    gl3 = F.gl3.get(np.zeros(F.gb // 8))
    if batch or bad == 0:
        assert not gl3.any()
    else:
        assert not (gl3 == 1.0).any() and np.abs(gl3).max() > 1e-3


@pytest.mark.parametrize("shape, ps", [((4, 4, 4, 8), (1, 1)), ((16, 16, 16, 26), (1, 2))])
@pytest.mark.parametrize("window", [0, 8, 16])
def test_system_that_stops_where_a_batch_ends(shape, ps, window):
    """The second flavour's mass is chosen so that it stops at every iteration
    from 14 to 49 while the first goes on: before, at and after the end of the
    first batch (16), of the one that follows (at most 48) and of windows of 8,
    16 and 64 residuals.  The force is that of the one-by-one solves bit for
    bit, in the iterations of those."""
    F = Nf21(shape)
    lat, vb = F.lat, F.lat.vec3_bytes
    F.chi = Dev(nbytes=sum(ps) * vb)
    for k in range(sum(ps)):
        lib.ostp_generate_vec3_soa_gauss(F.chi.p + k * vb, 77, 10 + k)
    for f in range(2):
        F.fps[f].number_of_ps, F.fps[f].index_of_the_first_ps = ps[f], f * ps[0]
    F.fps[0].ferm_mass = 0.02
    du, ipd = Dev(F.u0), Dev(nbytes=F.tb)
    count = C.c_int.in_dll(lib, "multishift_invert_iterations")

    def force(batch, nflav=2):
        old = lib.ostp_set_multishift_batching(batch), lib.ostp_set_multishift_window(window)
        try:
            before = count.value
            lib.fermion_force_soloopenacc(du.p, F.arr.p, F.gl3.p, ipd.p, F.fps, nflav, F.chi.p, F.res, F.taux.p, F.xs.p,
                                          F.ip(du.p), 50000)
            ost.check(0, "fermion_force_soloopenacc")
            return ipd.get(np.zeros(F.tb // 8)), count.value - before
        finally:
            lib.ostp_set_multishift_batching(old[0])
            lib.ostp_set_multishift_window(old[1])

    slow = force(0, 1)[1] // ps[0]
    stops = {}
    for mass in np.geomspace(4.5, 0.05, 800 if shape[0] == 4 else 100):
        F.fps[1].ferm_mass = mass
        f0, its0 = force(0)
        stop = (its0 - slow * ps[0]) / ps[1]
        if stop in stops or not 14 <= stop <= 49:
            continue
        f1, its1 = force(1)
        stops[stop] = np.abs(f0).max() > 1e-3 and np.array_equal(f1, f0) and its1 == its0
    assert slow > 60 and {16} | set(range(14, 50) if shape[0] == 4 else []) <= set(stops), (slow, sorted(stops))
    assert all(stops.values()), [k for k, ok in stops.items() if not ok]


def test_config5_trajectory_reversible_48x48x48x12():
    F = Nf21((48, 48, 48, 12), eps=0.5, seed=7, res=1e-10)
    moved, back_u, back_m = forward_back(F, 10, 5, 1.0, 2026)
    assert moved > 1e-3 and back_u < 1e-9 and back_m < 1e-9, (moved, back_u, back_m)
