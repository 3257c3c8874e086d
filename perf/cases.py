"""Measured cases of the library, through its C entry points on torch tensors.

What a staggered RHMC program and its measurements spend their time on: the Dslash, the CG, mixed-precision,
multi-shift and batched solvers, stout smearing, the gauge part of the molecular dynamics and the fermion force.
Fields are generated with torch from a seed; `exact` computes the same outputs with torch in 64 bits from the
formulas (hop by hop, loop by loop, the force by automatic differentiation through the smearing).

Layouts (reference structure of arrays, S = half-sites): gauge field [8 link arrays 2 mu + parity][18 S doubles: row,
column, site, re/im; + S doubles K under parallel tempering], vector [3][S] complex, phases [8][S], tamat/thmat
[8][3 S complex c01, c02, c12; S c00; S c11].
"""
import ctypes as C
import math

import torch

RHO, LEVELS = 0.15, 2
C0, C1 = 5.0 / 3.0, -1.0 / 12.0
BETA, GAUGE_STEPS, TAU, OUTER = 3.8, 5, 1.0, 10
DELTA = 0.1         # mixed precision: reliable update when the residual has fallen by this
GRAPH_ITERATIONS = 16

# thin links: plaquette about 0.56, that of a thermalised ensemble; links as the fermions see them after smearing: 0.9
THIN, SMOOTH = 0.235, 0.115


# ------------------------------------------------------------------------------------------------ the cases
def _case(op, shape, **more):
    c = {"op": op, "n0": shape[0], "n1": shape[1], "n2": shape[2], "n3": shape[3], "phases": "signs", "par_temp": False}
    c.update(more)
    return c


def listed():
    return [
        # one D_oe, D_eo pair on the smallest test lattice, entry points that wait: launch latency
        _case("hop", (8, 8, 8, 8), name="hop_8x8x8x8", queued=False),
        # the headline benchmark: the pair at 32^4, queued back to back
        _case("hop", (32, 32, 32, 32), name="hop_32x32x32x32", queued=True),
        # M^+ M in single precision with a background field and imaginary chemical potential, ragged extents
        _case("matrix_f", (30, 26, 22, 18), name="matrix_f32_30x26x22x18", phases="field"),
        # plain CG on a small finite-temperature lattice, no background field
        _case("cg", (16, 16, 16, 4), name="cg_16x16x16x4", mass=0.02, res=1e-10),
        # mixed-precision CG of a measurement on a production finite-temperature lattice
        _case("mixed", (32, 32, 32, 8), name="mixed_32x32x32x8", mass=0.01, res=1e-10, phases="field"),
        # the rational solve of a heat bath or an acceptance test at 32^4
        _case("rational", (32, 32, 32, 32), name="rational_32x32x32x32", mass=0.01, res=1e-10, order=19),
        # the same for a small ragged lattice with a background field
        _case("rational", (12, 14, 10, 6), name="rational_12x14x10x6", mass=0.05, res=1e-8, order=9, phases="field"),
        # noise sources of a measurement solved together, FP16 inner storage
        _case("batch", (24, 24, 24, 8), name="batch_24x24x24x8", mass=0.02, res=1e-9, systems=12),
        # stout smearing of an RHMC lattice
        _case("stout", (48, 48, 48, 12), name="stout_48x48x48x12"),
        # the gauge sub-integrator between two fermion forces of an RHMC trajectory
        _case("gauge", (48, 48, 48, 12), name="gauge_48x48x48x12"),
        # the same on a small ragged parallel-tempering replica
        _case("gauge", (18, 14, 10, 6), name="gauge_18x14x10x6", par_temp=True),
        # the fermion force of two flavours: rational solves, outer products, the smearing's force chain
        _case("force", (32, 32, 32, 8), name="force_32x32x32x8", res=1e-8, order=19),
    ]


def _even(rng, lo, hi):
    """An even extent, spread over the logarithm of the range."""
    return 2 * max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2))


def _extents(rng, lo, hi, half_sites):
    while True:
        n = [_even(rng, lo, hi) for _ in range(3)] + [_even(rng, 4, hi)]
        if rng.random() < 0.5:  # finite-temperature lattice: equal space, short time
            n = [n[0]] * 3 + [_even(rng, 4, max(4, n[0] // 2))]
        if n[0] * n[1] * n[2] * n[3] // 2 <= half_sites:
            return tuple(n)


def draw(rng):
    op = rng.choice(["hop", "matrix_f", "cg", "mixed", "rational", "batch", "stout", "gauge", "force"])
    ph = rng.choice(["signs", "field"])
    if op in ("hop", "matrix_f"):
        more = {"phases": ph}
        if op == "hop":
            more["queued"] = rng.random() < 0.5
        return _case(op, _extents(rng, 6, 48, 2 ** 19), **more)
    if op in ("cg", "mixed"):
        return _case(op, _extents(rng, 6, 36, 2 ** 18), mass=rng.choice([0.01, 0.02, 0.05]),
                     res=rng.choice([1e-8, 1e-9, 1e-10]), phases=ph)
    if op == "rational":
        return _case(op, _extents(rng, 6, 32, 2 ** 18), mass=rng.choice([0.01, 0.02, 0.05]),
                     res=rng.choice([1e-8, 1e-9]), order=rng.choice([8, 9, 15, 19]), phases=ph)
    if op == "batch":
        return _case(op, _extents(rng, 6, 24, 2 ** 16), mass=rng.choice([0.02, 0.05]), res=rng.choice([1e-8, 1e-9]),
                     systems=rng.randint(2, 16), phases=ph)
    if op == "stout":
        return _case(op, _extents(rng, 6, 48, 2 ** 19))
    if op == "gauge":
        return _case(op, _extents(rng, 6, 40, 2 ** 18), par_temp=rng.random() < 0.3)
    return _case(op, _extents(rng, 6, 28, 2 ** 17), res=1e-8, order=rng.choice([9, 15, 19]), phases=ph)


# --------------------------------------------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _shape(case):
    return case["n0"], case["n1"], case["n2"], case["n3"]


def _half(case):
    n = _shape(case)
    return n[0] * n[1] * n[2] * n[3] // 2


def _coordinates(case, dev):
    """[parity][direction] coordinates of the half-sites."""
    n = _shape(case)
    i = torch.arange(_half(case), device=dev)
    h, i = i % (n[0] // 2), i // (n[0] // 2)
    x1, i = i % n[1], i // n[1]
    x2, x3 = i % n[2], i // n[2]
    return [[2 * h + (x1 + x2 + x3 + p) % 2, x1, x2, x3] for p in (0, 1)]


def _normal(g, dev, *shape):
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, device=dev, dtype=torch.float64)) / math.sqrt(2.0)


def _links(case, g, dev, eps):
    """Random SU(3) near the identity: [8][3][3][S] (Gram-Schmidt of 1 + eps times complex normal entries)."""
    S = _half(case)
    u = torch.empty(8, 3, 3, S, dtype=torch.complex128, device=dev)
    for l in range(8):
        a = eps * math.sqrt(2.0) * _normal(g, dev, 2, 3, S)
        a[0, 0] += 1.0
        a[1, 1] += 1.0
        r0 = a[0] / a[0].abs().square().sum(0).sqrt()
        r1 = a[1] - (r0.conj() * a[1]).sum(0) * r0
        r1 = r1 / r1.abs().square().sum(0).sqrt()
        u[l, 0], u[l, 1] = r0, r1
        u[l, 2] = torch.linalg.cross(r0, r1, dim=0).conj()
    return u


def _phases(case, dev):
    """Staggered signs with antiperiodic time, and for "field" a magnetic field along direction 2 and an imaginary
    chemical potential (fractions of a turn reduced to [-1/2, 1/2], times 2 pi)."""
    n = _shape(case)
    out = torch.zeros(8, _half(case), dtype=torch.float64, device=dev)
    x = _coordinates(case, dev)
    for p in (0, 1):
        for mu in range(4):
            turns = 0.5 * (sum(x[p][:mu], torch.zeros_like(x[p][0])) % 2).double()
            if mu == 3:
                turns = turns + 0.5 * (x[p][3] == n[3] - 1)
            if case["phases"] == "field":
                flux = 4.0 / (n[0] * n[1])
                if mu == 0:
                    turns = turns - flux * n[0] * x[p][1] * (x[p][0] == n[0] - 1)
                if mu == 1:
                    turns = turns + flux * x[p][0]
                if mu == 3:
                    turns = turns + 0.05 / n[3]
            turns = turns - torch.ceil(turns - 0.5)
            out[2 * mu + p] = 2 * math.pi * turns
    return out


def _approximation(order, power, lo, hi):
    """x^(-power) on [lo, hi] as sum_k a_k / (x + b_k): trapezoidal rule in log s of the integral
    sin(pi power) / pi int ds s^(-power) / (x + s)."""
    t0, t1 = math.log(lo / 10.0), math.log(hi * 10.0)
    h = (t1 - t0) / (order - 1)
    t = [t0 + k * h for k in range(order)]
    return [math.sin(math.pi * power) / math.pi * h * math.exp((1.0 - power) * v) for v in t], [math.exp(v) for v in t]


# the two flavours of the force: mass, degeneracy and power of the molecular-dynamics approximation
FLAVOURS = ((0.01, 0.5), (0.05, 0.25))


def _rational(case):
    if case["op"] == "force":
        return [_approximation(case["order"], p, m * m, 8.0) for m, p in FLAVOURS]
    return [_approximation(case["order"], 0.25, case["mass"] ** 2, 8.0)]


def _inputs(case, seed):
    dev, op = _device(), case["op"]
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) + 1)
    S = _half(case)
    i = {"links": _links(case, g, dev, THIN if op in ("stout", "gauge", "force") else SMOOTH)}
    if op not in ("stout", "gauge"):
        i["phases"] = _phases(case, dev)
    if op == "batch":
        # Z2 noise
        i["b"] = (2.0 * torch.randint(0, 2, (case["systems"], 3, S), generator=g, device=dev) - 1.0).to(torch.complex128)
    elif op == "force":
        i["b"] = _normal(g, dev, len(FLAVOURS), 3, S)
    elif op not in ("stout", "gauge"):
        i["b"] = _normal(g, dev, 3, S)
    if op == "gauge":
        # momenta of the standard normal distribution in the Gell-Mann basis
        e = torch.randn(8, 8, S, generator=g, device=dev, dtype=torch.float64) / math.sqrt(2.0)
        i["mom"] = {"c": torch.complex(e[:, (0, 3, 5)], -e[:, (1, 4, 6)]),
                    "d": torch.stack([e[:, 2] + e[:, 7] / math.sqrt(3.0), -e[:, 2] + e[:, 7] / math.sqrt(3.0)], 1)}
        if case["par_temp"]:
            # a replica's defect: half the links through the last slice along direction 0
            n, x = _shape(case), _coordinates(case, dev)
            k = torch.ones(8, S, dtype=torch.float64, device=dev)
            for p in (0, 1):
                on = (x[p][0] == n[0] - 1) & (x[p][1] < n[1] // 2) & (x[p][2] < n[2] // 2) & (x[p][3] < n[3])
                k[p][on] = 0.4
            i["K"] = k
    return i


def _pack(links, k=None, single=False):
    v = torch.view_as_real(links).reshape(8, -1)
    if k is not None:
        v = torch.cat([v, k], 1)
    return (v.float() if single else v).contiguous()


def _pack_hermitian(m):
    return torch.cat([torch.view_as_real(m["c"].contiguous()).reshape(8, -1), m["d"].reshape(8, -1)], 1).contiguous()


# ------------------------------------------------------------------------------------------ prepare and run
def _at(t, offset=0):
    return t.data_ptr() + offset


def prepare(case, seed):
    import openstaple_amd as ost
    from openstaple_amd import lib
    op, S, dev = case["op"], _half(case), _device()
    ost.Lattice(*_shape(case), par_temp=case["par_temp"]).init()
    lib.ostp_set_sync_at_return(0 if case.get("queued") else 1)
    lib.ostp_set_stout(RHO, LEVELS, 0.0, 0, 0, 1)
    lib.ostp_set_inverter_tricks(0, 0, DELTA, 10000)
    i = _inputs(case, seed)
    vec = lambda *n: torch.zeros(*n, 3, S, dtype=torch.complex128, device=dev)  # noqa: E731
    vecf = lambda *n: torch.zeros(*n, 3, S, dtype=torch.complex64, device=dev)  # noqa: E731
    s = {"case": dict(case), "lib": lib, "ost": ost, "u": _pack(i["links"], i.get("K")), "cg": C.c_int(0)}
    s["gb"] = s["u"].numel() * 8
    if "phases" in i:
        s["ph"] = i["phases"]
    if "b" in i:
        s["b"] = i["b"]
    if op in ("matrix_f", "mixed", "batch"):
        s["uf"], s["phf"] = _pack(i["links"], single=True), i["phases"].float()
    if op == "hop":
        s["h"], s["out"] = vec(), vec()
    elif op == "matrix_f":
        s["b"] = s["b"].to(torch.complex64)
        s["t"], s["out"] = vecf(), vecf()
        s["fp"] = ost.ferm_param(0.02, _at(s["ph"]), _at(s["phf"]))
    elif op in ("cg", "mixed", "rational"):
        s["fp"] = ost.ferm_param(case["mass"], _at(s["ph"]), _at(s["phf"]) if op == "mixed" else None)
        s["work"] = vec(4)
        s["w"] = [_at(s["work"], 48 * S * k) for k in range(4)]
        if op == "rational":
            a, b = _rational(case)[0]
            s["ra"] = ost.rational_approx(0.0, a, b)
            s["out"], s["dirs"] = vec(case["order"]), vec(case["order"])
        else:
            s["out"] = vec()
        if op == "mixed":
            s["work_f"] = vecf(5)
            f = [_at(s["work_f"], 24 * S * k) for k in range(5)]
            ip = s["ip"] = ost.InverterPackage()
            ip.u, ip.u_f = _at(s["u"]), _at(s["uf"])
            ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = s["w"]
            ip.loc_r_f, ip.loc_h_f, ip.loc_s_f, ip.loc_p_f, ip.out_f = f
    elif op == "batch":
        n = case["systems"]
        s["out"] = vec(n)
        s["systems"] = (ost.BatchSystem * n)()
        for k, q in enumerate(s["systems"]):
            q.nd[:] = _shape(case)
            q.par_temp, q.mass = 0, case["mass"]
            q.u, q.u_f, q.phases, q.phases_f = _at(s["u"]), _at(s["uf"]), _at(s["ph"]), _at(s["phf"])
            q.in_, q.out = _at(s["b"], 48 * S * k), _at(s["out"], 48 * S * k)
        s["counts"] = ((C.c_int * n)(), (C.c_int * n)(), (C.c_double * n)())
    elif op == "stout":
        s["out"] = torch.zeros(LEVELS, *s["u"].shape, dtype=torch.float64, device=dev)
    elif op == "gauge":
        s["mom"] = _pack_hermitian(i["mom"])
        s["ipdot"], s["staples"] = torch.zeros_like(s["mom"]), torch.zeros_like(s["u"])
        ost.ActionParam.in_dll(lib, "act_params").beta = BETA
        md = ost.MdParam(no_md=OUTER, gauge_scale=GAUGE_STEPS, t=TAU)
        C.memmove(C.addressof(ost.MdParam.in_dll(lib, "md_parameters")), C.addressof(md), C.sizeof(md))
        lib.initialize_md_global_variables(md)
    elif op == "force":
        n = case["order"]
        s["smeared"] = torch.zeros(LEVELS, *s["u"].shape, dtype=torch.float64, device=dev)
        s["gl3"], s["aux"] = torch.zeros_like(s["u"]), torch.zeros_like(s["u"])
        s["ipdot"] = torch.zeros(8, 8 * S, dtype=torch.float64, device=dev)
        s["shifted"], s["dirs"], s["work"] = vec(n), vec(n), vec(4)
        s["flavours"] = (ost.FermParam * len(FLAVOURS))()
        for k, (fp, (mass, _), (a, b)) in enumerate(zip(s["flavours"], FLAVOURS, _rational(case))):
            fp.ferm_mass, fp.degeneracy, fp.number_of_ps, fp.index_of_the_first_ps = mass, 1, 1, k
            fp.phases = _at(s["ph"])
            fp.approx_md = ost.rational_approx(0.0, a, b)
        ip = s["ip"] = ost.InverterPackage()
        ip.u, ip.ferm_shift_temp, ip.nshifts = _at(s["u"]), _at(s["dirs"]), n
        ip.loc_r, ip.loc_h, ip.loc_s, ip.loc_p = [_at(s["work"], 48 * S * k) for k in range(4)]
    if dev.type == "cuda":
        torch.cuda.synchronize()  # torch's stream and the library's are not ordered against each other
    return s


def run(s):
    lib, case = s["lib"], s["case"]
    op = case["op"]
    if op == "hop":
        lib.acc_Doe(_at(s["u"]), _at(s["h"]), _at(s["b"]), _at(s["ph"]))
        lib.acc_Deo(_at(s["u"]), _at(s["out"]), _at(s["h"]), _at(s["ph"]))
        return {"odd": s["h"], "even": s["out"]}
    if op == "matrix_f":
        lib.fermion_matrix_multiplication_shifted_f(_at(s["uf"]), _at(s["out"]), _at(s["b"]), _at(s["t"]),
                                                    C.byref(s["fp"]), 0.01)
        return s["out"]
    if op in ("cg", "mixed"):
        lib.set_vec3_soa_to_zero(_at(s["out"]))
        if op == "cg":
            ok = lib.ker_invert_openacc(_at(s["u"]), C.byref(s["fp"]), _at(s["out"]), _at(s["b"]), case["res"], *s["w"],
                                        20000, 0.0, C.byref(s["cg"]))
        else:
            ok = lib.inverter_mixed_precision(s["ip"], C.byref(s["fp"]), _at(s["out"]), _at(s["b"]), case["res"], 20000,
                                              0.0, C.byref(s["cg"]))
        if ok != s["ost"].INVERTER_SUCCESS:
            raise RuntimeError("%s did not converge (%d iterations)" % (op, s["cg"].value))
        return s["out"]
    if op == "rational":
        ok = lib.multishift_invert(_at(s["u"]), C.byref(s["fp"]), C.byref(s["ra"]), _at(s["out"]), _at(s["b"]),
                                   case["res"], *s["w"], _at(s["dirs"]), 20000, C.byref(s["cg"]))
        if ok != s["ost"].INVERTER_SUCCESS:
            raise RuntimeError("rational solve did not converge (%d iterations)" % s["cg"].value)
        return s["out"]
    if op == "batch":
        for q in s["systems"]:
            lib.set_vec3_soa_to_zero(q.out)
        done = lib.ostp_batched_half_solve(case["systems"], s["systems"], case["res"], 20000, DELTA, GRAPH_ITERATIONS,
                                           *s["counts"])
        if done != case["systems"]:
            raise RuntimeError("%d of %d systems converged" % (done, case["systems"]))
        return s["out"]
    if op == "stout":
        lib.stout_wrapper(_at(s["u"]), _at(s["out"]), 0)
        return s["out"]
    if op == "gauge":
        lib.multistep_2MN_gauge(_at(s["u"]), _at(s["staples"]), _at(s["ipdot"]), _at(s["mom"]))
        return {"links": s["u"], "momenta": s["mom"], "force": s["ipdot"], "staples": s["staples"]}
    lib.fermion_force_soloopenacc(_at(s["u"]), _at(s["smeared"]), _at(s["gl3"]), _at(s["ipdot"]), s["flavours"],
                                  len(FLAVOURS), _at(s["b"]), case["res"], _at(s["aux"]), _at(s["shifted"]), s["ip"], 20000)
    return {"force": s["ipdot"], "smeared": s["smeared"]}


# ------------------------------------------------------------------------------------------------------ work
def _iterations(case, mass, shift):
    """About what CG takes: the smallest eigenvalue is m^2 plus that of the lowest momentum, the largest about 4."""
    low = mass * mass + shift + 0.6 * math.sin(math.pi / case["n3"]) ** 2
    return max(10.0, 0.4 * math.sqrt(4.0 / low) * math.log(2.0 / case["res"]))


def work(case):
    """Each kernel-level operation's inputs read once and outputs written once: a hop reads 8 links of two rows (768 B a
    half-site in FP64), 8 phases and a vector and writes one; a CG iteration is two hops and the recurrence's vectors."""
    S, op = _half(case), case["op"]
    hop, flops = 768 + 64 + 48 + 48, 570.0
    if op == "hop":
        return {"bytes": 2 * hop * S, "flops": 2 * flops * S}
    if op == "matrix_f":
        return {"bytes": (hop + 24) * S, "flops": 2 * flops * S}
    if op == "cg":
        n = _iterations(case, case["mass"], 0.0)
        return {"bytes": n * (2 * hop + 48 + 288 + 144) * S, "flops": n * (2 * flops + 60) * S}
    if op == "mixed":
        n = _iterations(case, case["mass"], 0.0)
        return {"bytes": n * (hop + 240) * S, "flops": n * (2 * flops + 60) * S}
    if op == "rational":
        n = _iterations(case, case["mass"], _rational(case)[0][1][0])
        return {"bytes": (n * (2 * hop + 48 + 288) + 2 * 96 * case["order"]) * S, "flops": n * (2 * flops + 48) * S}
    if op == "batch":
        # FP16 inner storage: links read once an iteration for the systems that share them, vectors a system
        n = _iterations(case, case["mass"], 0.0)
        return {"bytes": n * (2 * 224 + case["systems"] * 150) * S, "flops": n * case["systems"] * (2 * flops + 60) * S}
    if op == "stout":
        return {"bytes": LEVELS * 192 * 8 * S, "flops": LEVELS * 2500.0 * 8 * S}
    if op == "gauge":
        forces, moves = 2 * GAUGE_STEPS + 1, 2 * GAUGE_STEPS
        return {"bytes": (forces * (96 + 192) + moves * 256 + 144) * 8 * S, "flops": (forces * 16830.0 + moves * 1200.0) * 8 * S}
    r = _rational(case)
    its = [_iterations(case, m, b[0]) for (m, _), (_, b) in zip(FLAVOURS, r)]
    solve = max(its) * 2 * (768 + 64) + sum(its) * (2 * 96 + 48 + 288) + sum(2 * 96 * case["order"] for _ in its)
    chain = LEVELS * (192 + 350 + 600) * 8 + len(FLAVOURS) * 8 * (2 * 144 + 48)
    return {"bytes": (solve + chain) * S, "flops": (sum(its) * (2 * flops + 48) + LEVELS * 14000.0 * 8) * S}


def tolerance(case):
    """About four times what is seen against `exact` (hop 2.5e-16, M^+ M in single precision 1.1e-7, stout 2.5e-16, gauge 6e-16,
    force 0.7 res).  A solver's solution is off by its residual times the operator's condition (up to 40 res seen), and
    another correct solver may stop an iteration earlier or later."""
    op = case["op"]
    if op in ("hop", "stout"):
        return {"rel": 1e-15}
    if op == "matrix_f":
        return {"rel": 5e-7}
    if op == "gauge":
        return {"rel": 4e-15}
    if op == "force":
        return {"rel": 20.0 * case["res"], "max": 800.0 * case["res"]}
    return {"rel": 160.0 * case["res"], "max": 6400.0 * case["res"]}


# ----------------------------------------------------------------------------------- the same in plain torch
class _Lattice:
    """Half-site fields as [even, odd] lists of [S][3][3] matrices or [S][3] vectors."""

    def __init__(self, case, dev):
        n, x = _shape(case), _coordinates(case, dev)
        self.to = {}
        for p in (0, 1):
            for mu in range(4):
                for sign in (1, -1):
                    y = list(x[p])
                    y[mu] = (y[mu] + sign) % n[mu]
                    self.to[p, mu, sign] = (y[0] + n[0] * (y[1] + n[1] * (y[2] + n[2] * y[3]))) // 2

    def shift(self, f, mu, sign):
        """f(x + sign mu) at every x."""
        return [f[1 - p][self.to[p, mu, sign]] for p in (0, 1)]


def _mm(a, b):
    return a[..., :, 0:1] * b[..., 0:1, :] + a[..., :, 1:2] * b[..., 1:2, :] + a[..., :, 2:3] * b[..., 2:3, :]


def _mul(a, b):
    return [_mm(x, y) for x, y in zip(a, b)]


def _dag(a):
    return [x.conj().transpose(-1, -2) for x in a]


def _add(a, b, f=1.0):
    return [x + f * y for x, y in zip(a, b)]


def _matrices(links):
    """[mu][parity] matrices of [8][3][3][S] link arrays."""
    return [[links[2 * mu + p].permute(2, 0, 1).contiguous() for p in (0, 1)] for mu in range(4)]


def _ta(m):
    """Traceless anti-Hermitian part."""
    a = 0.5 * (m - m.conj().transpose(-1, -2))
    tr = (a[..., 0, 0] + a[..., 1, 1] + a[..., 2, 2]) / 3.0
    return a - tr[..., None, None] * torch.eye(3, dtype=a.dtype, device=a.device)


def _exp(a, terms=26):
    """Taylor series of matrices of norm below about 2."""
    one = torch.eye(3, dtype=a.dtype, device=a.device).expand_as(a)
    e = one
    for k in range(terms, 0, -1):
        e = one + _mm(a, e) / k
    return e


def _hop(lat, w, v, parity):
    """1/2 sum_mu [W_mu(x) v(x+mu) - W_mu(x-mu)^+ v(x-mu)] on the sites of `parity`, v on the others."""
    out = 0
    for mu in range(4):
        out = out + (w[mu][parity] * v[lat.to[parity, mu, 1]][:, None, :]).sum(-1)
        back = lat.to[parity, mu, -1]
        out = out - (w[mu][1 - parity][back].conj() * v[back][:, :, None]).sum(-2)
    return 0.5 * out


def _phased(u, phases):
    return [[u[mu][p] * torch.polar(torch.ones_like(phases[0]), phases[2 * mu + p])[:, None, None] for p in (0, 1)]
            for mu in range(4)]


def _solve(lat, w, mass, shifts, b, res):
    """(m^2 + sigma_k - D_eo D_oe) x_k = b for all shifts together (CG of the smallest one and the shifted recurrences)."""
    op = lambda v: (mass * mass + shifts[0]) * v - _hop(lat, w, _hop(lat, w, v, 1), 0)  # noqa: E731
    ds = [x - shifts[0] for x in shifts]
    n = len(shifts)
    x, p = [torch.zeros_like(b) for _ in range(n)], [b.clone() for _ in range(n)]
    r, rr = b.clone(), float(b.abs().square().sum())
    z_old, z = [1.0] * n, [1.0] * n
    a_old, beta, stop = 1.0, 0.0, rr * res * res
    for _ in range(20000):
        q = op(p[0])
        a = rr / float((p[0].conj() * q).sum().real)
        r -= a * q
        new = float(r.abs().square().sum())
        b_new = new / rr
        x[0] += a * p[0]
        for k in range(1, n):
            if z[k] * z[k] * rr < 1e-4 * stop:
                continue
            zn = z[k] * z_old[k] * a_old / (a * beta * (z_old[k] - z[k]) + z_old[k] * a_old * (1.0 + ds[k] * a))
            x[k] += (a * zn / z[k]) * p[k]
            p[k] = zn * r + (b_new * (zn / z[k]) ** 2) * p[k]
            z_old[k], z[k] = z[k], zn
        p[0] = r + b_new * p[0]
        a_old, beta, rr = a, b_new, new
        if rr < stop:
            return x
    raise RuntimeError("the reference solve did not converge")


def _staples(lat, u, mu, nu):
    """(up, down) plaquette staples of the links along mu in the plane (mu, nu)."""
    a, m, n = lat.shift(u[nu], mu, 1), _dag(lat.shift(u[mu], nu, 1)), _dag(u[nu])
    up = _mul(_mul(a, m), n)
    a, m, n = _dag(lat.shift(lat.shift(u[nu], mu, 1), nu, -1)), _dag(lat.shift(u[mu], nu, -1)), lat.shift(u[nu], nu, -1)
    return up, _mul(_mul(a, m), n)


def _stout(lat, u):
    out = []
    for mu in range(4):
        c = None
        for nu in range(4):
            if nu != mu:
                for st in _staples(lat, u, mu, nu):
                    c = st if c is None else _add(c, st)
        out.append([_mm(_exp(-RHO * _ta(x)), v) for x, v in zip(_mul(u[mu], c), u[mu])])
    return out


def _gauge_staples(lat, u):
    """Sum of the plaquette (times C0) and rectangle (times C1) staples of every link."""
    plaq = {(mu, nu): _staples(lat, u, mu, nu) for mu in range(4) for nu in range(4) if mu != nu}
    out = []
    for mu in range(4):
        c = None
        for nu in range(4):
            if nu == mu:
                continue
            for side in (0, 1):
                if side == 0:
                    a, m, n = lat.shift(u[nu], mu, 1), _dag(lat.shift(u[mu], nu, 1)), _dag(u[nu])
                    far = lat.shift(plaq[mu, nu][0], nu, 1)
                    right = _mul(_mul(u[mu], lat.shift(u[nu], mu, 1)), m)
                    left = _mul(_mul(m, n), u[mu])
                else:
                    a = _dag(lat.shift(lat.shift(u[nu], mu, 1), nu, -1))
                    m, n = _dag(lat.shift(u[mu], nu, -1)), lat.shift(u[nu], nu, -1)
                    far = lat.shift(plaq[mu, nu][1], nu, -1)
                    right = _mul(_mul(u[mu], a), m)
                    left = _mul(_mul(m, n), u[mu])
                right, left = lat.shift(right, mu, 1), lat.shift(left, mu, -1)
                t = [C0 * x for x in plaq[mu, nu][side]]
                t = _add(t, _mul(_mul(a, far), n), C1)
                t = _add(t, _mul(_mul(right, m), n), C1)
                t = _add(t, _mul(_mul(a, m), left), C1)
                c = t if c is None else _add(c, t)
        out.append(c)
    return out


def _tamat(m):
    """tamat planes of [mu][parity] anti-Hermitian matrices."""
    c = torch.stack([torch.stack([m[mu][p][:, 0, 1], m[mu][p][:, 0, 2], m[mu][p][:, 1, 2]]) for mu in range(4) for p in (0, 1)])
    d = torch.stack([torch.stack([m[mu][p][:, 0, 0].imag, m[mu][p][:, 1, 1].imag]) for mu in range(4) for p in (0, 1)])
    return torch.cat([torch.view_as_real(c).reshape(8, -1), d.reshape(8, -1)], 1)


def _planes(m, rows=3):
    """Link arrays of [mu][parity] matrices; rows from `rows` on are zero."""
    u = torch.stack([m[mu][p].permute(1, 2, 0) for mu in range(4) for p in (0, 1)])
    if rows < 3:
        u = u.clone()
        u[:, rows:] = 0
    return u


def _exact_gauge(lat, i):
    u0 = _matrices(i["links"])
    k = [[i["K"][2 * mu + p][:, None, None] if "K" in i else 1.0 for p in (0, 1)] for mu in range(4)]
    u = u0
    mom = []
    for mu in range(4):
        mom.append([])
        for p in (0, 1):
            c, d = i["mom"]["c"][2 * mu + p], i["mom"]["d"][2 * mu + p]
            h = torch.zeros(d.shape[1], 3, 3, dtype=torch.complex128, device=d.device)
            h[:, 0, 1], h[:, 0, 2], h[:, 1, 2] = c[0], c[1], c[2]
            h = h + h.conj().transpose(-1, -2)
            h[:, 0, 0], h[:, 1, 1], h[:, 2, 2] = d[0], d[1], -d[0] - d[1]
            mom[mu].append(h)
    lam, unit = 0.1931833275037836, TAU / (2 * OUTER * GAUGE_STEPS)
    kick = [-unit * lam * BETA / 3.0, -unit * (1 - 2 * lam) * BETA / 3.0, -unit * 2 * lam * BETA / 3.0]
    steps = [kick[0]] + [kick[1], kick[2]] * (GAUGE_STEPS - 1) + [kick[1], kick[0]]
    for j, f in enumerate(steps):
        st = _gauge_staples(lat, [[u[mu][p] * k[mu][p] for p in (0, 1)] for mu in range(4)])
        st = [[st[mu][p] * k[mu][p] for p in (0, 1)] for mu in range(4)]
        force = [[_ta(_mm(u[mu][p], st[mu][p])) for p in (0, 1)] for mu in range(4)]
        mom = [[mom[mu][p] - 1j * f * force[mu][p] for p in (0, 1)] for mu in range(4)]
        if j + 1 < len(steps):
            u = [[_mm(_exp(0.5j * unit * mom[mu][p]), u[mu][p]) for p in (0, 1)] for mu in range(4)]
    links = _planes(u)
    links[:, 2] = i["links"][:, 2]  # the third rows are not written
    staples = _pack(_planes(st), torch.zeros_like(i["K"]) if "K" in i else None)
    momenta = _tamat([[1j * h for h in m] for m in mom])
    c = torch.view_as_complex(momenta[:, : 6 * i["links"].shape[-1]].reshape(8, -1, 2).contiguous()) / 1j
    momenta = torch.cat([torch.view_as_real(c).reshape(8, -1), momenta[:, 6 * i["links"].shape[-1]:]], 1)
    return {"links": _pack(links, i.get("K")), "momenta": momenta, "force": _tamat(force), "staples": staples}


def _exact_force(lat, case, i):
    thin = [[m.requires_grad_(True) for m in f] for f in _matrices(i["links"])]
    smeared, levels = thin, []
    for _ in range(LEVELS):
        smeared = _stout(lat, smeared)
        levels.append(_pack(_planes([[m.detach() for m in f] for f in smeared], rows=2)))
    w = _phased([[m.detach() for m in f] for f in smeared], i["phases"])
    x = _phased(smeared, i["phases"])
    total = 0
    for (mass, _), (a, b), src in zip(FLAVOURS, _rational(case), i["b"]):
        sols = _solve(lat, w, mass, b, src.transpose(0, 1).contiguous(), 1e-12)
        for ak, xk in zip(a, sols):
            hk = _hop(lat, w, xk, 1)
            for mu in range(4):
                # Re Tr of the phased link times the outer products that the force accumulates
                total = total + ak * (xk.conj() * (x[mu][0] * hk[lat.to[0, mu, 1]][:, None, :]).sum(-1)).sum().real
                total = total - ak * (hk.conj() * (x[mu][1] * xk[lat.to[1, mu, 1]][:, None, :]).sum(-1)).sum().real
    flat = [m for f in thin for m in f]
    g = torch.autograd.grad(total, flat)
    force = [-_ta(_mm(m.detach(), d.conj().transpose(-1, -2))) for m, d in zip(flat, g)]
    return {"force": _tamat([force[2 * mu:2 * mu + 2] for mu in range(4)]), "smeared": torch.stack(levels)}


def exact(case, seed):
    op, dev = case["op"], _device()
    i = _inputs(case, seed)
    lat = _Lattice(case, dev)
    if op == "gauge":
        return _exact_gauge(lat, i)
    if op == "force":
        return _exact_force(lat, case, i)
    if op == "stout":
        u, out = _matrices(i["links"]), []
        for _ in range(LEVELS):
            u = _stout(lat, u)
            out.append(_pack(_planes(u, rows=2)))
        return torch.stack(out)
    back = lambda v: v.transpose(0, 1).contiguous()  # noqa: E731
    if op == "matrix_f":
        # the single-precision inputs, in 64 bits
        w = _phased(_matrices(i["links"].to(torch.complex64).to(torch.complex128)), i["phases"].float().double())
        b = back(i["b"].to(torch.complex64).to(torch.complex128))
        return back((0.02 ** 2 + 0.01) * b - _hop(lat, w, _hop(lat, w, b, 1), 0))
    w = _phased(_matrices(i["links"]), i["phases"])
    if op == "hop":
        h = _hop(lat, w, back(i["b"]), 1)
        return {"odd": back(h), "even": back(_hop(lat, w, h, 0))}
    if op == "rational":
        return torch.stack([back(x) for x in _solve(lat, w, case["mass"], _rational(case)[0][1], back(i["b"]), 1e-13)])
    if op == "batch":
        return torch.stack([back(_solve(lat, w, case["mass"], [0.0], back(b), 1e-13)[0]) for b in i["b"]])
    return back(_solve(lat, w, case["mass"], [0.0], back(i["b"]), 1e-13)[0])
