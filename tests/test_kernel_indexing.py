"""CPU checks of the index arithmetic the HIP kernels use, before any launch:
the Dslash neighbour formula (k_dslash in openstaple_amd/csrc/dslash.hip) must
reproduce the oracle's neighbour tables and stay in [0, sizeh), and the
XCD-aware workgroup remap must be a bijection of [0, G)."""
import itertools
import subprocess

import numpy as np
import pytest

from oracle import Oracle
from test_krylov_host import build_host


def kernel_neighbours(nd, eo):
    """Vectorised restatement of the k_dslash index block for all threads."""
    nd0, nd1, nd2, nd3 = nd
    nd0h = nd0 // 2
    sizeh = nd0 * nd1 * nd2 * nd3 // 2
    idx = np.arange(sizeh, dtype=np.int64)
    t = idx // nd0h
    hd0 = idx - t * nd0h
    t2 = t // nd1
    d1 = t - t2 * nd1
    d3 = t2 // nd2
    d2 = t2 - d3 * nd2
    d0 = 2 * hd0 + ((d1 + d2 + d3 + eo) & 1)
    row = idx - hd0
    s1, s2 = nd0h, nd0h * nd1
    s3 = s2 * nd2
    ip0 = row + np.where(d0 + 1 == nd0, 0, (d0 + 1) >> 1)
    im0 = row + np.where(d0 == 0, (nd0 - 1) >> 1, (d0 - 1) >> 1)
    ip1 = idx + np.where(d1 == nd1 - 1, -(nd1 - 1) * s1, s1)
    im1 = idx + np.where(d1 == 0, (nd1 - 1) * s1, -s1)
    ip2 = idx + np.where(d2 == nd2 - 1, -(nd2 - 1) * s2, s2)
    im2 = idx + np.where(d2 == 0, (nd2 - 1) * s2, -s2)
    ip3 = idx + np.where(d3 == nd3 - 1, -(nd3 - 1) * s3, s3)
    im3 = idx + np.where(d3 == 0, (nd3 - 1) * s3, -s3)
    return np.stack([ip0, ip1, ip2, ip3], 1), np.stack([im0, im1, im2, im3], 1), sizeh


@pytest.mark.parametrize("shape", [(4, 4, 4, 4), (4, 6, 8, 10), (16, 4, 6, 2), (2, 2, 2, 2), (32, 32, 32, 32),
                                   (24, 24, 24, 8), (48, 48, 48, 12)])
@pytest.mark.parametrize("eo", [0, 1])
def test_dslash_neighbours_match_tables(shape, eo):
    ip, im, sizeh = kernel_neighbours(shape, eo)
    assert ip.min() >= 0 and ip.max() < sizeh and im.min() >= 0 and im.max() < sizeh
    if np.prod(shape) > 300000:
        return  # bounds only; the table comparison runs on the smaller shapes
    o = Oracle(*shape)
    nnp, nnm = o.nn_tables()
    par = 0 if eo == 0 else 1  # Deo writes even sites, Doe odd sites
    np.testing.assert_array_equal(ip, nnp[:, :, par])
    np.testing.assert_array_equal(im, nnm[:, :, par])


def xcd_block_id(i, G):
    q, r = G >> 3, G & 7
    x, k = i & 7, i >> 3
    return x * q + (x if x < r else r) + k


@pytest.mark.parametrize("G", list(range(1, 70)) + [256, 257, 1000, 2048, 4095, 4096, 5185])
def test_xcd_remap_is_a_bijection(G):
    ids = sorted(xcd_block_id(i, G) for i in range(G))
    assert ids == list(range(G))


def decode(idxh, parity, nd):
    """Restatement of `decode` in openstaple_amd/csrc/stout.hip."""
    nd0h = nd[0] >> 1
    t = idxh // nd0h
    hd0 = idxh - t * nd0h
    t2 = t // nd[1]
    d1 = t - t2 * nd[1]
    d3 = t2 // nd[2]
    d2 = t2 - d3 * nd[2]
    d0 = 2 * hd0 + ((d1 + d2 + d3 + parity) & 1)
    return [d0, d1, d2, d3]


def snum(d, nd):
    return (d[0] + nd[0] * (d[1] + nd[1] * (d[2] + nd[2] * d[3]))) >> 1


def shifted(d, mu, s, nu, t, nd):
    e = list(d)
    e[mu] = (e[mu] + s) % nd[mu]
    if t:
        e[nu] = (e[nu] + t) % nd[nu]
    return snum(e, nd)


@pytest.mark.parametrize("shape", [(4, 4, 4, 4), (4, 6, 8, 10), (16, 4, 6, 2)])
def test_link_kernel_site_decoding(shape):
    """decode/shifted of the per-link kernels (stout.hip, force.hip) agree with
    the neighbour tables and stay in bounds."""
    o = Oracle(*shape)
    nnp, nnm = o.nn_tables()
    sizeh = o.sizeh
    for parity in (0, 1):
        for i in range(sizeh):
            d = decode(i, parity, shape)
            assert snum(d, shape) == i and sum(d) % 2 == parity
            for mu in range(4):
                assert shifted(d, mu, 1, 0, 0, shape) == nnp[i, mu, parity]
                assert shifted(d, mu, -1, 0, 0, shape) == nnm[i, mu, parity]
                for nu in range(4):
                    if nu == mu:
                        continue
                    j = shifted(d, mu, 1, nu, -1, shape)
                    assert 0 <= j < sizeh
                    assert j == nnm[nnp[i, mu, parity], nu, 1 - parity]


def dslash_site_of_thread(G, nd3, sizeh, tmajor, block=256):
    """Restatement of the workgroup -> site mapping of k_dslash (dslash.hip)."""
    i = np.arange(G)
    q, r = G >> 3, G & 7
    x, k = i & 7, i >> 3
    blk = x * q + np.where(x < r, x, r) + k
    if tmajor:
        s3 = sizeh // nd3
        tile, tt = blk // nd3, blk % nd3
        base = tt * s3 + tile * block
    else:
        base = blk * block
    return (base[:, None] + np.arange(block)[None, :]).ravel()


@pytest.mark.parametrize("shape", [(32, 32, 32, 32), (24, 24, 24, 8), (32, 32, 32, 8), (48, 48, 48, 12),
                                   (16, 16, 16, 16), (4, 4, 4, 4), (4, 6, 8, 10)])
def test_dslash_workgroup_mapping_is_a_bijection(shape):
    sizeh = np.prod(shape) // 2
    s3 = sizeh // shape[3]
    tmajor = s3 % 256 == 0  # the launcher's condition
    G = (sizeh + 255) // 256
    idx = dslash_site_of_thread(G, shape[3], sizeh, tmajor)
    valid = idx[idx < sizeh]
    assert len(np.unique(valid)) == sizeh and valid.min() == 0
    if tmajor:
        assert idx.max() == sizeh - 1  # no thread beyond the lattice


def test_gauge_force_tile_arrays():
    """The LDS arrays of the gauge force's plane tiles (gf_plan and k_gf_tile in
    openstaple_amd/csrc/stout.hip): every record that a corner, a staple or a
    side reads lies inside its array, for every tile the plan accepts, and the
    multiply-shift division of item numbers is exact."""
    M, N, Cm, Cn, SMp, SMm, SNp, SNm = range(8)
    tiles = 0
    for tm, tn in itertools.product(range(1, 65), repeat=2):
        R = [(-2, -2, tm + 3, tn + 4), (-2, -2, tm + 4, tn + 3), (-1, -2, tm + 2, tn + 2), (-2, -1, tm + 2, tn + 2),
             (-1, 1, tm + 1, tn), (-1, -1, tm + 1, tn + 1), (1, -1, tm, tn + 1), (-1, -1, tm + 1, tn + 1)]
        n = [r[2] * r[3] for r in R]
        np_ = n[SMp] + n[SNp]
        links, items = n[M] + n[N], -(-np_ // 64) * 64 + n[SMm] + n[SNm]
        if not (tm * tn <= 64 and sum(n) <= 826 and links <= 292 and links <= 340 and n[Cm] + n[Cn] <= 256 and
                items <= 512 and links + 384 <= 826):
            continue
        tiles += 1
        for r in R:
            q = np.arange(512)
            assert np.array_equal((q * (-(-65536 // r[2]))) >> 16, q // r[2])

        def inside(role, i, j):
            a = R[role]
            assert a[0] <= i < a[0] + a[2] and a[1] <= j < a[1] + a[3], (tm, tn, role, i, j)

        def sites(role):
            a = R[role]
            return itertools.product(range(a[0], a[0] + a[2]), range(a[1], a[1] + a[3]))

        for role, reads in ((Cm, [(M, 0, 0), (N, 1, 0)]), (Cn, [(N, 0, 0), (M, 0, 1)]), (SMp, [(N, 1, 0), (Cn, 0, 0)]),
                            (SNp, [(M, 0, 1), (Cm, 0, 0)]), (SMm, [(Cm, 0, -1), (N, 0, -1)]),
                            (SNm, [(Cn, -1, 0), (M, -1, 0)])):
            for (i, j), (r, di, dj) in itertools.product(sites(role), reads):
                inside(r, i + di, j + dj)
        for d in (0, 1):  # links along mu, along nu; offsets along the own and the other direction
            O, P, Co, Cp, SOp, SOm, SPp, SPm = ((M, N, Cm, Cn, SMp, SMm, SNp, SNm), (N, M, Cn, Cm, SNp, SNm, SMp, SMm))[d]
            reads = [(P, 1, 0), (SOp, 0, 1), (P, 0, 0), (O, 0, 1), (SPm, 0, 0), (SPp, 1, 0), (Cp, 0, 0), (P, 0, -1),
                     (P, 1, -1), (SOm, 0, -1), (SPp, 1, -1), (O, 0, -1), (SPm, 0, -1), (Co, 0, -1), (O, 0, 0),
                     # K of the staples' links
                     (P, 1, 1), (O, 0, 2), (P, 0, 1), (P, -1, 0), (O, -1, 1), (O, -1, 0), (O, 1, 1), (P, 2, 0), (O, 1, 0),
                     (P, 1, -2), (O, 0, -2), (P, 0, -2), (P, 2, -1), (O, 1, -1), (P, -1, -1), (O, -1, -1)]
            for i, j, (r, o, p) in itertools.product((0, tm - 1), (0, tn - 1), reads):
                inside(r, i + (p if d else o), j + (o if d else p))
    assert tiles > 100


def test_link_record_offsets(tmp_path):
    """link_record (ostp_su3.h) over the largest array that the gauge force's
    tiles take (96 sizeh just below 2^32), with arithmetic overflow trapped."""
    src = tmp_path / "rec.cpp"
    src.write_text(r"""
#include "ostp_su3.h"
int main() {
    const int last = (int)(((1LL << 32) - 1) / 96) - 1;
    for (long long h : {0LL, 1LL, 22369621LL, 22369622LL, (long long)last})
        for (int e = 0; e < 6; e++)
            if (ostp::link_record((int)h, e) != h * 96 + e * 16) return 1;
    return 0;
}
""")
    build_host(src, tmp_path / "rec", "-fsanitize=signed-integer-overflow", "-fno-sanitize-recover=all")
    subprocess.run([str(tmp_path / "rec")], check=True)
