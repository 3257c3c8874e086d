// Stout smearing and its force chain on gfx950 (FP64).
//
//  smearing   U' = exp(-QA) U, QA = (rho/c0) TA(U * C), C = c0 * sum of the 6
//             staples (OpenAcc/stouting.c:27-165, plaquettes.c:196-259,
//             su3_utilities.c:210-239; Morningstar-Peardon hep-lat/0311018)
//  force      Sigma' -> Lambda -> Sigma (stouting.c:171-1302,
//             fermion_force.c:52-162; MP eqs. 57-75)
//
// One thread per link (8 link arrays x sizeh half-sites); the staple loop
// re-reads neighbouring links, which the L2 of the owning XCD serves
// (workgroups are remapped so each XCD walks a contiguous slab).  With about
// 2.5 kflop per link against 192 B of compulsory link traffic these kernels sit
// near the FP64 ridge; everything stays in FP64 as the reference does.
#include "ostp_blas.h"
#include "ostp_su3.h"

#include <algorithm>
#include <cmath>

extern "C" {
// action.h:23 and the staple normalisation of the gauge action (common_defines.h:71-84)
double gl_stout_rho = 0.15;
double gl_topo_rho = 0.0;
}

namespace ostp {

static double g_c_zero = 5.0 * 0.33333333333333333333333;  // tree-level Symanzik C_ZERO
static int g_stout_steps = 2;
static int g_topo_steps = 0;
static int g_topo_action = 0;
static bool g_tlsm = true;

bool gauge_action_tlsm() { return g_tlsm; }

struct LinkGeom {
    int nd[4];
    int sizeh;
};

// the 8 link arrays of a gauge field, contiguous at a fixed stride: a link
// array's address is arithmetic on a per-lane index, not a load from an
// array of pointers
struct GaugePtrs {
    const char* base;  // r0.c0 plane of link array 0; rows at +3k*sizeh, cols at +c*sizeh
    size_t stride;     // bytes between link arrays
    __device__ __forceinline__ const double2* at(int l) const { return (const double2*)(base + (size_t)l * stride); }
};

__device__ __forceinline__ void decode(int idxh, int parity, const LinkGeom& g, int d[4]) {
    const int nd0h = g.nd[0] >> 1;
    int t = idxh / nd0h;
    const int hd0 = idxh - t * nd0h;
    int t2 = t / g.nd[1];
    d[1] = t - t2 * g.nd[1];
    d[3] = t2 / g.nd[2];
    d[2] = t2 - d[3] * g.nd[2];
    d[0] = 2 * hd0 + ((d[1] + d[2] + d[3] + parity) & 1);
}

__device__ __forceinline__ int snum(const int d[4], const LinkGeom& g) {
    return (d[0] + g.nd[0] * (d[1] + g.nd[1] * (d[2] + g.nd[2] * d[3]))) >> 1;
}

// half-site index of x + s*e_mu (+ t*e_nu), periodic
__device__ __forceinline__ int shifted(const int d[4], int mu, int s, int nu, int t, const LinkGeom& g) {
    int e[4] = {d[0], d[1], d[2], d[3]};
    e[mu] += s;
    if (e[mu] < 0) e[mu] += g.nd[mu];
    if (e[mu] >= g.nd[mu]) e[mu] -= g.nd[mu];
    if (t != 0) {
        e[nu] += t;
        if (e[nu] < 0) e[nu] += g.nd[nu];
        if (e[nu] >= g.nd[nu]) e[nu] -= g.nd[nu];
    }
    return snum(e, g);
}

__device__ __forceinline__ void load_link(const double2* __restrict__ U, int sizeh, int i, Su3& m) {
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) m.c[r][c] = U[(3 * r + c) * sizeh + i];
    rebuild3row(m);
}
__device__ __forceinline__ void load_gl3(const double2* __restrict__ U, int sizeh, int i, Su3& m) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) m.c[r][c] = U[(3 * r + c) * sizeh + i];
}
__device__ __forceinline__ void store_rows(double2* __restrict__ U, int sizeh, int i, const Su3& m, int rows) {
    for (int r = 0; r < rows; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) U[(3 * r + c) * sizeh + i] = m.c[r][c];
}

__device__ __constant__ int c_perp[4][3] = {{1, 2, 3}, {0, 2, 3}, {0, 1, 3}, {0, 1, 2}};

// sum of the 6 staples of link (x, mu) times c0 (plaquettes.c:196-259)
__device__ __forceinline__ void staple_sum(const GaugePtrs& G, const LinkGeom& g, const int d[4], int idxh, int mu,
                                           int parity, double c0, Su3& acc) {
    su3_zero(acc);
    const int sh = g.sizeh;
    const int i_pmu = shifted(d, mu, 1, 0, 0, g);
    for (int it = 0; it < 3; it++) {
        const int nu = c_perp[mu][it];
        Su3 A, B, C, T;
        // right: U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+
        load_link(G.at(2 * nu + !parity), sh, i_pmu, A);
        load_link(G.at(2 * mu + !parity), sh, shifted(d, nu, 1, 0, 0, g), B);
        load_link(G.at(2 * nu + parity), sh, idxh, C);
        su3_mul_dag(A, B, T);
        su3_mul_dag(T, C, T);
        rebuild3row(T);
        su3_scale_add(c0, T, acc);
        // left: U_nu(x+mu-nu)^+ U_mu(x-nu)^+ U_nu(x-nu)
        const int i_mnu = shifted(d, nu, -1, 0, 0, g);
        load_link(G.at(2 * nu + parity), sh, shifted(d, mu, 1, nu, -1, g), A);
        load_link(G.at(2 * mu + !parity), sh, i_mnu, B);
        load_link(G.at(2 * nu + !parity), sh, i_mnu, C);
        Su3 AB;
        su3_mul(B, A, AB);      // A^+ B^+ = (B A)^+
        su3_dag_mul(AB, C, T);  // (B A)^+ C
        rebuild3row(T);
        su3_scale_add(c0, T, acc);
    }
}

__device__ __forceinline__ void link_of(int gid, int sizeh, int& dir, int& idxh) {
    dir = gid / sizeh;
    idxh = gid - dir * sizeh;
}
// The link of this thread in the kernels that read neighbour links (staples):
// blocks run over the 8 link arrays fastest, then over tiles of kBlock
// half-sites, and each XCD takes a contiguous range of blocks, so an XCD
// owns a slab of the lattice for every link array and re-reads the slab's
// neighbour links from its own L2 (with the link array slowest, every XCD
// swept the whole lattice for one array and fetched every neighbour link).
// Grid: 8 blocks per tile (nblk_tiles); false past the last half-site.
__device__ __forceinline__ bool link_of_tile(int sizeh, int& dir, int& idxh) {
    const int blk = xcd_block_id();
    dir = blk & 7;
    idxh = (blk >> 3) * kBlock + (int)threadIdx.x;
    return idxh < sizeh;
}


// ============================================================ gauge force
// Tree-level Symanzik (or Wilson) gauge force and action: plaquette staples
// times C_ZERO (plaquettes.c calc_loc_staples_nnptrick_all), rectangle
// staples of types A, B, C times C_ONE (rectangles.c:643-916), with the
// PAR_TEMP defect coefficients K (products of the staple's links, then the
// link's own K, su3_utilities.c:582-604), and ipdot = TA(U * staple)
// (conf_times_staples_ta_part, su3_utilities.c:146-174).

constexpr double kCOne = -0.25 * 0.33333333333333333333333;  // common_defines.h:75

// y = x + a e_mu + b e_nu, periodic (|a|, |b| <= 2 and every extent >= 2)
__device__ __forceinline__ void site_off(const int x[4], int mu, int a, int nu, int b, const LinkGeom& g, int y[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) y[i] = x[i];
    int v = y[mu] + a;
    v += v < 0 ? g.nd[mu] : 0;
    v -= v >= g.nd[mu] ? g.nd[mu] : 0;
    y[mu] = v;
    v = y[nu] + b;
    v += v < 0 ? g.nd[nu] : 0;
    v -= v >= g.nd[nu] ? g.nd[nu] : 0;
    y[nu] = v;
}

// U_dir(y): rows 0,1 loaded (row 2 is left for the caller to rebuild when a
// product needs it); *k = its K when the layout has one
__device__ __forceinline__ void link2_y(const GaugePtrs& G, const LinkGeom& g, int dir, const int y[4], int pt, Su3& m,
                                        double& k) {
    const int par = (y[0] + y[1] + y[2] + y[3]) & 1;
    const int i = snum(y, g);
    const double2* U = G.at(2 * dir + par);
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) m.c[r][c] = U[(size_t)(3 * r + c) * g.sizeh + i];
    k = pt ? ((const double*)(U + 9 * (size_t)g.sizeh))[i] : 1.0;
}
__device__ __forceinline__ void link_y(const GaugePtrs& G, const LinkGeom& g, int dir, const int y[4], int pt, Su3& m,
                                       double& k) {
    link2_y(G, g, dir, y, pt, m, k);
    rebuild3row(m);
}

// rows 0,1 of A B, A B^+ (A: rows 0,1; B: all rows); O may alias A
__device__ __forceinline__ void mul_r2(const Su3& A, const Su3& B, Su3& O) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
        double2 o[3];
#pragma unroll
        for (int c = 0; c < 3; c++) o[c] = cfma(A.c[r][2], B.c[2][c], cfma(A.c[r][1], B.c[1][c], cmul(A.c[r][0], B.c[0][c])));
#pragma unroll
        for (int c = 0; c < 3; c++) O.c[r][c] = o[c];
    }
}
__device__ __forceinline__ void mul_dag_r2(const Su3& A, const Su3& B, Su3& O) {
#pragma unroll
    for (int r = 0; r < 2; r++) {
        double2 o[3];
#pragma unroll
        for (int c = 0; c < 3; c++)
            o[c] = cfma(A.c[r][2], cconj(B.c[c][2]), cfma(A.c[r][1], cconj(B.c[c][1]), cmul(A.c[r][0], cconj(B.c[c][0]))));
#pragma unroll
        for (int c = 0; c < 3; c++) O.c[r][c] = o[c];
    }
}
// rows 0,1 of A^+ B (A, B: all rows); O must not alias A
__device__ __forceinline__ void dag_mul_r2(const Su3& A, const Su3& B, Su3& O) {
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            O.c[r][c] = cfma(cconj(A.c[2][r]), B.c[2][c], cfma(cconj(A.c[1][r]), B.c[1][c], cmul(cconj(A.c[0][r]), B.c[0][c])));
}

// five-link staple term m1^(d1) m2^(d2) m3^+ m4^(d4) m5^(d5) for the three
// shapes of rectangles.c: PPMMM (d = 0,0,1,1,1), PMMMP (0,1,1,1,0), MMMPP (1,1,1,0,0)
enum Shape : int { kPPMMM = 0, kPMMMP = 1, kMMMPP = 2 };
struct Hop {
    int dir, a, b;  // link U_dir at x + a e_mu + b e_nu
};
// rows 0,1 of m^+ (m: all rows)
__device__ __forceinline__ void dag_r2(const Su3& m, Su3& O) {
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) O.c[r][c] = cconj(m.c[c][r]);
}
// acc += s T (transposed = 0) or s T^+ (transposed = 1), T with all rows
__device__ __forceinline__ void add_term(double s, const Su3& T, int transposed, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double2 v = transposed ? cconj(T.c[c][r]) : T.c[r][c];
            acc.c[r][c] = make_double2(acc.c[r][c].x + s * v.x, acc.c[r][c].y + s * v.y);
        }
}
// The links of a wave's staple terms.  A wave of the gauge force covers 64
// sites of one link array (direction mu, parity p) and one plane nu, so mu,
// nu, p, the strides and the link array of every hop are wave-uniform and
// live in scalar registers; a lane keeps its site's lexicographic index and
// its mu, nu coordinates, and a neighbour x + a e_mu + b e_nu is
// (lex + a s_mu + b s_nu, wrapped) / 2 in the link array of parity
// p + a + b.  Loads are a scalar base plus a 32-bit lane offset.
struct PlaneCtx {
    const char* base;
    size_t stride;
    unsigned plane;  // bytes per colour plane (16 sizeh)
    int mu, nu, p, sm, sn, ndm, ndn;
    int lex, xm, xn;
};
__device__ __forceinline__ int pc_idx(const PlaneCtx& c, int a, int b) {
    const int ym = c.xm + a, yn = c.xn + b;
    int l = c.lex + a * c.sm + b * c.sn;
    l += ym < 0 ? c.ndm * c.sm : (ym >= c.ndm ? -c.ndm * c.sm : 0);
    l += yn < 0 ? c.ndn * c.sn : (yn >= c.ndn ? -c.ndn * c.sn : 0);
    return l >> 1;
}
// rows 0,1 of U_d(x + a e_mu + b e_nu), d = mu (which = 0) or nu (1); *k its K
__device__ __forceinline__ void pc_link2(const PlaneCtx& c, int which, int a, int b, int pt, Su3& m, double& k) {
    const int arr = __builtin_amdgcn_readfirstlane(2 * (which ? c.nu : c.mu) + ((c.p + a + b) & 1));
    const char* U = c.base + (size_t)arr * c.stride;
    const unsigned i16 = (unsigned)pc_idx(c, a, b) * 16u;
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int col = 0; col < 3; col++)
            m.c[r][col] = *(const double2*)(U + (i16 + (unsigned)(3 * r + col) * c.plane));
    k = pt ? *(const double*)(U + (size_t)9 * c.plane + (i16 >> 1)) : 1.0;
}
__device__ __forceinline__ void pc_link(const PlaneCtx& c, int which, int a, int b, int pt, Su3& m, double& k) {
    pc_link2(c, which, a, b, pt, m, k);
    rebuild3row(m);
}

// rows 0,1 (src_link2) or all rows (src_link) of a staple term's link and its K
__device__ __forceinline__ void src_link2(const PlaneCtx& c, int which, int a, int b, int pt, Su3& m, double& k) {
    pc_link2(c, which, a, b, pt, m, k);
}
__device__ __forceinline__ void src_link(const PlaneCtx& c, int which, int a, int b, int pt, Su3& m, double& k) {
    pc_link(c, which, a, b, pt, m, k);
}
// Each term is a chain of SU(3) products that carries only rows 0,1 and
// rebuilds row 2 at the end.  MMMPP is formed as its conjugate
// m5^+ m4^+ m3 m2 m1, a chain of the same kind, and added transposed.
template <int SH>
__device__ __forceinline__ void five(const PlaneCtx& pc, const Hop* h, int pt, double c1, Su3& acc) {
    double k = 1.0;
    auto ld = [&](int j, Su3& m, bool full) {
        double kj;
        pc_link2(pc, h[j].dir, h[j].a, h[j].b, pt, m, kj);
        if (full) rebuild3row(m);
        k *= kj;
    };
    // dagger pattern of the chain, in chain order
    constexpr int d1 = SH == kPPMMM ? 0 : SH == kPMMMP ? 0 : 1;
    constexpr int d2 = SH == kPPMMM ? 0 : 1;
    constexpr int d4 = SH == kPMMMP ? 1 : SH == kPPMMM ? 1 : 0;
    constexpr int d5 = SH == kPMMMP ? 0 : SH == kPPMMM ? 1 : 0;
    Su3 T, M;
    if (SH != kMMMPP) {
        ld(0, T, false);
        ld(1, M, true);
        if (d2) mul_dag_r2(T, M, T); else mul_r2(T, M, T);
        ld(2, M, true);
        mul_dag_r2(T, M, T);
        ld(3, M, true);
        if (d4) mul_dag_r2(T, M, T); else mul_r2(T, M, T);
        ld(4, M, true);
        if (d5) mul_dag_r2(T, M, T); else mul_r2(T, M, T);
    } else {
        (void)d1;
        ld(4, M, true);
        dag_r2(M, T);
        ld(3, M, true);
        mul_dag_r2(T, M, T);
        ld(2, M, true);
        mul_r2(T, M, T);
        ld(1, M, true);
        mul_r2(T, M, T);
        ld(0, M, true);
        mul_r2(T, M, T);
    }
    rebuild3row(T);
    add_term(k * c1, T, SH == kMMMPP, acc);
}

// rectangle staple terms A right/left, B right/left, C right/left
// (rectangles.c:691-718, 780-807, 865-892): the five links and the shape
__device__ __constant__ Hop c_rect_hops[6][5] = {
    {{1, 1, 0}, {1, 1, 1}, {0, 0, 2}, {1, 0, 1}, {1, 0, 0}},
    {{1, 1, -1}, {1, 1, -2}, {0, 0, -2}, {1, 0, -2}, {1, 0, -1}},
    {{0, 1, 0}, {1, 2, 0}, {0, 1, 1}, {0, 0, 1}, {1, 0, 0}},
    {{0, 1, 0}, {1, 2, -1}, {0, 1, -1}, {0, 0, -1}, {1, 0, -1}},
    {{1, 1, 0}, {0, 0, 1}, {0, -1, 1}, {1, -1, 0}, {0, -1, 0}},
    {{1, 1, -1}, {0, 0, -1}, {0, -1, -1}, {1, -1, -1}, {0, -1, 0}},
};
__device__ __constant__ int c_rect_shape[6] = {kPPMMM, kMMMPP, kPPMMM, kPMMMP, kPMMMP, kMMMPP};

// the staple terms of link (x, mu) in the plane (mu, nu), in the reference's
// order within the plane: plaquettes right and left times C_ZERO (plaquettes.c:
// 83-195), rectangles of types A, B, C right and left times C_ONE (rectangles.c:
// 691-718, 780-807, 865-892); K products of each term's links when pt
// A link of a staple term: U_d(x + a e_mu + b e_nu), d = mu (which = 0) or
// nu (1), daggered when dag.
struct HopD {
    int which, a, b, dag;
};
// T = L0 L1 ... L(N-1) with all rows; *k the product of the links' K
template <int N, class Src>
__device__ __forceinline__ void chain(const Src& pc, const HopD (&h)[N], int pt, Su3& T, double& k) {
    Su3 M;
    double kj;
    if (h[0].dag) {
        src_link(pc, h[0].which, h[0].a, h[0].b, pt, M, kj);
        dag_r2(M, T);
    } else {
        src_link2(pc, h[0].which, h[0].a, h[0].b, pt, T, kj);
    }
    k = kj;
#pragma unroll
    for (int j = 1; j < N; j++) {
        src_link(pc, h[j].which, h[j].a, h[j].b, pt, M, kj);
        if (h[j].dag) mul_dag_r2(T, M, T); else mul_r2(T, M, T);
        k *= kj;
    }
    rebuild3row(T);
}
// sl[e kGfLinks] (e = 2 (3 r + c) + re/im) += s T: a thread's staple sum in its
// own LDS slots, which keeps 36 registers free for the product chains
constexpr int kGfLinks = 64;
__device__ __forceinline__ void lds_axpy(double s, const Su3& T, double* sl) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const int e = 2 * (3 * r + c);
            sl[e * kGfLinks] = fma(s, T.c[r][c].x, sl[e * kGfLinks]);
            sl[(e + 1) * kGfLinks] = fma(s, T.c[r][c].y, sl[(e + 1) * kGfLinks]);
        }
}
// acc += s T (all rows)
__device__ __forceinline__ void axpy3(double s, const Su3& T, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            acc.c[r][c] = make_double2(fma(s, T.c[r][c].x, acc.c[r][c].x), fma(s, T.c[r][c].y, acc.c[r][c].y));
}

// The staple terms of link (x, mu) on one side of the plane (mu, nu): the
// plaquette a m n and the rectangles of types A, B, C on that side
// (plaquettes.c:83-195, rectangles.c:691-718, 780-807, 865-892), each
// times C_ZERO or C_ONE and the K of its links.  On the upper side
//   a = U_nu(x+mu), m = U_mu(x+nu)^+, n = U_nu(x)^+,
//   A = a Q0 n, B = Q2 m n, C = a m Q4 with
//   Q0 = U_nu(x+mu+nu) U_mu(x+2nu)^+ U_nu(x+nu)^+,
//   Q2 = U_mu(x+mu) U_nu(x+2mu) U_mu(x+mu+nu)^+,
//   Q4 = U_mu(x-mu+nu)^+ U_nu(x-mu)^+ U_mu(x-mu),
// and the lower side is its mirror in nu (a = U_nu(x+mu-nu)^+,
// m = U_mu(x-nu)^+, n = U_nu(x-nu)).  The four terms share factors:
//   (c0 a m + c1 a Q0 + c1 Q2 m) n + c1 (a m) Q4,
// 14 link loads and 207 complex multiply-adds instead of 18 and 252 for
// the terms taken one by one; the sum is the same up to rounding.
// c_side[side] = {a, m, n, Q0[3], Q2[3], Q4[3]}
__device__ __constant__ HopD c_side[2][12] = {
    {{1, 1, 0, 0}, {0, 0, 1, 1}, {1, 0, 0, 1},
     {1, 1, 1, 0}, {0, 0, 2, 1}, {1, 0, 1, 1},
     {0, 1, 0, 0}, {1, 2, 0, 0}, {0, 1, 1, 1},
     {0, -1, 1, 1}, {1, -1, 0, 1}, {0, -1, 0, 0}},
    {{1, 1, -1, 1}, {0, 0, -1, 1}, {1, 0, -1, 0},
     {1, 1, -2, 1}, {0, 0, -2, 1}, {1, 0, -2, 0},
     {0, 1, 0, 0}, {1, 2, -1, 1}, {0, 1, -1, 1},
     {0, -1, -1, 1}, {1, -1, -1, 0}, {0, -1, 0, 0}},
};

// one side (c_side[side]) of the plane's staple terms; add(s, T) receives
// each product to be summed with its coefficient
template <class Src, class Add>
__device__ __forceinline__ void plane_side(const Src& pc, const HopD* d, int pt, int tlsm, double c0, Add add) {
    Su3 G, T;
    double k;
    su3_zero(G);
    {
        // a m: into G with c0, and with Q4 into S
        Su3 am;
        double k_am;
        const HopD h[2] = {d[0], d[1]};
        chain(pc, h, pt, am, k_am);
        axpy3(c0 * k_am, am, G);
        if (tlsm) {
            const HopD h4[3] = {d[9], d[10], d[11]};
            chain(pc, h4, pt, T, k);
            Su3 X;
            mul_r2(am, T, X);
            rebuild3row(X);
            add(kCOne * k_am * k, X);
        }
    }
    if (tlsm) {
        const HopD h0[4] = {d[0], d[3], d[4], d[5]};
        chain(pc, h0, pt, T, k);
        axpy3(kCOne * k, T, G);
        const HopD h2[4] = {d[6], d[7], d[8], d[1]};
        chain(pc, h2, pt, T, k);
        axpy3(kCOne * k, T, G);
    }
    // (...) n
    Su3 n;
    double kn;
    src_link(pc, d[2].which, d[2].a, d[2].b, pt, T, kn);
    if (d[2].dag) {
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) n.c[r][c] = cconj(T.c[c][r]);
    } else {
        n = T;
    }
    su3_mul(G, n, T);
    add(kn, T);
}

__device__ __forceinline__ void plane_staple(const PlaneCtx& pc, int pt, int tlsm, double c0, double* sl) {
#pragma unroll 1
    for (int side = 0; side < 2; side++)
        plane_side(pc, c_side[side], pt, tlsm, c0, [&](double s, const Su3& T) { lds_axpy(s, T, sl); });
}

// Gauge force, one thread per (link, plane): a block is three waves over the
// same 64 links, wave w summing the staple terms of plane nu = perp(mu)[w].
// Each wave forms TA(U S_w) (TA is linear, so the planes' parts add up to
// TA(U S)); the three parts (and, when requested, the staples) are summed
// through LDS in plane order and multiplied by K_mu(x).  Wave 0 then writes
// ipdot and, with mom, the momentum step of mom_sum_mult
// (su3_utilities.h:1383-1394).
__global__ __launch_bounds__(3 * kGfLinks, 2) void k_gauge_force(GaugePtrs G, double2* __restrict__ stap,
                                                             size_t su3_stride, void* __restrict__ ipdot, LinkGeom g,
                                                             int pt, int tlsm, double c0, void* __restrict__ mom,
                                                             double fact) {
    __shared__ double red[3][18][kGfLinks];
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // A block covers 64 half-sites of one link array (dir uniform).  Logical
    // blocks run over the link array fastest, then t, then the 64-site tile
    // of the t-slice, and each XCD takes a contiguous range of them: an XCD
    // owns a slab of tiles for every t and every link array, and the blocks
    // it runs together cover one tile at neighbouring t, so the neighbour
    // links of a staple are re-read from its L2 (with each XCD sweeping the
    // whole lattice for one link array, every XCD fetched every neighbour
    // link from memory: 22 GB per launch at 48^3x12).  A t-slice that is not
    // a whole number of tiles keeps the plain half-site order.
    const int blk = xcd_block_id();
    const int dir = __builtin_amdgcn_readfirstlane(blk & 7);
    const int rest = blk >> 3;
    const int s3 = g.sizeh / g.nd[3];
    int idxh;
    if (s3 % kGfLinks == 0) {
        const int tile = rest / g.nd[3], tt = rest - tile * g.nd[3];
        idxh = tt * s3 + tile * kGfLinks + lane;
    } else {
        idxh = rest * kGfLinks + lane;
    }
    const bool live = idxh < g.sizeh;
    const int mu = dir >> 1;
    double* sl = &red[w][0][lane];
#pragma unroll
    for (int e = 0; e < 18; e++) sl[e * kGfLinks] = 0.0;
    Tamat q = {};
    if (live) {
        int x[4];
        decode(idxh, dir & 1, g, x);
        PlaneCtx pc;
        pc.base = G.base;
        pc.stride = G.stride;
        pc.plane = 16u * (unsigned)g.sizeh;
        pc.mu = mu;
        pc.nu = __builtin_amdgcn_readfirstlane(c_perp[mu][w]);
        pc.p = dir & 1;
        const int st[4] = {1, g.nd[0], g.nd[0] * g.nd[1], g.nd[0] * g.nd[1] * g.nd[2]};
        auto sel = [](const int* v, int i) { return i == 0 ? v[0] : i == 1 ? v[1] : i == 2 ? v[2] : v[3]; };
        pc.sm = sel(st, pc.mu);
        pc.sn = sel(st, pc.nu);
        pc.ndm = sel(g.nd, pc.mu);
        pc.ndn = sel(g.nd, pc.nu);
        pc.lex = x[0] + st[1] * x[1] + st[2] * x[2] + st[3] * x[3];
        pc.xm = sel(x, pc.mu);
        pc.xn = sel(x, pc.nu);
        plane_staple(pc, pt, tlsm, c0, sl);
        Su3 S, U, X;
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++)
                S.c[r][c] = make_double2(sl[2 * (3 * r + c) * kGfLinks], sl[(2 * (3 * r + c) + 1) * kGfLinks]);
        double k;
        pc_link(pc, 0, 0, 0, pt, U, k);
        su3_mul(U, S, X);
        ta_part(X, 1.0, q);
    }
    const double kmu = (live && pt) ? ((const double*)(G.at(dir) + 9 * (size_t)g.sizeh))[idxh] : 1.0;
    if (stap) {
        // the three planes' staple sums are in red
        __syncthreads();
        if (w == 0 && live) {
            double2* O = (double2*)((char*)stap + dir * su3_stride);
#pragma unroll
            for (int e = 0; e < 9; e++) {
                const double re = kmu * (red[0][2 * e][lane] + red[1][2 * e][lane] + red[2][2 * e][lane]);
                const double im = kmu * (red[0][2 * e + 1][lane] + red[1][2 * e + 1][lane] + red[2][2 * e + 1][lane]);
                O[(size_t)e * g.sizeh + idxh] = make_double2(re, im);
            }
        }
    }
    __syncthreads();
    red[w][0][lane] = q.c01.x;
    red[w][1][lane] = q.c01.y;
    red[w][2][lane] = q.c02.x;
    red[w][3][lane] = q.c02.y;
    red[w][4][lane] = q.c12.x;
    red[w][5][lane] = q.c12.y;
    red[w][6][lane] = q.ic00;
    red[w][7][lane] = q.ic11;
    __syncthreads();
    if (w == 0 && live) {
        double t[8];
#pragma unroll
        for (int j = 0; j < 8; j++) t[j] = kmu * (red[0][j][lane] + red[1][j][lane] + red[2][j][lane]);
        Tamat o;
        o.c01 = make_double2(t[0], t[1]);
        o.c02 = make_double2(t[2], t[3]);
        o.c12 = make_double2(t[4], t[5]);
        o.ic00 = t[6];
        o.ic11 = t[7];
        ta_store(ipdot, dir, g.sizeh, idxh, o);
        if (mom) mom_step(mom, dir, g.sizeh, idxh, o, fact);
    }
}

// Gauge force by planes, for the action with rectangles (gf_planes_pay says
// where).  TA(U S) is linear, so every plane (mu, nu) forms its own part
// TA(U S_plane) of its two directions' links, in a buffer of its own (three
// planes per direction), and the kernels that consume the force add the three
// parts.
//
// A block takes tm x tn tiles (at most 64 sites, one lane each) of a plane at
// fixed coordinates along the other two directions.  Within a tile every
// product that several links need is formed once, in LDS.  With M = U_mu and
// N = U_nu:
//   corners            Cm(y) = M(y) N(y+mu),             Cn(y) = N(y) M(y+nu)
//   plaquette staples  SM+(y) = N(y+mu) Cn(y)^+,         SM-(y) = Cm(y-nu)^+ N(y-nu)     (of M)
//                      SN+(y) = M(y+nu) Cm(y)^+,         SN-(y) = Cn(y-mu)^+ M(y-mu)     (of N)
// A rectangle's staple is a plaquette staple with one link replaced by that
// link's own plaquette staple on the far side, so one side of a link O
// (direction o, the plane's other direction p, links P) is four products:
//   up:   (c0 P(x+o) + c1 SP+(x+o)^+) Cp(x)^+ + c1 P(x+o) [SO+(x+p) P(x)^+ + O(x+p)^+ SP-(x)]
//   down: Co(x-p)^+ (c0 P(x-p) + c1 SP-(x-p)^+) + c1 [P(x+o-p)^+ SO-(x-p) + SP+(x+o-p) O(x-p)^+] P(x-p)
// A wave takes one side of one direction's links (its roles, and so the
// arrays, are wave-uniform).
//
// The links come from a copy in records (rows 0,1 of a link, 96 B), so that a
// tile's loads use whole sectors in every plane: with the field's colour
// planes, a plane without direction 0 fetches a 128-B line per 16-B entry
// (67 M requests per plane at 48^3x12, 12 TB/s from the L2).  The blocks are
// persistent and hold the next tile's links in registers while they work on
// the current one.
//
// Bound by FP64 issue and the latency between a tile's phases: 1116 vector
// instructions a wave and tile (1551 with every operand's address formed from
// the plan, 2900 for the term-by-term sides), 52% of the issue slots at the
// 2.1 GHz the card holds; LDS and two blocks per CU leave two waves per SIMD.
// 48^3x12: 1.85 ms per force, 2.4 ms with the records' and the force's passes
// (term-by-term sides, six launches: 3.1 ms); gauge sub-integrator, whose last
// force goes by links, 39.0 -> 27.8 ms.  Tried and slower: summing the sides of both directions in two waves
// that the second staple pass spares (more exchange through LDS, 2.0 ms).
// Entry e (of six: rows 0, 1) of the LDS arrays' record r is pool[e kGfPool +
// r]: an operand's six reads share one address with constant offsets, and
// sixteen lanes on consecutive sites read all 64 banks once, so that tiles
// with rows of 16 sites meet no bank conflicts (records of 96 B: 2.2 times the
// LDS cycles).
struct GfArr {
    int off, n, rw, org;  // record of site (i, j): off + j rw + i - org
    int inv;              // 65536 / rw, rounded up: q / rw = q inv >> 16 for q < 512
};
enum GfRole : int { gM = 0, gN, gCm, gCn, gSMp, gSMm, gSNp, gSNm, gRoles };
struct GfPlan {
    int mu, nu, tm, tn, tiles_m, tiles_n, tiles, inv_tm;
    GfArr a[gRoles];
};
struct GfPlans {
    int tiles[8];  // of each plane (p[k].tiles)
    GfPlan p[6];
};
// records and K values of the largest tile (16 x 4): 81,632 B with K, so that two blocks fit a CU
constexpr int kGfPool = 826;
constexpr int kGfPoolLinks = 292;
constexpr int kGfFetch = 4;  // links per thread: 85 triples of lanes, two 16-B entries a lane
// part of plane (d, other) in direction d's three buffers
__device__ __forceinline__ int gf_slot(int d, int other) { return other - (other > d ? 1 : 0); }

__device__ __forceinline__ int sel4(int k, int v0, int v1, int v2, int v3) {
    return k == 0 ? v0 : k == 1 ? v1 : k == 2 ? v2 : v3;
}
// rows 0,1 (gf_load2) or all rows (gf_load) of a record in LDS
__device__ __forceinline__ void gf_load2(const double2* e, Su3& m) {
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) m.c[r][c] = e[(3 * r + c) * kGfPool];
}
__device__ __forceinline__ void gf_load(const double2* e, Su3& m) {
    gf_load2(e, m);
    rebuild3row(m);
}
__device__ __forceinline__ void gf_store2(double2* e, const Su3& m) {
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) e[(3 * r + c) * kGfPool] = m.c[r][c];
}
// acc = s m, acc += s m^+
__device__ __forceinline__ void su3_scale(double s, const Su3& m, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) acc.c[r][c] = cscale(m.c[r][c], s);
}
__device__ __forceinline__ void axpy3_dag(double s, const Su3& m, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            acc.c[r][c] = make_double2(fma(s, m.c[c][r].x, acc.c[r][c].x), fma(-s, m.c[c][r].y, acc.c[r][c].y));
}
// acc += a b ; a b^+ ; a^+ b
__device__ __forceinline__ void su3_mul_add(const Su3& a, const Su3& b, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            acc.c[r][c] = cfma(a.c[r][2], b.c[2][c], cfma(a.c[r][1], b.c[1][c], cfma(a.c[r][0], b.c[0][c], acc.c[r][c])));
}
__device__ __forceinline__ void su3_mul_dag_add(const Su3& a, const Su3& b, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            acc.c[r][c] = cfma(a.c[r][2], cconj(b.c[c][2]),
                               cfma(a.c[r][1], cconj(b.c[c][1]), cfma(a.c[r][0], cconj(b.c[c][0]), acc.c[r][c])));
}
__device__ __forceinline__ void su3_dag_mul_add(const Su3& a, const Su3& b, Su3& acc) {
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            acc.c[r][c] = cfmac(a.c[2][r], b.c[2][c], cfmac(a.c[1][r], b.c[1][c], cfmac(a.c[0][r], b.c[0][c], acc.c[r][c])));
}

// A plan's numbers in scalar registers.  The readfirstlane keeps the compiler
// from turning a per-lane choice between two of them into a per-lane load
// from the kernel arguments, a memory round trip each (3.3 -> 2.6 ms per force
// at 48^3x12).
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ GfArr uni(const GfArr& a) {
    return GfArr{uni(a.off), uni(a.n), uni(a.rw), uni(a.org), uni(a.inv)};
}
// The force parts of one plane (mu, nu) are records of four 16-B entries (c01,
// c02, c12, (ic00, ic11)) at part[((slot 8 + link array) sizeh + site) 4].
template <bool PT>
__global__ __launch_bounds__(256, 2) void k_gf_tile(const double2* __restrict__ rec, GaugePtrs G,
                                                    double2* __restrict__ part, LinkGeom g, GfPlans plans, double c0) {
    __shared__ double2 pool[6 * kGfPool];
    __shared__ double lk[PT ? kGfPoolLinks : 1];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int w = uni(tid >> 6), dsel = w >> 1, side = w & 1;
    const int nd0 = g.nd[0], nd1 = g.nd[1], nd2 = g.nd[2], nd3 = g.nd[3];
    const int st1 = nd0, st2 = nd0 * nd1, st3 = st2 * nd2;
    const unsigned rec_stride = 96u * (unsigned)g.sizeh;
    // Every XCD takes a contiguous eighth of each plane's tiles, and each of its
    // blocks (hardware ids round-robin over the XCDs) a contiguous run of those:
    // a block sets a plane up once and re-reads its tiles' halos from the L2.
    const int xcd = (int)blockIdx.x & 7, nbx = ((int)gridDim.x - xcd + 7) >> 3, bx = (int)blockIdx.x >> 3;
    auto share = [](int tiles, int x) { return (tiles >> 3) * x + ((tiles & 7) * x >> 3); };
    int total = 0;
#pragma unroll
    for (int p = 0; p < 6; p++) total += share(plans.tiles[p], xcd + 1) - share(plans.tiles[p], xcd);
    const int each = total / nbx, rest = total - each * nbx;
    int q = each * bx + min(bx, rest), left = each + (bx < rest ? 1 : 0);
    for (int p = 0; p < 6 && left > 0; p++) {
        const GfPlan& pl = plans.p[p];
        const int tiles = uni(pl.tiles), base = share(tiles, xcd), count = share(tiles, xcd + 1) - base;
        if (q >= count) {
            q -= count;
            continue;
        }
        const int end = min(count, q + left);  // this plane's tiles [q, end)
        left -= end - q;
        const int mu = uni(pl.mu), nu = uni(pl.nu), TM = uni(pl.tm), TN = uni(pl.tn);
        const int tiles_m = uni(pl.tiles_m), tiles_n = uni(pl.tiles_n);
        const int oa = (mu != 0 && nu != 0) ? 0 : ((mu != 1 && nu != 1) ? 1 : 2), ob = 6 - mu - nu - oa;
        const int nda = sel4(oa, nd0, nd1, nd2, nd3), ndm = sel4(mu, nd0, nd1, nd2, nd3), ndn = sel4(nu, nd0, nd1, nd2, nd3);
        const int sa = sel4(oa, 1, st1, st2, st3), sb = sel4(ob, 1, st1, st2, st3);
        const int sm = sel4(mu, 1, st1, st2, st3), sn = sel4(nu, 1, st1, st2, st3);
        const GfArr M = uni(pl.a[gM]), N = uni(pl.a[gN]), Cm = uni(pl.a[gCm]), Cn = uni(pl.a[gCn]);
        const GfArr SMp = uni(pl.a[gSMp]), SMm = uni(pl.a[gSMm]), SNp = uni(pl.a[gSNp]), SNm = uni(pl.a[gSNm]);
        const int nL = M.n + N.n;

        // What depends on the plane alone: this thread's links of the tile and
        // its halo, and the records (pool indices) of its corner and staples.
        int li[kGfFetch];  // i, j (+2) and direction of the link
        auto link_pos = [&](int s) {
            const bool d = s >= M.n;
            const int r = d ? s - M.n : s;
            const int j = (r * (d ? N.inv : M.inv)) >> 16, i = r - j * (d ? N.rw : M.rw);
            return i | j << 8 | (d ? 1 << 16 : 0);
        };
        const int ltri = tid / 3, lpart = 2 * (tid - 3 * ltri);
#pragma unroll
        for (int k = 0; k < kGfFetch; k++) li[k] = link_pos(min(ltri + 85 * k, nL - 1));
        int cA, cB, cO;
        {
            const int s = min(tid, Cm.n + Cn.n - 1);
            const bool d = s >= Cm.n;
            const int r = d ? s - Cm.n : s;
            const int jj = (r * Cm.inv) >> 16, ii = r - jj * Cm.rw;  // Cn has Cm's shape
            const int i = ii - (d ? 2 : 1), j = jj - (d ? 1 : 2);
            const int rM = M.off + (j + (d ? 1 : 0)) * M.rw + i - M.org, rN = N.off + j * N.rw + i + (d ? 0 : 1) - N.org;
            cA = (d ? rN : rM);
            cB = (d ? rM : rN);
            cO = ((d ? Cn.off : Cm.off) + r);
        }
        // staples: link x corner^+ (SM+, SN+) first, then corner^+ x link (SM-, SN-) from a whole wave on
        const int np = SMp.n + SNp.n, p64 = (np + 63) & ~63, ns = p64 + SMm.n + SNm.n;
        int sA[2], sC[2], sO[2];
        auto item = [&](int k) { return tid + 256 * k; };
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int s = item(k);
            if (s < p64) {
                const int e = min(s, np - 1);
                const bool d = e >= SMp.n;
                const int r = d ? e - SMp.n : e;
                const int jj = (r * (d ? SNp.inv : SMp.inv)) >> 16, ii = r - jj * (d ? SNp.rw : SMp.rw);
                const int i = ii + (d ? 1 : -1), j = jj + (d ? -1 : 1);
                sA[k] = (d ? M.off + (j + 1) * M.rw + i - M.org : N.off + j * N.rw + i + 1 - N.org);
                sC[k] = (d ? Cm.off + j * Cm.rw + i - Cm.org : Cn.off + j * Cn.rw + i - Cn.org);
                sO[k] = ((d ? SNp.off : SMp.off) + r);
            } else {
                const int e = min(s, ns - 1) - p64;
                const bool d = e >= SMm.n;
                const int r = d ? e - SMm.n : e;
                const int jj = (r * SMm.inv) >> 16, ii = r - jj * SMm.rw;  // SN- has SM-'s shape
                const int i = ii - 1 - (d ? 1 : 0), j = jj - 1 - (d ? 0 : 1);  // the plaquette's own site
                sA[k] = (d ? M.off + j * M.rw + i - M.org : N.off + j * N.rw + i - N.org);
                sC[k] = (d ? Cn.off + j * Cn.rw + i - Cn.org : Cm.off + j * Cm.rw + i - Cm.org);
                sO[k] = ((d ? SNm.off : SMm.off) + r);
            }
        }
        const int inv_tm = uni(pl.inv_tm);
        const int jn = (lane * inv_tm) >> 16, im = lane - jn * TM;
        const bool inside = lane < TM * TN;

        // tile r of the plane: its corner (om, on) and the sites' constant part.
        // Consecutive tiles are neighbours along mu, then nu; in a plane without
        // direction 0 the tiles of consecutive x, which share the records' lines,
        // follow each other.
        struct Tile {
            int om, on, xa, xb;
        };
        auto place = [&](int r) {
            int tm, tn, xa, xb;
            if (mu == 0) {
                tm = r % tiles_m;
                r /= tiles_m;
                tn = r % tiles_n;
                r /= tiles_n;
                xa = r % nda;
                xb = r / nda;
            } else {
                xa = r % nda;
                r /= nda;
                tm = r % tiles_m;
                r /= tiles_m;
                tn = r % tiles_n;
                xb = r / tiles_n;
            }
            return Tile{tm * TM, tn * TN, xa, xb};
        };
        auto advance = [&](Tile t) {  // the tile after t
            auto up = [](int& v, int step, int n) {
                v += step;
                if (v < n) return false;
                v = 0;
                return true;
            };
            if (mu == 0) {
                if (up(t.om, TM, ndm) && up(t.on, TN, ndn) && up(t.xa, 1, nda)) t.xb++;
            } else {
                if (up(t.xa, 1, nda) && up(t.om, TM, ndm) && up(t.on, TN, ndn)) t.xb++;
            }
            return t;
        };
        // link array (0..7) and half-site of a link; a tile that reaches past the lattice's end wraps (its
        // lanes there write nothing).  The unsigned minimum picks the wrapped coordinate.
        auto link_at = [&](const Tile& t, int l, int& arr, int& h) {
            unsigned ym = (unsigned)(t.om - 2 + (l & 255)), yn = (unsigned)(t.on - 2 + ((l >> 8) & 255));
            ym = min(ym, ym + (unsigned)ndm);
            ym = min(ym, ym - (unsigned)ndm);
            yn = min(yn, yn + (unsigned)ndn);
            yn = min(yn, yn - (unsigned)ndn);
            arr = 2 * (l >> 16 ? nu : mu) + (int)((unsigned)(t.xa + t.xb) + ym + yn & 1u);
            h = (int)((unsigned)(t.xa * sa + t.xb * sb) + __umul24(ym, sm) + __umul24(yn, sn)) >> 1;
        };
        ostp_dvec2 pre[2 * kGfFetch];
        double prek[kGfFetch];
        auto fetch = [&](const Tile& t) {
#pragma unroll
            for (int k = 0; k < kGfFetch; k++) {
                int arr, h;
                link_at(t, li[k], arr, h);
                const ostp_dvec2* R = (const ostp_dvec2*)((const char*)rec + (size_t)((unsigned)arr) * rec_stride +
                                                          link_record(h, lpart));
                pre[2 * k] = R[0];
                pre[2 * k + 1] = R[1];
                if (PT) prek[k] = ((const double*)(G.at(arr) + (size_t)9 * g.sizeh))[h];
            }
        };
        Tile t = place(base + q);
        fetch(t);
        for (;;) {
#pragma unroll
            for (int k = 0; k < kGfFetch; k++)
                if (tid < 255 && ltri + 85 * k < nL) {
                    ostp_dvec2* e = (ostp_dvec2*)(pool + lpart * kGfPool + ltri + 85 * k);
                    e[0] = pre[2 * k];
                    e[kGfPool] = pre[2 * k + 1];
                    if (PT && lpart == 0) lk[ltri + 85 * k] = prek[k];
                }
            __syncthreads();
            if (tid < Cm.n + Cn.n) {
                Su3 A, B;
                gf_load2(pool + cA, A);
                gf_load(pool + cB, B);
                mul_r2(A, B, A);
                gf_store2(pool + cO, A);
            }
            __syncthreads();
            // the next tile's links, while this one is worked on
            const bool more = q + 1 < end;
            Tile tn = t;
            if (more) {
                tn = advance(t);
                fetch(tn);
            }
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int s = item(k);
                if (s < np) {
                    Su3 A, C;
                    gf_load2(pool + sA[k], A);
                    gf_load(pool + sC[k], C);
                    mul_dag_r2(A, C, A);
                    gf_store2(pool + sO[k], A);
                } else if (s >= p64 && s < ns) {
                    Su3 A, C, X;
                    gf_load(pool + sA[k], A);
                    gf_load(pool + sC[k], C);
                    dag_mul_r2(C, A, X);
                    gf_store2(pool + sO[k], X);
                }
            }
            __syncthreads();
            // one side of one direction's links per wave
            const bool live = inside && t.om + im < ndm && t.on + jn < ndn;
            auto pick = [&](const GfArr& a, const GfArr& b) {  // dsel ? b : a, in scalar registers
                return GfArr{uni(dsel ? b.off : a.off), 0, uni(dsel ? b.rw : a.rw), uni(dsel ? b.org : a.org), 0};
            };
            const GfArr aO = pick(M, N), aP = pick(N, M);
            const GfArr aC = side ? pick(Cm, Cn) : pick(Cn, Cm);  // Co down, Cp up
            const GfArr aSO = side ? pick(SMm, SNm) : pick(SMp, SNp), aSPp = pick(SNp, SMp), aSPm = pick(SNm, SMm);
            // record of x + do e_o + dp e_p
            auto at = [&](const GfArr& a, int dO, int dP) {
                const int di = dsel ? dP : dO, dj = dsel ? dO : dP;
                return (jn * a.rw + im) + (a.off + dj * a.rw + di - a.org);
            };
            auto ld = [&](const GfArr& a, int dO, int dP, Su3& m) { gf_load(pool + at(a, dO, dP), m); };
            auto ld2 = [&](const GfArr& a, int dO, int dP, Su3& m) { gf_load2(pool + at(a, dO, dP), m); };
            auto kO = [&](int dO, int dP) { return PT ? lk[at(aO, dO, dP)] : 1.0; };
            auto kP = [&](int dO, int dP) { return PT ? lk[at(aP, dO, dP)] : 1.0; };
            Su3 T;
            if (live) {
                Su3 A, B;
                if (side == 0) {
                    const double ka = kP(1, 0), kc = kP(0, 0) * kO(0, 1);
                    ld(aP, 1, 0, A);
                    Su3 X, W;
                    ld2(aSO, 0, 1, X);
                    ld(aP, 0, 0, B);
                    mul_dag_r2(X, B, X);
                    rebuild3row(X);
                    su3_scale(kCOne * ka * kP(1, 1) * kO(0, 2) * kP(0, 1) * kP(0, 0), X, W);
                    ld(aO, 0, 1, B);
                    Su3 Y;
                    ld(aSPm, 0, 0, Y);
                    dag_mul_r2(B, Y, X);
                    rebuild3row(X);
                    axpy3(kCOne * ka * kO(0, 1) * kP(-1, 0) * kO(-1, 1) * kO(-1, 0), X, W);
                    su3_mul(A, W, T);
                    su3_scale(c0 * ka * kc, A, A);
                    ld(aSPp, 1, 0, B);
                    axpy3_dag(kCOne * kc * kO(1, 1) * kP(2, 0) * kO(1, 0), B, A);
                    ld(aC, 0, 0, B);
                    su3_mul_dag_add(A, B, T);
                } else {
                    const double kn = kP(0, -1), kc = kO(0, -1) * kP(1, -1);
                    ld(aP, 0, -1, A);
                    Su3 X, Y, W;
                    ld(aP, 1, -1, B);
                    ld(aSO, 0, -1, Y);
                    dag_mul_r2(B, Y, X);
                    rebuild3row(X);
                    su3_scale(kCOne * kn * kP(1, -1) * kP(1, -2) * kO(0, -2) * kP(0, -2), X, W);
                    ld2(aSPp, 1, -1, X);
                    ld(aO, 0, -1, B);
                    mul_dag_r2(X, B, X);
                    rebuild3row(X);
                    axpy3(kCOne * kn * kO(0, -1) * kO(1, 0) * kP(2, -1) * kO(1, -1), X, W);
                    su3_mul(W, A, T);
                    su3_scale(c0 * kc * kn, A, A);
                    ld(aSPm, 0, -1, B);
                    axpy3_dag(kCOne * kc * kP(-1, -1) * kO(-1, 0) * kO(-1, -1), B, A);
                    ld(aC, 0, -1, B);
                    su3_dag_mul_add(B, A, T);
                }
            }
            // the lower sides' sums go to the upper sides' threads through the pool past the links
            // (entries 0-5 of the first 128 records, 0-2 of the next)
            double2* xch = pool + nL + dsel * 64 + lane;
            auto xe = [&](int e) -> double2& { return xch[e < 6 ? e * kGfPool : (e - 6) * kGfPool + 128]; };
            __syncthreads();
            if (side == 1 && live) {
#pragma unroll
                for (int e = 0; e < 9; e++) xe(e) = T.c[e / 3][e % 3];
            }
            __syncthreads();
            double2* out = pool + nL + 256;  // force records of the tile's 2 x 64 links
            auto site = [&](int i, int j, int d, int& arr, int& h) {
                const int ym = t.om + i, yn = t.on + j;
                arr = 2 * (d ? nu : mu) + ((t.xa + t.xb + ym + yn) & 1);
                h = (t.xa * sa + t.xb * sb + ym * sm + yn * sn) >> 1;
            };
            if (side == 0 && live) {
#pragma unroll
                for (int e = 0; e < 9; e++) T.c[e / 3][e % 3] = cadd(T.c[e / 3][e % 3], xe(e));
                Su3 U, X;
                ld(aO, 0, 0, U);
                const double ku = kO(0, 0);
                su3_mul(U, T, X);
                Tamat f;
                ta_part(X, ku, f);
                double2* o = out + dsel * 64 + lane;
                o[0] = f.c01;
                o[kGfPool] = f.c02;
                o[2 * kGfPool] = f.c12;
                o[3 * kGfPool] = make_double2(f.ic00, f.ic11);
            }
            __syncthreads();
            // four lanes write one link's 64-B record
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int l = tid >> 2;
                const int j = (l * inv_tm) >> 16, i = l - j * TM;
                if (l < TM * TN && t.om + i < ndm && t.on + j < ndn) {
                    int arr, h;
                    site(i, j, k, arr, h);
                    const int slot = gf_slot(k ? nu : mu, k ? mu : nu);
                    part[((size_t)(slot * 8 + arr) * g.sizeh + h) * 4 + (tid & 3)] = out[(tid & 3) * kGfPool + 64 * k + l];
                }
            }
            if (!more) break;
            q++;
            t = tn;
        }
        q = 0;
    }
}

// records of a block's links through LDS: the field's colour planes and the
// force parts on one side, whole records with consecutive lanes on the other
struct GfRecs {
    double2 u[6 * kBlock];
};
// rows 0,1 of every link into records
__global__ __launch_bounds__(kBlock) void k_gf_pack(GaugePtrs G, double2* __restrict__ rec, int sizeh) {
    __shared__ GfRecs s;
    const int l = (int)blockIdx.y, i0 = (int)blockIdx.x * kBlock, t = (int)threadIdx.x;
    const int n = sizeh - i0 < kBlock ? sizeh - i0 : kBlock;
    const double2* U = G.at(l) + i0;
    if (t < n)
#pragma unroll
        for (int k = 0; k < 6; k++) s.u[6 * t + k] = U[(size_t)k * sizeh + t];
    __syncthreads();
    double2* R = rec + ((size_t)l * sizeh + i0) * 6;
#pragma unroll
    for (int k = 0; k < 6; k++)
        if (t + k * kBlock < 6 * n) R[t + k * kBlock] = s.u[t + k * kBlock];
}
// and back
__global__ __launch_bounds__(kBlock) void k_gf_unpack(const double2* __restrict__ rec, GaugePtrs G, int sizeh) {
    __shared__ GfRecs s;
    const int l = (int)blockIdx.y, i0 = (int)blockIdx.x * kBlock, t = (int)threadIdx.x;
    const int n = sizeh - i0 < kBlock ? sizeh - i0 : kBlock;
    const double2* R = rec + ((size_t)l * sizeh + i0) * 6;
#pragma unroll
    for (int k = 0; k < 6; k++)
        if (t + k * kBlock < 6 * n) s.u[t + k * kBlock] = R[t + k * kBlock];
    __syncthreads();
    double2* U = const_cast<double2*>(G.at(l)) + i0;
    if (t < n)
#pragma unroll
        for (int k = 0; k < 6; k++) U[(size_t)k * sizeh + t] = s.u[6 * t + k];
}

// sum of the three planes' parts of the block's links, a link per thread, through the block's LDS
__device__ __forceinline__ void gf_parts_sum(const double2* __restrict__ part, int sizeh, int l, int i0, int n,
                                             double2* lds, Tamat& q) {
    const int t = (int)threadIdx.x;
    const size_t s8 = (size_t)8 * sizeh * 4;
    const double2* P = part + ((size_t)l * sizeh + i0) * 4;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int c = t + k * kBlock;
        if (c < 4 * n) lds[c] = cadd(cadd(P[c], P[s8 + c]), P[2 * s8 + c]);
    }
    __syncthreads();
    if (t < n) {
        q.c01 = lds[4 * t];
        q.c02 = lds[4 * t + 1];
        q.c12 = lds[4 * t + 2];
        q.ic00 = lds[4 * t + 3].x;
        q.ic11 = lds[4 * t + 3].y;
    }
}

// ipdot = sum of the planes' parts; with mom, the momentum step of mom_sum_mult (su3_utilities.h:1383-1394)
__global__ __launch_bounds__(kBlock) void k_gf_ipdot(const double2* __restrict__ part, void* __restrict__ ipdot,
                                                     void* __restrict__ mom, int sizeh, double fact) {
    __shared__ double2 lds[4 * kBlock];
    const int l = (int)blockIdx.y, i0 = (int)blockIdx.x * kBlock, t = (int)threadIdx.x;
    const int n = sizeh - i0 < kBlock ? sizeh - i0 : kBlock;
    Tamat q;
    gf_parts_sum(part, sizeh, l, i0, n, lds, q);
    if (t >= n) return;
    ta_store(ipdot, l, sizeh, i0 + t, q);
    if (mom) mom_step(mom, l, sizeh, i0 + t, q, fact);
}

// momentum step with the sum of the planes' parts, then U <- exp(i delta P) U
// on the records.  Memory-bound (512 B per link); every load is issued before
// the first wait.
__global__ __launch_bounds__(kBlock) void k_gf_move(const double2* __restrict__ part, void* __restrict__ mom,
                                                    double2* __restrict__ rec, int sizeh, double fact, double delta) {
    __shared__ GfRecs s;
    __shared__ double2 lds[4 * kBlock];
    const int l = (int)blockIdx.y, i0 = (int)blockIdx.x * kBlock, t = (int)threadIdx.x;
    const int n = sizeh - i0 < kBlock ? sizeh - i0 : kBlock;
    double2* R = rec + ((size_t)l * sizeh + i0) * 6;
    ostp_dvec2 u6[6];
    Thmat h;
#pragma unroll
    for (int k = 0; k < 6; k++) u6[k] = *(const ostp_dvec2*)(R + min(t + k * kBlock, 6 * n - 1));
    th_load(mom, l, sizeh, i0 + min(t, n - 1), h);
    Tamat q;
    gf_parts_sum(part, sizeh, l, i0, n, lds, q);
#pragma unroll
    for (int k = 0; k < 6; k++) *(ostp_dvec2*)(s.u + t + k * kBlock) = u6[k];
    Su3 E;
    if (t < n) {
        th_step(h, q, fact);
        th_store(mom, l, sizeh, i0 + t, h);
        exp_ip(h, delta, E);
    }
    __syncthreads();
    if (t < n) {
        double2 u[2][3];
#pragma unroll
        for (int e = 0; e < 6; e++) u[e / 3][e % 3] = s.u[6 * t + e];
        move_link(E, u);
#pragma unroll
        for (int e = 0; e < 6; e++) s.u[6 * t + e] = u[e / 3][e % 3];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 6; k++)
        if (t + k * kBlock < 6 * n) R[t + k * kBlock] = s.u[t + k * kBlock];
}

// per site (both parities): sum over the six planes of Re tr of the
// plaquette (kind 0, plaquettes.c:14-78 times K) or of the 2x1 + 1x2
// rectangles (kind 1, rectangles.c:16-160 times K); block partials
__global__ __launch_bounds__(kBlock) void k_action_sum(GaugePtrs G, LinkGeom g, int pt, int kind, SolverCtl ctl) {
    const int gid = blockIdx.x * kBlock + (int)threadIdx.x;
    double v = 0.0;
    if (gid < 2 * g.sizeh) {
        const int parity = gid / g.sizeh, idxh = gid - parity * g.sizeh;
        int x[4];
        decode(idxh, parity, g, x);
#pragma unroll 1
        for (int mu = 0; mu < 3; mu++)
#pragma unroll 1
            for (int nu = mu + 1; nu < 4; nu++) {
                int y[4];
                Su3 A, B, C, T;
                double ka, kb, kc, kd;
                if (kind == 0) {
                    // A = U_mu(x), B = U_nu(x+mu), C = U_mu(x+nu), D = U_nu(x): Re tr(A B C^+ D^+)
                    link_y(G, g, mu, x, pt, A, ka);
                    site_off(x, mu, 1, nu, 0, g, y);
                    link_y(G, g, nu, y, pt, B, kb);
                    site_off(x, mu, 0, nu, 1, g, y);
                    link_y(G, g, mu, y, pt, C, kc);
                    Su3 D;
                    link_y(G, g, nu, x, pt, D, kd);
                    su3_mul(A, B, T);
                    su3_mul_dag(T, C, T);
                    su3_mul_dag(T, D, T);
                    v += (T.c[0][0].x + T.c[1][1].x + T.c[2][2].x) * (ka * kb * kc * kd);
                } else {
                    const Hop r21[6] = {{0, 0, 0}, {0, 1, 0}, {1, 2, 0}, {0, 1, 1}, {0, 0, 1}, {1, 0, 0}};
                    const Hop r12[6] = {{0, 0, 0}, {1, 1, 0}, {1, 1, 1}, {0, 0, 2}, {1, 0, 1}, {1, 0, 0}};
#pragma unroll
                    for (int shape = 0; shape < 2; shape++) {
                        const Hop* h = shape == 0 ? r21 : r12;
                        double k = 1.0;
#pragma unroll
                        for (int j = 0; j < 6; j++) {
                            Su3 M;
                            site_off(x, mu, h[j].a, nu, h[j].b, g, y);
                            double kj;
                            link_y(G, g, h[j].dir == 0 ? mu : nu, y, pt, j == 0 ? T : M, kj);
                            k *= kj;
                            if (j == 1 || j == 2) su3_mul(T, M, T);
                            else if (j >= 3) su3_mul_dag(T, M, T);
                        }
                        v += (T.c[0][0].x + T.c[1][1].x + T.c[2][2].x) * k;
                    }
                }
            }
    }
    block_partial<1>(v, 0.0, ctl);
}

// Fused smearing: U'(rows 0,1) = exp(-QA) U; optional side outputs of the
// reference's parking arrays (staples, QA, exp rows 0,1).
__global__ __launch_bounds__(kBlock) void k_stout(GaugePtrs G, double2* __restrict__ uout, size_t su3_stride,
                                                 LinkGeom g, double rho, double c0, double2* __restrict__ stap_out,
                                                 void* __restrict__ qa_out, double2* __restrict__ exp_out) {
    int dir, idxh;
    if (!link_of_tile(g.sizeh, dir, idxh)) return;
    const int mu = dir >> 1, parity = dir & 1;
    int d[4];
    decode(idxh, parity, g, d);
    Su3 S, U, X, E, O;
    staple_sum(G, g, d, idxh, mu, parity, c0, S);
    load_link(G.at(dir), g.sizeh, idxh, U);
    su3_mul(U, S, X);
    Tamat q;
    ta_part(X, rho / c0, q);
    ch_exp_minus_qa(q, E);
    // rows 0,1 of E * U
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double2 s = cmul(E.c[r][0], U.c[0][c]);
            s = cfma(E.c[r][1], U.c[1][c], s);
            s = cfma(E.c[r][2], U.c[2][c], s);
            O.c[r][c] = s;
        }
    double2* Uo = (double2*)((char*)uout + dir * su3_stride);
    store_rows(Uo, g.sizeh, idxh, O, 2);
    if (stap_out) store_rows((double2*)((char*)stap_out + dir * su3_stride), g.sizeh, idxh, S, 3);
    if (qa_out) ta_store(qa_out, dir, g.sizeh, idxh, q);
    if (exp_out) store_rows((double2*)((char*)exp_out + dir * su3_stride), g.sizeh, idxh, E, 2);
}

// staples accumulated into `stap` (calc_loc_staples_nnptrick_all_onlyferms adds)
__global__ __launch_bounds__(kBlock) void k_staples(GaugePtrs G, double2* __restrict__ stap, size_t su3_stride,
                                                   LinkGeom g, double c0) {
    int dir, idxh;
    if (!link_of_tile(g.sizeh, dir, idxh)) return;
    int d[4];
    decode(idxh, dir & 1, g, d);
    Su3 S, old;
    staple_sum(G, g, d, idxh, dir >> 1, dir & 1, c0, S);
    double2* P = (double2*)((char*)stap + dir * su3_stride);
    load_gl3(P, g.sizeh, idxh, old);
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) old.c[r][c] = cadd(old.c[r][c], S.c[r][c]);
    store_rows(P, g.sizeh, idxh, old, 3);
}

// QA = (rho/c0) TA(U * stap) (RHO_times_conf_times_staples_ta_part)
__global__ __launch_bounds__(kBlock) void k_rho_ta(GaugePtrs G, const double2* __restrict__ stap, size_t su3_stride,
                                                  void* __restrict__ qa, LinkGeom g, double rho, double c0) {
    const int gid = blockIdx.x * kBlock + (int)threadIdx.x;
    if (gid >= 8 * g.sizeh) return;
    int dir, idxh;
    link_of(gid, g.sizeh, dir, idxh);
    Su3 U, S, X;
    load_link(G.at(dir), g.sizeh, idxh, U);
    load_gl3((const double2*)((const char*)stap + dir * su3_stride), g.sizeh, idxh, S);
    su3_mul(U, S, X);
    Tamat q;
    ta_part(X, rho / c0, q);
    ta_store(qa, dir, g.sizeh, idxh, q);
}

// U_out(rows 0,1) = exp(-QA) U (exp_minus_QA_times_conf); exp rows 0,1 to exp_aux
__global__ __launch_bounds__(kBlock) void k_exp_times_conf(GaugePtrs G, const void* __restrict__ qa,
                                                          double2* __restrict__ uout, double2* __restrict__ exp_aux,
                                                          size_t su3_stride, LinkGeom g) {
    const int gid = blockIdx.x * kBlock + (int)threadIdx.x;
    if (gid >= 8 * g.sizeh) return;
    int dir, idxh;
    link_of(gid, g.sizeh, dir, idxh);
    Tamat q;
    ta_load(qa, dir, g.sizeh, idxh, q);
    Su3 E, U, O;
    ch_exp_minus_qa(q, E);
    load_link(G.at(dir), g.sizeh, idxh, U);
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double2 s = cmul(E.c[r][0], U.c[0][c]);
            s = cfma(E.c[r][1], U.c[1][c], s);
            s = cfma(E.c[r][2], U.c[2][c], s);
            O.c[r][c] = s;
        }
    store_rows((double2*)((char*)uout + dir * su3_stride), g.sizeh, idxh, O, 2);
    if (exp_aux) store_rows((double2*)((char*)exp_aux + dir * su3_stride), g.sizeh, idxh, E, 2);
}

// ------------------------------------------------------------- force chain
// Lambda of one link (compute_loc_Lambda, stouting.c:171-512): the derivative
// coefficients b_{1j}, b_{2j} of Morningstar-Peardon eqs. 57-58 (small-c1
// series as in NISSA), B_k = b_k0 + b_k1 Q + b_k2 Q^2, tr_k = Tr(Sigma' B_k U),
// Gamma = tr1 Q + tr2 Q^2 + f1 U Sigma' + f2 (Q U Sigma' + U Sigma' Q),
// Lambda = (Gamma + Gamma^+)/2 - Tr(Gamma + Gamma^+)/6.
__device__ void lambda_local(const Tamat& q, const Su3& SP, const Su3& U, Thmat& L) {
    double c0 = det_i_times_qa(q);
    const double c1 = 0.5 * tr_i_times_qa_sq(q);
    const double c0max = 2 * pow(c1 / 3, 1.5);
    double2 f0, f1, f2, b10, b11, b12, b20, b21, b22;
    if (c1 < 4e-3) {
        ch_coefficients(q, f0, f1, f2);
        b10 = make_double2(0.0, c0 / 120 * (1 - c1 / 21));
        b11 = make_double2(-c0 / 360 * (1 - 3 * c1 / 56), -1.0 / 6 * (1 - c1 / 10 * (1.0 - c1 / 28)));
        b12 = make_double2(0.5 * (1.0 / 12 * (1 - 2 * c1 / 30 * (1 - 3 * c1 / 112))), 0.5 * (-c0 / 1260 * (1 - c1 / 24)));
        b20 = make_double2(-c0 / 360, -1.0 / 6 * (1 - c1 / 20 * (1 - c1 / 42)));
        b21 = make_double2(1.0 / 24 * (1 - c1 / 15 * (1 - 3 * c1 / 112)), -c0 / 2520);
        b22 = make_double2(0.5 * c0 / 10080, 0.5 * (1.0 / 60 * (1 - c1 / 21 * (1 - c1 / 48))));
    } else {
        int sign = 1;
        if (c0 < 0) {
            sign = -1;
            c0 = -c0;
        }
        const double eps = (c0max - c0) / c0max;
        double theta;
        if (eps < 0) theta = 0.0;
        else if (eps < 1e-3)
            theta = sqrt(2 * eps) *
                    (1 + (1.0 / 12 + (3.0 / 160 + (5.0 / 896 + (35.0 / 18432 + 63.0 / 90112 * eps) * eps) * eps) * eps) * eps);
        else theta = acos(c0 / c0max);
        const double u = sqrt(c1 / 3) * cos(theta / 3);
        const double w = sqrt(c1) * sin(theta / 3);
        const double u2 = u * u, w2 = w * w, u2mw2 = u2 - w2, w2p3u2 = w2 + 3 * u2, w2m3u2 = w2 - 3 * u2;
        const double cu = cos(u), c2u = cos(2 * u), su = sin(u), s2u = sin(2 * u), cw = cos(w);
        double xi0w, xi1w;
        if (fabs(w) < 0.05) {
            const double t0 = w * w, t1 = 1 - t0 / 42, t2 = 1.0 - t0 / 20 * t1;
            xi0w = 1 - t0 / 6 * t2;
            xi1w = -(1 - w2 * (1 - w2 * (1 - w2 / 54) / 28) / 10) / 3;
        } else {
            xi0w = sin(w) / w;
            xi1w = cw / w2 - sin(w) / (w2 * w);
        }
        const double denom = 1 / (9 * u * u - w * w);
        f0 = make_double2((u2mw2 * c2u + cu * 8 * u2 * cw + 2 * su * u * w2p3u2 * xi0w) * denom,
                          (u2mw2 * s2u - su * 8 * u2 * cw + cu * 2 * u * w2p3u2 * xi0w) * denom);
        f1 = make_double2((2 * u * c2u - cu * 2 * u * cw - su * w2m3u2 * xi0w) * denom,
                          (2 * u * s2u + su * 2 * u * cw - cu * w2m3u2 * xi0w) * denom);
        f2 = make_double2((c2u - cu * cw - 3 * su * u * xi0w) * denom, (s2u + su * cw - cu * 3 * u * xi0w) * denom);
        const double2 r01 = make_double2(
            2 * c2u * u + s2u * (-2 * u2 + 2 * w2) + 2 * cu * u * (8 * cw + 3 * u2 * xi0w + w2 * xi0w) +
                su * (-8 * cw * u2 + 18 * u2 * xi0w + 2 * w2 * xi0w),
            -8 * cw * (2 * su * u + cu * u2) + 2 * (s2u * u + c2u * u2 - c2u * w2) +
                2 * (9 * cu * u2 - 3 * su * u * u2 + cu * w2 - su * u * w2) * xi0w);
        const double2 r11 = make_double2(2 * c2u - 4 * s2u * u + su * (2 * cw * u + 6 * u * xi0w) +
                                             cu * (-2 * cw + 3 * u2 * xi0w - w2 * xi0w),
                                         2 * s2u + 4 * c2u * u + 2 * cw * (su + cu * u) + (6 * cu * u - 3 * su * u2 + su * w2) * xi0w);
        const double2 r21 = make_double2(-2 * s2u + cw * su - 3 * (su + cu * u) * xi0w,
                                         2 * c2u + cu * cw + (-3 * cu + 3 * su * u) * xi0w);
        const double2 r02 = make_double2(-2 * c2u + 2 * cw * su * u + 2 * su * u * xi0w - 8 * cu * u2 * xi0w +
                                             6 * su * u * u2 * xi1w,
                                         2 * (-s2u + 4 * su * u2 * xi0w + cu * u * (cw + xi0w + 3 * u2 * xi1w)));
        const double2 r12 = make_double2(2 * cu * u * xi0w + su * (-cw - xi0w + 3 * u2 * xi1w),
                                         -2 * su * u * xi0w - cu * (cw + xi0w - 3 * u2 * xi1w));
        const double2 r22 = make_double2(cu * xi0w - 3 * su * u * xi1w, -(su * xi0w) - 3 * cu * u * xi1w);
        const double h = 0.5 * denom * denom;
        const double a1 = 2.0 * u, a2 = 3.0 * u * u - w * w, a3 = -2.0 * (15.0 * u * u + w * w);
        auto B1 = [&](double2 r1, double2 r2, double2 f) {
            return make_double2(h * (a1 * r1.x + a2 * r2.x + a3 * f.x), h * (a1 * r1.y + a2 * r2.y + a3 * f.y));
        };
        auto B2 = [&](double2 r1, double2 r2, double2 f) {
            return make_double2(h * (r1.x - 3.0 * u * r2.x - 24.0 * u * f.x), h * (r1.y - 3.0 * u * r2.y - 24.0 * u * f.y));
        };
        b10 = B1(r01, r02, f0);
        b11 = B1(r11, r12, f1);
        b12 = B1(r21, r22, f2);
        b20 = B2(r01, r02, f0);
        b21 = B2(r11, r12, f1);
        b22 = B2(r21, r22, f2);
        if (sign == -1) {
            b10 = cconj(b10);
            b11 = make_double2(-b11.x, b11.y);
            b12 = cconj(b12);
            b20 = make_double2(-b20.x, b20.y);
            b21 = cconj(b21);
            b22 = make_double2(-b22.x, b22.y);
            f0 = cconj(f0);
            f1 = make_double2(-f1.x, f1.y);
            f2 = cconj(f2);
        }
    }
    const double2 z = make_double2(0.0, 0.0), one = make_double2(1.0, 0.0);
    Su3 Bm, Q, Q2, T, USP, QU, UQ;
    itamat_poly_no3rdrow(z, one, z, q, Q);
    itamat_poly_row2(z, one, z, q, Q);
    itamat_poly_no3rdrow(z, z, one, q, Q2);
    itamat_poly_row2(z, z, one, q, Q2);
    // tr_k = Tr(Sigma' B_k U)
    double2 tr1 = z, tr2 = z;
    itamat_poly_no3rdrow(b10, b11, b12, q, Bm);
    itamat_poly_row2(b10, b11, b12, q, Bm);
    su3_mul(Bm, U, T);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) tr1 = cfma(SP.c[a][b], T.c[b][a], tr1);
    itamat_poly_no3rdrow(b20, b21, b22, q, Bm);
    itamat_poly_row2(b20, b21, b22, q, Bm);
    su3_mul(Bm, U, T);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) tr2 = cfma(SP.c[a][b], T.c[b][a], tr2);
    su3_mul(U, SP, USP);
    su3_mul(Q, USP, QU);
    su3_mul(USP, Q, UQ);
    Su3 G;
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
            double2 s = cmul(tr1, Q.c[a][b]);
            s = cfma(tr2, Q2.c[a][b], s);
            s = cfma(f1, USP.c[a][b], s);
            s = cfma(f2, cadd(QU.c[a][b], UQ.c[a][b]), s);
            G.c[a][b] = s;
        }
    const double third = 0.33333333333333333333333;
    L.rc00 = (2 * G.c[0][0].x - G.c[1][1].x - G.c[2][2].x) * third;
    L.rc11 = (2 * G.c[1][1].x - G.c[0][0].x - G.c[2][2].x) * third;
    L.c01 = cscale(cadd(G.c[0][1], cconj(G.c[1][0])), 0.5);
    L.c02 = cscale(cadd(G.c[0][2], cconj(G.c[2][0])), 0.5);
    L.c12 = cscale(cadd(G.c[1][2], cconj(G.c[2][1])), 0.5);
}

// staples -> QA -> Lambda for every link (compute_sigma_from_sigma_prime ... first half);
// GIVEN: QA is there already, which leaves 368 bytes and the Cayley-Hamilton
// coefficients per link instead of 18 neighbour links (225 -> 100 us on 32^3 x 8
// for 6 us more in k_stout, which stores it)
template <bool GIVEN>
__global__ __launch_bounds__(kBlock) void k_qa_lambda(GaugePtrs G, const double2* __restrict__ SP, size_t su3_stride,
                                                     void* __restrict__ qa, void* __restrict__ lam, LinkGeom g,
                                                     double rho, double c0) {
    int dir, idxh;
    if (!link_of_tile(g.sizeh, dir, idxh)) return;
    Su3 U, S;
    load_link(G.at(dir), g.sizeh, idxh, U);
    Tamat q;
    if (GIVEN) {
        ta_load(qa, dir, g.sizeh, idxh, q);
    } else {
        int d[4];
        decode(idxh, dir & 1, g, d);
        Su3 C, X;
        staple_sum(G, g, d, idxh, dir >> 1, dir & 1, c0, C);
        su3_mul(U, C, X);
        ta_part(X, rho / c0, q);
        ta_store(qa, dir, g.sizeh, idxh, q);
    }
    load_gl3((const double2*)((const char*)SP + dir * su3_stride), g.sizeh, idxh, S);
    Thmat L;
    lambda_local(q, S, U, L);
    th_store(lam, dir, g.sizeh, idxh, L);
}

// Sigma = Sigma' exp(iQ) + i rho (staple terms with Lambda) (compute_sigma, stouting.c:1175-1302)
//
// Bound by FP64 issue and, with its eight matrices in flight, by registers.  The
// six terms of a plane share their products (12 instead of 14, five of them with
// the Hermitian Lambdas), all terms add up in T, and exp(iQ) is formed after the
// planes, so that two waves fit a SIMD: 405 -> 279 us on 32^3 x 8 (5.2 GFMA
// before, 146 us at the FP64 rate; 4.1 now).
__global__ __launch_bounds__(kBlock, 2) void k_sigma(GaugePtrs G, const void* __restrict__ lam,
                                                    const void* __restrict__ qa, double2* __restrict__ S,
                                                    size_t su3_stride, LinkGeom g, double rho) {
    int dir, idxh;
    if (!link_of_tile(g.sizeh, dir, idxh)) return;
    const int mu = dir >> 1, parity = dir & 1, sh = g.sizeh;
    int d[4];
    decode(idxh, parity, g, d);
    Su3 T;
    su3_zero(T);
    Thmat ld;
    th_load(lam, dir, sh, idxh, ld);
    const int i_pmu = shifted(d, mu, 1, 0, 0, g);
#pragma unroll 1
    for (int it = 0; it < 3; it++) {
        const int nu = c_perp[mu][it];
        const int i_pnu = shifted(d, nu, 1, 0, 0, g), i_mnu = shifted(d, nu, -1, 0, 0, g);
        const int i_pmu_mnu = shifted(d, mu, 1, nu, -1, g);
        Thmat l1, l2;
        {
            // right part: A = U_nu(x+mu), B = U_mu(x+nu), C = U_nu(x):
            //   A B^+ [C^+ (L_mu(x) - L_nu(x)) - L_mu(x+nu) C^+] + L_nu(x+mu) A B^+ C^+
            Su3 A, B, C, AB, Z;
            load_link(G.at(2 * nu + !parity), sh, i_pmu, A);
            load_link(G.at(2 * mu + !parity), sh, i_pnu, B);
            su3_mul_dag(A, B, AB);
            load_link(G.at(2 * nu + parity), sh, idxh, C);
            th_load(lam, 2 * nu + parity, sh, idxh, l1);
            th_sub(ld, l1, l1);
            su3_zero(Z);
#pragma unroll
            for (int r = 0; r < 3; r++)
                th_row(cconj(C.c[0][r]), cconj(C.c[1][r]), cconj(C.c[2][r]), l1, Z.c[r]);
            th_load(lam, 2 * mu + !parity, sh, i_pnu, l2);
            Su3 Cd;
#pragma unroll
            for (int r = 0; r < 3; r++)
#pragma unroll
                for (int c = 0; c < 3; c++) Cd.c[r][c] = cconj(C.c[c][r]);
            th_mul_acc(th_neg(l2), Cd, Z);
            su3_mul_acc(AB, Z, T);
            su3_mul(AB, Cd, Z);
            th_load(lam, 2 * nu + !parity, sh, i_pmu, l1);
            th_mul_acc(l1, Z, T);
        }
        {
            // left part: A = U_nu(x+mu-nu), B = U_mu(x-nu), C = U_nu(x-nu):
            //   A^+ [B^+ ((L_nu(x-nu) - L_mu(x-nu)) C + C L_mu(x)) - L_nu(x+mu-nu) B^+ C]
            Su3 A, B, C, P, Q;
            load_link(G.at(2 * nu + !parity), sh, i_mnu, C);
            th_load(lam, 2 * nu + !parity, sh, i_mnu, l1);
            th_load(lam, 2 * mu + !parity, sh, i_mnu, l2);
            th_sub(l1, l2, l1);
            su3_zero(Q);
            th_mul_acc(l1, C, Q);
#pragma unroll
            for (int r = 0; r < 3; r++) th_row(C.c[r][0], C.c[r][1], C.c[r][2], ld, Q.c[r]);
            load_link(G.at(2 * mu + !parity), sh, i_mnu, B);
            su3_dag_mul(B, Q, Q);
            su3_dag_mul(B, C, P);
            th_load(lam, 2 * nu + parity, sh, i_pmu_mnu, l2);
            th_mul_acc(th_neg(l2), P, Q);
            load_link(G.at(2 * nu + parity), sh, i_pmu_mnu, A);
            su3_dag_mul_acc(A, Q, T);
        }
    }
    Tamat q;
    ta_load(qa, dir, sh, idxh, q);
    Su3 E, SPm, res;
    ch_exp_minus_qa(q, E);
    rebuild3row(E);
    double2* Sd = (double2*)((char*)S + dir * su3_stride);
    load_gl3(Sd, sh, idxh, SPm);
    su3_mul(SPm, E, res);
    su3_axpy(make_double2(0.0, rho), T, res);
    store_rows(Sd, sh, idxh, res, 3);
}

// unitarize_conf (su3_utilities.c:17-40, loc_unitarize_conf su3_utilities.h:68-113)
__global__ __launch_bounds__(kBlock) void k_unitarize(double2* __restrict__ u, size_t su3_stride, int sizeh) {
    const int gid = blockIdx.x * kBlock + (int)threadIdx.x;
    if (gid >= 8 * sizeh) return;
    int dir, i;
    link_of(gid, sizeh, dir, i);
    double2* U = (double2*)((char*)u + dir * su3_stride);
    double2 a0 = U[i], a1 = U[sizeh + i], a2 = U[2 * sizeh + i];
    double2 b0 = U[3 * sizeh + i], b1 = U[4 * sizeh + i], b2 = U[5 * sizeh + i];
    double n = 1.0 / sqrt(cnorm2(a0) + cnorm2(a1) + cnorm2(a2));
    a0 = cscale(a0, n);
    a1 = cscale(a1, n);
    a2 = cscale(a2, n);
    double2 sp = cmulc(a0, b0);
    sp = cfmac(a1, b1, sp);
    sp = cfmac(a2, b2, sp);
    b0 = csub(b0, cmul(sp, a0));
    b1 = csub(b1, cmul(sp, a1));
    b2 = csub(b2, cmul(sp, a2));
    n = 1.0 / sqrt(cnorm2(b0) + cnorm2(b1) + cnorm2(b2));
    U[i] = a0;
    U[sizeh + i] = a1;
    U[2 * sizeh + i] = a2;
    U[3 * sizeh + i] = cscale(b0, n);
    U[4 * sizeh + i] = cscale(b1, n);
    U[5 * sizeh + i] = cscale(b2, n);
}

// ---------------------------------------------------------------- launchers
static LinkGeom link_geom() {
    const Lattice& L = ctx().lat;
    LinkGeom g;
    for (int i = 0; i < 4; i++) g.nd[i] = L.nd[i];
    g.sizeh = (int)L.sizeh;
    return g;
}
static GaugePtrs gauge_ptrs(const void* u) {
    GaugePtrs G;
    const size_t st = ctx().lat.su3_bytes();
    G.base = (const char*)u;
    G.stride = st;
    return G;
}
static int nblk8() { return blocks_for(8 * ctx().lat.sizeh); }
static int nblk_tiles() { return 8 * blocks_for(ctx().lat.sizeh); }  // link_of_tile kernels

bool launch_stout(const void* u, void* uout, double rho, double c0, void* stap, void* qa, void* expo) {
    hipLaunchKernelGGL(k_stout, dim3(nblk_tiles()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(u), (double2*)uout,
                       ctx().lat.su3_bytes(), link_geom(), rho, c0, (double2*)stap, qa, (double2*)expo);
    return hip_ok(hipGetLastError(), "k_stout");
}

// the stout levels arr_1 .. arr_steps of u; qa (or null) receives each level's QA
bool launch_stout_levels(const void* u, char* arr, int steps, double rho, char* qa) {
    const size_t gb = 8 * ctx().lat.su3_bytes(), tb = (size_t)8 * 64 * ctx().lat.sizeh;
    for (int level = 0; level < steps; level++)
        if (!launch_stout(level ? arr + (level - 1) * gb : u, arr + level * gb, rho, g_c_zero, nullptr,
                          qa ? qa + level * tb : nullptr, nullptr))
            return false;
    return true;
}

static bool launch_qa_lambda(bool given, const void* u, const void* sp, void* qa, void* lam, double rho, double c0) {
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nblk_tiles()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(u), (const double2*)sp,
                           ctx().lat.su3_bytes(), qa, lam, link_geom(), rho, c0);
    };
    if (given) go(k_qa_lambda<true>);
    else go(k_qa_lambda<false>);
    return hip_ok(hipGetLastError(), "k_qa_lambda");
}

// qa_given: qa holds u's QA, else it is formed from the staples and left there
bool launch_sigma_chain(void* sigma, void* lam, void* qa, const void* u, double rho, double c0, bool qa_given) {
    const size_t st = ctx().lat.su3_bytes();
    if (!launch_qa_lambda(qa_given, u, sigma, qa, lam, rho, c0)) return false;
    hipLaunchKernelGGL(k_sigma, dim3(nblk_tiles()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(u), (const void*)lam,
                       (const void*)qa, (double2*)sigma, st, link_geom(), rho);
    return hip_ok(hipGetLastError(), "k_sigma");
}

static int g_gf_planes = 1;  // the plane kernel where it is faster (2: wherever it can; 0: the per-link kernel)

// the LDS arrays of a tm x tn tile; false when they exceed the pool
static bool gf_plan(int tm, int tn, GfPlan& p) {
    // first i, j and numbers of sites along i, j of each role (GfRole)
    const int rng[gRoles][4] = {{-2, -2, tm + 3, tn + 4}, {-2, -2, tm + 4, tn + 3}, {-1, -2, tm + 2, tn + 2},
                                {-2, -1, tm + 2, tn + 2}, {-1, 1, tm + 1, tn},      {-1, -1, tm + 1, tn + 1},
                                {1, -1, tm, tn + 1},      {-1, -1, tm + 1, tn + 1}};
    p.tm = tm;
    p.tn = tn;
    p.inv_tm = (65536 + tm - 1) / tm;
    int off = 0;
    for (int r = 0; r < gRoles; r++) {
        GfArr& a = p.a[r];
        a.off = off;
        a.rw = rng[r][2];
        a.n = rng[r][2] * rng[r][3];
        a.org = rng[r][1] * a.rw + rng[r][0];
        a.inv = (65536 + a.rw - 1) / a.rw;
        off += a.n;
    }
    // links and corners one pass each, the staples two; the sides' exchange (256 records) and the force
    // records (128) lie past the links
    const int nl = p.a[gM].n + p.a[gN].n, np = p.a[gSMp].n + p.a[gSNp].n;
    return tm * tn <= 64 && off <= kGfPool && nl <= kGfPoolLinks && nl <= 85 * kGfFetch &&
           p.a[gCm].n + p.a[gCn].n <= 256 && ((np + 63) & ~63) + p.a[gSMm].n + p.a[gSNm].n <= 512 &&
           nl + 256 + 128 <= kGfPool;
}

// The tile for a plane of extents nm x nn: the least work per site, counted
// in complex multiply-adds of the block's waves (corners 24, staples 30, a
// side 140 and U S with its share of the rest 40 per wave), the links loaded
// and a fifth on top where the rows are not whole groups of 16 lanes (bank
// conflicts), over the sites a tile covers on average (a tile that does not
// divide the extent wastes the lanes past it).
static GfPlan gf_best_plan(int nm, int nn) {
    GfPlan best{}, p;
    double cost = 0.0;
    for (int tm = 1; tm <= nm && tm <= 64; tm++)
        for (int tn = 1; tn <= nn && tm * tn <= 64; tn++) {
            if (!gf_plan(tm, tn, p)) continue;
            auto waves = [](int n) { return (n + 63) / 64; };
            const double c = (24.0 * waves(p.a[gCm].n + p.a[gCn].n) +
                              30.0 * (waves(p.a[gSMp].n + p.a[gSNp].n) + waves(p.a[gSMm].n + p.a[gSNm].n)) +
                              4.0 * 140.0 + 2.0 * 40.0 + 24.0 * (p.a[gM].n + p.a[gN].n) / 64.0) *
                             (tm % 16 == 0 ? 1.0 : 1.2);
            p.tiles_m = (nm + tm - 1) / tm;
            p.tiles_n = (nn + tn - 1) / tn;
            if (cost == 0.0 || c * p.tiles_m * p.tiles_n < cost) {
                cost = c * p.tiles_m * p.tiles_n;
                best = p;
            }
        }
    return best;
}

// link records (96 B per link) and the three planes' force parts (3 x 64 B per link) of the current lattice
static Workspace g_gf_rec, g_gf_part;

struct GfPlanned {
    int nd[4] = {0, 0, 0, 0};
    GfPlans plans;
};
static const GfPlans& gf_plans() {
    static const int planes[6][2] = {{0, 1}, {0, 2}, {0, 3}, {1, 2}, {1, 3}, {2, 3}};
    static GfPlanned c;
    const Lattice& L = ctx().lat;
    if (!std::equal(c.nd, c.nd + 4, L.nd)) {
        for (int p = 0; p < 6; p++) {
            GfPlan& q = c.plans.p[p];
            const int mu = planes[p][0], nu = planes[p][1];
            q = gf_best_plan(L.nd[mu], L.nd[nu]);
            q.mu = mu;
            q.nu = nu;
            q.tiles = q.tiles_m * q.tiles_n;
            for (int k = 0; k < 4; k++)
                if (k != mu && k != nu) q.tiles *= L.nd[k];
            c.plans.tiles[p] = q.tiles;
        }
        std::copy(L.nd, L.nd + 4, c.nd);
    }
    return c.plans;
}

// lane offsets within a link array are 32-bit in the per-link kernel (up to 6 planes of 16 sizeh bytes)
static bool gf_size_ok() { return (size_t)96 * ctx().lat.sizeh < ((size_t)1 << 32); }

// Whether the plane kernel is the faster one; moves: for the integrator, whose links stay in records between the
// forces.  Only for the action with rectangles, whose staples share products (per force on 24^4: tiles 591 us, links
// 782; Wilson 417, 261), and not where the staples are asked for (their sums over the planes took a launch a plane:
// 1161 us, 840 by links).  The tiles come 512 at a time, two blocks per CU, the per-link kernel a block per CU for
// every 2048 half-sites, at 6 to 10 us a round, so few sites a tile (extents of 2) or a last round that is nearly
// empty decide: steps of the integrator, links against tiles, 16^3 x 4 (2 rounds of tiles, 4 of links) 51 -> 41 us, 12^3 x 4
// (2, 2) 30.2 -> 27.8, 10^3 x 8 (3, 2) 30.6 -> 32.5 with defect coefficients, 16^3 x 2 (3, 2) 28.9 -> 29.4,
// 64 x 64 x 2 x 2 (13, 4) 51 -> 82.  A force by itself also packs the records: 12x18x4x14 (6048) 33.6 -> 36.7,
// 18x10x12x6 (6480) 43.5 -> 36.7, 16^4 166 -> 112.
static bool gf_planes_pay(bool moves) {
    const long sizeh = ctx().lat.sizeh;
    long tiles = 0;
    for (const GfPlan& q : gf_plans().p) tiles += q.tiles;
    return (tiles + 511) / 512 <= (sizeh + 2047) / 2048 && (moves || sizeh > 6144);
}

// the plane kernel's buffers, or false: the per-link kernel then (its halo wraps at most once along a direction)
bool gf_planes_ready(bool moves) {
    const Lattice& L = ctx().lat;
    if (!g_gf_planes || !gf_size_ok() || !g_tlsm) return false;
    // even extents: a wrap keeps the site's parity
    for (int k = 0; k < 4; k++)
        if (L.nd[k] < 2 || (L.nd[k] & 1)) return false;
    // 24-bit products of a coordinate and its stride
    if ((long)L.nd[0] * L.nd[1] * L.nd[2] >= (1L << 24) || L.nd[3] >= (1 << 24)) return false;
    if (g_gf_planes == 1 && !gf_planes_pay(moves)) return false;
    const size_t links = (size_t)8 * L.sizeh;
    if (g_gf_rec.try_get(96 * links) && g_gf_part.try_get(3 * 64 * links)) return true;
    g_gf_rec.release();  // one without the other is of no use
    return false;
}
static dim3 gf_grid8() { return dim3(blocks_for(ctx().lat.sizeh), 8); }

bool gf_pack(const void* u) {
    hipLaunchKernelGGL(k_gf_pack, gf_grid8(), dim3(kBlock), 0, ctx().stream, gauge_ptrs(u), (double2*)g_gf_rec.p,
                       (int)ctx().lat.sizeh);
    return hip_ok(hipGetLastError(), "k_gf_pack");
}
bool gf_unpack(void* u) {
    hipLaunchKernelGGL(k_gf_unpack, gf_grid8(), dim3(kBlock), 0, ctx().stream, (const double2*)g_gf_rec.p,
                       gauge_ptrs(u), (int)ctx().lat.sizeh);
    return hip_ok(hipGetLastError(), "k_gf_unpack");
}

// the planes' force parts of the records' links (K planes from u): the planes are independent, one launch, two
// blocks per CU (and at least a block for each XCD's share of the tiles)
bool gf_parts(const void* u) {
    const GfPlans& plans = gf_plans();
    long tiles = 0;
    for (const GfPlan& q : plans.p) tiles += q.tiles;
    const unsigned nb = (unsigned)std::max(8L, std::min(tiles, 512L));
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nb), dim3(256), 0, ctx().stream, (const double2*)g_gf_rec.p, gauge_ptrs(u),
                           (double2*)g_gf_part.p, link_geom(), plans, g_c_zero);
    };
    if (ctx().lat.par_temp) go(k_gf_tile<true>);
    else go(k_gf_tile<false>);
    return hip_ok(hipGetLastError(), "k_gf_tile");
}
bool gf_ipdot(void* ipdot, void* mom, double fact) {
    hipLaunchKernelGGL(k_gf_ipdot, gf_grid8(), dim3(kBlock), 0, ctx().stream, (const double2*)g_gf_part.p, ipdot, mom,
                       (int)ctx().lat.sizeh, fact);
    return hip_ok(hipGetLastError(), "k_gf_ipdot");
}
// momentum step with the parts, then U <- exp(i delta P) U on the records
bool gf_move(void* mom, double fact, double delta) {
    hipLaunchKernelGGL(k_gf_move, gf_grid8(), dim3(kBlock), 0, ctx().stream, (const double2*)g_gf_part.p, mom,
                       (double2*)g_gf_rec.p, (int)ctx().lat.sizeh, fact, delta);
    return hip_ok(hipGetLastError(), "k_gf_move");
}
bool launch_gauge_force(const void* u, void* stap, void* ipdot, void* mom, double fact) {
    const Lattice& L = ctx().lat;
    if (!gf_size_ok()) return fail("gauge force: lattice too large (sizeh %ld)", (long)L.sizeh);
    if (!stap && gf_planes_ready(false)) return gf_pack(u) && gf_parts(u) && gf_ipdot(ipdot, mom, fact);
    // whole blocks per link array (the kernel takes the direction from the block)
    const int nb = 8 * (int)((L.sizeh + kGfLinks - 1) / kGfLinks);
    hipLaunchKernelGGL(k_gauge_force, dim3(nb), dim3(3 * kGfLinks), 0, ctx().stream, gauge_ptrs(u), (double2*)stap,
                       L.su3_bytes(), ipdot, link_geom(), L.par_temp, g_tlsm ? 1 : 0, g_c_zero, mom, fact);
    return hip_ok(hipGetLastError(), "k_gauge_force");
}

// kind 0: plaquettes, 1: rectangles; the sum returned on the host
bool gauge_action_sum(const void* u, int kind, double* out) {
    const Lattice& L = ctx().lat;
    const int nb = blocks_for(2 * L.sizeh);
    SolverCtl c = plain_ctl();
    hipLaunchKernelGGL(k_action_sum, dim3(nb), dim3(kBlock), 0, ctx().stream, gauge_ptrs(u), link_geom(),
                       L.par_temp, kind, c);
    if (!hip_ok(hipGetLastError(), "k_action_sum") || !launch_finalize(kFinStore, c, nb)) return false;
    double v = 0.0;
    if (!hip_ok(hipMemcpyAsync(&v, &ctx().state->sum, sizeof(double), hipMemcpyDeviceToHost, ctx().stream),
                "action readback") ||
        !hip_ok(hipStreamSynchronize(ctx().stream), "action readback"))
        return false;
    *out = v;
    return true;
}

double stout_c_zero() { return g_c_zero; }
bool stout_tlsm() { return g_tlsm; }

}  // namespace ostp

using namespace ostp;

// ------------------------------------------------------------ C entry points
static bool sync(const char* nm) { return hip_ok(hipStreamSynchronize(ctx().stream), nm); }
static double rho_of(int istopo) { return istopo ? gl_topo_rho : gl_stout_rho; }

extern "C" {

int ostp_stout_steps(void) { return g_stout_steps; }

void ostp_set_stout(double rho, int steps, double topo_rho, int topo_steps, int topo_action, int tlsm) {
    gl_stout_rho = rho;
    gl_topo_rho = topo_rho;
    g_stout_steps = steps;
    g_topo_steps = topo_steps;
    g_topo_action = topo_action;
    g_c_zero = tlsm ? 5.0 * 0.33333333333333333333333 : 1.0;
    g_tlsm = tlsm != 0;
}

void stout_isotropic(const su3_soa* u, su3_soa* uprime, su3_soa* local_staples, su3_soa* auxiliary,
                     tamat_soa* tipdot, const int istopo) {
    const char* nm = "stout_isotropic";
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes(), tb = (size_t)8 * 64 * L.sizeh;
    const void* du = resolve(u, gb, nm);
    void* dout = resolve(uprime, gb, nm);
    void* dst = local_staples ? resolve(local_staples, gb, nm) : nullptr;
    void* dex = auxiliary ? resolve(auxiliary, gb, nm) : nullptr;
    void* dqa = tipdot ? resolve(tipdot, tb, nm) : nullptr;
    if (!du || !dout || (local_staples && !dst) || (auxiliary && !dex) || (tipdot && !dqa)) return;
    if (launch_stout(du, dout, rho_of(istopo), g_c_zero, dst, dqa, dex)) sync(nm);
}

void stout_wrapper(const su3_soa* tconf_acc, su3_soa* tstout_conf_acc_arr, const int istopo) {
    const char* nm = "stout_wrapper";
    if (!require_init(nm)) return;
    const int steps = (istopo & g_topo_action) ? g_topo_steps : g_stout_steps;
    if (steps <= 0) return;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes();
    const void* du = resolve(tconf_acc, gb, nm);
    char* arr = (char*)resolve(tstout_conf_acc_arr, steps * gb, nm);
    if (!du || !arr) return;
    if (launch_stout_levels(du, arr, steps, rho_of(istopo), nullptr)) sync(nm);
}

void exp_minus_QA_times_conf(const su3_soa* tu, const tamat_soa* QA, su3_soa* tu_out, su3_soa* exp_aux) {
    const char* nm = "exp_minus_QA_times_conf";
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes(), tb = (size_t)8 * 64 * L.sizeh;
    const void* du = resolve(tu, gb, nm);
    const void* dq = resolve(QA, tb, nm);
    void* dout = resolve(tu_out, gb, nm);
    void* dex = exp_aux ? resolve(exp_aux, gb, nm) : nullptr;
    if (!du || !dq || !dout || (exp_aux && !dex)) return;
    hipLaunchKernelGGL(k_exp_times_conf, dim3(nblk8()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(du), dq,
                       (double2*)dout, (double2*)dex, L.su3_bytes(), link_geom());
    if (hip_ok(hipGetLastError(), nm)) sync(nm);
}

void calc_loc_staples_nnptrick_all_onlyferms(const su3_soa* u, su3_soa* loc_stap) {
    const char* nm = "calc_loc_staples_nnptrick_all_onlyferms";
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const void* du = resolve(u, 8 * L.su3_bytes(), nm);
    void* ds = resolve(loc_stap, 8 * L.su3_bytes(), nm);
    if (!du || !ds) return;
    hipLaunchKernelGGL(k_staples, dim3(nblk_tiles()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(du), (double2*)ds,
                       L.su3_bytes(), link_geom(), g_c_zero);
    if (hip_ok(hipGetLastError(), nm)) sync(nm);
}

void RHO_times_conf_times_staples_ta_part(const su3_soa* u, const su3_soa* loc_stap, tamat_soa* tipdot, int istopo) {
    const char* nm = "RHO_times_conf_times_staples_ta_part";
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const void* du = resolve(u, 8 * L.su3_bytes(), nm);
    const void* ds = resolve(loc_stap, 8 * L.su3_bytes(), nm);
    void* dq = resolve(tipdot, (size_t)8 * 64 * L.sizeh, nm);
    if (!du || !ds || !dq) return;
    hipLaunchKernelGGL(k_rho_ta, dim3(nblk8()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(du), (const double2*)ds,
                       L.su3_bytes(), dq, link_geom(), rho_of(istopo), g_c_zero);
    if (hip_ok(hipGetLastError(), nm)) sync(nm);
}

void compute_lambda(thmat_soa* Lm, const su3_soa* SP, const su3_soa* U, const tamat_soa* QA, su3_soa* TMP) {
    const char* nm = "compute_lambda";
    (void)TMP;
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes(), tb = (size_t)8 * 64 * L.sizeh;
    void* dl = resolve(Lm, tb, nm);
    const void* ds = resolve(SP, gb, nm);
    const void* du = resolve(U, gb, nm);
    const void* dq = resolve(QA, tb, nm);
    if (!dl || !ds || !du || !dq) return;
    if (launch_qa_lambda(true, du, ds, const_cast<void*>(dq), dl, 0.0, g_c_zero)) sync(nm);
}

void compute_sigma(const thmat_soa* Lm, const su3_soa* U, su3_soa* S, const tamat_soa* QA, su3_soa* TMP,
                   const int istopo) {
    const char* nm = "compute_sigma";
    (void)TMP;
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes(), tb = (size_t)8 * 64 * L.sizeh;
    const void* dl = resolve(Lm, tb, nm);
    const void* du = resolve(U, gb, nm);
    void* ds = resolve(S, gb, nm);
    const void* dq = resolve(QA, tb, nm);
    if (!dl || !ds || !du || !dq) return;
    hipLaunchKernelGGL(k_sigma, dim3(nblk_tiles()), dim3(kBlock), 0, ctx().stream, gauge_ptrs(du), dl, dq, (double2*)ds,
                       L.su3_bytes(), link_geom(), rho_of(istopo));
    if (hip_ok(hipGetLastError(), nm)) sync(nm);
}

void compute_sigma_from_sigma_prime_backinto_sigma_prime(su3_soa* Sigma, thmat_soa* Lambda, tamat_soa* QA,
                                                          const su3_soa* U, su3_soa* TMP, const int istopo) {
    const char* nm = "compute_sigma_from_sigma_prime_backinto_sigma_prime";
    (void)TMP;
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes(), tb = (size_t)8 * 64 * L.sizeh;
    void* ds = resolve(Sigma, gb, nm);
    void* dl = resolve(Lambda, tb, nm);
    void* dq = resolve(QA, tb, nm);
    const void* du = resolve(U, gb, nm);
    if (!ds || !dl || !dq || !du) return;
    if (launch_sigma_chain(ds, dl, dq, du, rho_of(istopo), g_c_zero, false)) sync(nm);
}

void unitarize_conf(su3_soa* u) {
    const char* nm = "unitarize_conf";
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    void* du = resolve(u, 8 * L.su3_bytes(), nm);
    if (!du) return;
    hipLaunchKernelGGL(k_unitarize, dim3(nblk8()), dim3(kBlock), 0, ctx().stream, (double2*)du, L.su3_bytes(),
                       (int)L.sizeh);
    if (hip_ok(hipGetLastError(), nm)) sync(nm);
}

// ipdot_gauge.c:361-372 (GAUGE_ACTION from ostp_set_stout's tlsm flag)
void calc_ipdot_gauge_soloopenacc(const su3_soa* tconf_acc, su3_soa* local_staples, tamat_soa* tipdot) {
    const char* nm = "calc_ipdot_gauge_soloopenacc";
    if (!require_init(nm)) return;
    const Lattice& L = ctx().lat;
    const void* du = resolve(tconf_acc, 8 * L.su3_bytes(), nm);
    void* ds = resolve(local_staples, 8 * L.su3_bytes(), nm);
    void* dt = resolve(tipdot, 8 * (size_t)64 * L.sizeh, nm);
    if (!du || !ds || !dt) return;
    if (launch_gauge_force(du, ds, dt, nullptr, 0.0)) sync(nm);
}

// su3_measurements.c:191-211: sum over sites and the six planes of Re tr of
// the plaquettes (times the defect coefficients with PAR_TEMP).  The
// reference's scratch arguments are not written.
double calc_plaquette_soloopenacc(const su3_soa* tconf_acc, su3_soa* local_plaqs, dcomplex_soa* tr_local_plaqs) {
    (void)local_plaqs;
    (void)tr_local_plaqs;
    const char* nm = "calc_plaquette_soloopenacc";
    if (!require_init(nm)) return NAN;
    const void* du = resolve(tconf_acc, 8 * ctx().lat.su3_bytes(), nm);
    double v = NAN;
    if (du && !gauge_action_sum(du, 0, &v)) return NAN;
    return v;
}

// rectangles.c:1890-1909: the same for the 2x1 and 1x2 rectangles
double calc_rettangolo_soloopenacc(const su3_soa* tconf_acc, su3_soa* local_plaqs, dcomplex_soa* tr_local_plaqs) {
    (void)local_plaqs;
    (void)tr_local_plaqs;
    const char* nm = "calc_rettangolo_soloopenacc";
    if (!require_init(nm)) return NAN;
    const void* du = resolve(tconf_acc, 8 * ctx().lat.su3_bytes(), nm);
    double v = NAN;
    if (du && !gauge_action_sum(du, 1, &v)) return NAN;
    return v;
}

// device time per launch of the gauge-force kernel (HIP events on the
// library stream), with the fused momentum step when mom is not null
int ostp_set_gauge_force_kernel(int planes) {
    const int prev = g_gf_planes;
    g_gf_planes = planes == 2 ? 2 : planes ? 1 : 0;
    return prev;
}

double ostp_time_gauge_force(const su3_soa* u, su3_soa* stap, tamat_soa* ipdot, thmat_soa* mom, double fact,
                             int reps) {
    const char* nm = "ostp_time_gauge_force";
    if (!require_init(nm)) return -1.0;
    const Lattice& L = ctx().lat;
    const size_t gb = 8 * L.su3_bytes(), tb = (size_t)8 * 64 * L.sizeh;
    const void* du = resolve(u, gb, nm);
    void* ds = stap ? resolve(stap, gb, nm) : nullptr;
    void* di = resolve(ipdot, tb, nm);
    void* dm = mom ? resolve(mom, tb, nm) : nullptr;
    if (!du || (stap && !ds) || !di || (mom && !dm) || reps <= 0) return -1.0;
    hipEvent_t e0, e1;
    if (!hip_ok(hipEventCreate(&e0), "event") || !hip_ok(hipEventCreate(&e1), "event")) return -1.0;
    (void)hipEventRecord(e0, ctx().stream);
    for (int r = 0; r < reps; r++)
        if (!launch_gauge_force(du, ds, di, dm, fact)) return -1.0;
    (void)hipEventRecord(e1, ctx().stream);
    (void)hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return 1000.0 * (double)ms / reps;
}

}  // extern "C"
