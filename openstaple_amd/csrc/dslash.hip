// Even-odd staggered Dirac operator on gfx950.
//
// D_eo / D_oe of OpenAcc/fermion_matrix.c:47-157 with the per-link algebra of
// OpenAcc/matvecmul.h:88-172: for an output half-site x of one parity,
//   out(x) = 1/2 [ sum_mu U_mu(x) e^{i th_mu(x)} in(x+mu)
//                - sum_mu U_mu(x-mu)^dag e^{-i th_mu(x-mu)} in(x-mu) ],
// with only rows 0,1 of each link read (row 2 = conj(row0 x row1)) and the
// U(1) phase e^{i th} = cos th + i sin th folded in at load time.
//
// One thread per output half-site (k_dslash; k_dslash_split spreads a site's
// hops over eight waves where that is faster); consecutive lanes own consecutive
// half-sites, so every SoA plane access is a fully coalesced 128-bit (FP64)
// or 64-bit (FP32) load.  Workgroups are remapped so each XCD streams a
// contiguous slab of the lattice and its L2 serves the neighbour-spinor
// re-reads.  The kernel is HBM-bound (about 0.6 flop/byte); no MFMA.
//
// Epilogues fuse fermion_matrix_multiplication_shifted's
// combine_in1xferm_mass_minus_in2 (fermionic_utilities.c:261-272) and the
// CG's alpha = (p, s) reduction (inverter_full.c:76) into the second hop.
#include "ostp_dslash.h"

namespace ostp {

template <typename R>
struct DslashArgs {
    using C = typename Cplx<R>::T;
    const C* u[8];      // start of r0.c0 of link array 2*mu+parity
    const R* ph[8];     // phase array 2*mu+parity
    const C* in;
    C* out;
    const C* x;         // epilogue input: out = m2*x - D in
    double m2;
    const double2* b;   // kMdagMResid
    float2* rf;
    const unsigned char* sg;  // signs of the hops (SGN), of this output parity
    SiteGeom g;
    int tmajor;         // workgroup order: t-slices fastest (see k_dslash)
    int rev;            // each XCD walks its slab backwards
    SolverCtl ctl;
};

template <typename C>
__device__ __forceinline__ void st_out(C* p, C v) {
    if constexpr (sizeof(C) == 16) st_nt(p, v);
    else *p = v;
}

// What a half-site's colour does with o = (D in): element k; the return value
// is its term of the fused reduction.
template <typename R, int MODE>
__device__ __forceinline__ double dslash_out(const DslashArgs<R>& a, long k, typename Cplx<R>::T o,
                                             typename Cplx<R>::T x) {
    using C = typename Cplx<R>::T;
    if constexpr (MODE == kPlain) {
        st_out(a.out + k, o);
        return 0.0;
    }
    // combine_in1xferm_mass_minus_in2: out = x*m2 - D in  (promoted to double)
    const double sx = (double)x.x * a.m2 - (double)o.x, sy = (double)x.y * a.m2 - (double)o.y;
    if constexpr (MODE == kMdagMResid) {
        // r_f = (float)(b - (x*m2 - D in)), |r_f|^2; the FP64 product itself is not stored
        const double2 bb = a.b[k];
        const float2 f = make_float2((float)(bb.x - sx), (float)(bb.y - sy));
        a.rf[k] = f;
        return (double)f.x * f.x + (double)f.y * f.y;
    }
    const C sv = mk<C>(sx, sy);
    st_out(a.out + k, sv);
    return MODE == kMdagMDot ? re_dot(x, sv) : 0.0;
}

// Workgroup -> sites: the XCD remap gives each XCD a contiguous range of
// logical tiles; with tmajor the logical tile index runs over t fastest,
// so the +-t neighbour slices of a tile are streamed by the same XCD at
// nearly the same time and its L2 serves their re-reads (FP64: 81.2 us vs
// 85.5 us per 32^4 Dslash).
template <typename R>
__device__ __forceinline__ int dslash_idx(const DslashArgs<R>& a, int blk, int sites, int i) {
    if (a.tmajor) {
        const int s3 = a.g.sizeh / a.g.nd3;
        const int tile = blk / a.g.nd3, tt = blk - tile * a.g.nd3;
        return tt * s3 + tile * sites + i;
    }
    return blk * sites + i;
}

// EO = 0: Deo (even output, odd input); EO = 1: Doe.
template <typename R, int EO, int MODE, bool SGN = false>
__global__ __launch_bounds__(kBlock) void k_dslash(DslashArgs<R> a) {
    using C = typename Cplx<R>::T;
    if (!pred_pass(a.ctl)) return;
    const int blk = xcd_block_id_dir(a.rev);
    const int idx = dslash_idx(a, blk, kBlock, (int)threadIdx.x);
    double dot = 0.0;
    if (idx < a.g.sizeh) {
        C o[3];
        dslash_site<R, EO, SGN>(a.u, a.ph, a.in, a.g, idx, o[0], o[1], o[2], SGN ? a.sg[idx] : 0u);
        C x[3];
#pragma unroll
        for (int c = 0; c < 3; c++) x[c] = MODE == kPlain ? o[c] : a.x[(long)c * a.g.sizeh + idx];
#pragma unroll
        for (int c = 0; c < 3; c++) dot += dslash_out<R, MODE>(a, (long)c * a.g.sizeh + idx, o[c], x[c]);
    }
    // partial slot = logical tile, so the reduction order is the same in both walk directions
    if (MODE >= kMdagMDot) block_partial_at<kBlock>(dot, 0.0, a.ctl.partials, blk);
}

// The same with a half-site's eight hops split over the waves of a block: 64
// sites a block, wave h takes hop h of k_dslash's order, and the results are
// added in that order, so the outputs are k_dslash's.
constexpr int kSplitSites = 64, kSplitWaves = 8;
template <typename R, int EO, int MODE>
__global__ __launch_bounds__(64 * kSplitWaves) void k_dslash_split(DslashArgs<R> a) {
    using C = typename Cplx<R>::T;
    if (!pred_pass(a.ctl)) return;
    constexpr int F = EO == 0 ? 0 : 1, B = 1 - F;
    __shared__ C con[kSplitWaves][3][64];
    const int lane = (int)threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int blk = xcd_block_id_dir(a.rev);
    const int site = dslash_idx(a, blk, kSplitSites, lane);
    const bool live = site < a.g.sizeh;
    const int idx = live ? site : 0, sh = a.g.sizeh;
    // colour c is finished by wave c; its x is loaded before the hop
    C x = mk<C>(0, 0);
    if (MODE != kPlain && w < 3) x = a.x[(long)w * sh + idx];
    const Nbrs nb = site_neighbours<EO>(a.g, idx);
    const int mu = w & 3;
    C o0 = mk<C>(0, 0), o1 = mk<C>(0, 0), o2 = mk<C>(0, 0);
    if (w < 4) {
        const int im = mu == 0 ? nb.im[0] : mu == 1 ? nb.im[1] : mu == 2 ? nb.im[2] : nb.im[3];
        hop<R, true>(a.u[2 * mu + B], a.ph[2 * mu + B], a.in, sh, im, im, o0, o1, o2);
    } else {
        const int ip = mu == 0 ? nb.ip[0] : mu == 1 ? nb.ip[1] : mu == 2 ? nb.ip[2] : nb.ip[3];
        hop<R, false>(a.u[2 * mu + F], a.ph[2 * mu + F], a.in, sh, idx, ip, o0, o1, o2);
    }
    con[w][0][lane] = o0;
    con[w][1][lane] = o1;
    con[w][2][lane] = o2;
    __syncthreads();
    double dot = 0.0;
    if (w < 3 && live) {
        C o = con[0][w][lane];
#pragma unroll
        for (int h = 1; h < kSplitWaves; h++) o = cadd(o, con[h][w][lane]);
        const R half = (R)0.5;
        o.x *= half;
        o.y *= half;
        dot = dslash_out<R, MODE>(a, (long)w * sh + idx, o, x);
    }
    if (MODE >= kMdagMDot) block_partial_at<64 * kSplitWaves>(dot, 0.0, a.ctl.partials, blk);
}

// ---------------------------------------------------------------- launchers

// Where the hops are split over eight waves (k_dslash_split).  Small lattices
// leave most of the chip idle with a site per thread, and each thread waits for
// its hops in turn.  The pair D_oe, D_eo queued back to back, whole against
// split: FP64 11.7 -> 8.2 us at 2048 half-sites, 16.6 -> 9.4 at 16384, 23.8 ->
// 21.4 at 65536, but 41.1 -> 43.8 at 131072 and 157 -> 181 at 524288, where the
// exchange through LDS costs more than the shorter chain gives; the line is that of
// the fused solver iterations, so that a solver's sums have one order on either
// side of it.  FP32 11.7 -> 7.8
// at 2048, 25.7 -> 23.8 at 154440, 78.7 -> 74.5 at 524288 (half the bytes a site)
// and 243 -> 235 on 48^3 x 24 (1.3 million); then the gain goes: 361 -> 365 on
// 64^3 x 14, 378 -> 393 on 128 x 32^3, 380 -> 373 on 64^3 x 16, 688 -> 697 on
// 56^3 x 40, 826 -> 874 on 64^3 x 32.  Two or four waves a site lie between.
constexpr long kHopSplitSizehF32 = 3L << 19;
template <typename R>
static bool dslash_split() {
    return ctx().lat.sizeh <= (sizeof(R) == 4 ? kHopSplitSizehF32 : kHopSplitSizeh);
}
template <typename R>
int dslash_blocks() {
    return blocks_for(ctx().lat.sizeh, dslash_split<R>() ? kSplitSites : kBlock);
}
template int dslash_blocks<double>();
template int dslash_blocks<float>();

template <typename R, int EO, int MODE>
static void go(const DslashArgs<R>& a) {
    const dim3 blocks(dslash_blocks<R>());
    if (!dslash_split<R>()) {
        if constexpr (sizeof(R) == 8 && (MODE == kPlain || MODE == kMdagMDot))
            if (a.sg) {
                hipLaunchKernelGGL((k_dslash<R, EO, MODE, true>), blocks, dim3(kBlock), 0, ctx().stream, a);
                return;
            }
        hipLaunchKernelGGL((k_dslash<R, EO, MODE>), blocks, dim3(kBlock), 0, ctx().stream, a);
        return;
    }
    hipLaunchKernelGGL((k_dslash_split<R, EO, MODE>), blocks, dim3(64 * kSplitWaves), 0, ctx().stream, a);
}

template <typename R>
static bool fill_args(DslashArgs<R>& a, const void* u_dev, const void* ph_dev, const void* in_dev, void* out_dev) {
    const Lattice& L = ctx().lat;
    using C = typename Cplx<R>::T;
    const size_t su3 = sizeof(R) == 8 ? L.su3_bytes() : L.su3f_bytes();
    const size_t soa = sizeof(R) == 8 ? L.dsoa_bytes() : L.fsoa_bytes();
    for (int l = 0; l < 8; l++) {
        a.u[l] = (const C*)((const char*)u_dev + l * su3);
        a.ph[l] = (const R*)((const char*)ph_dev + l * soa);
    }
    a.in = (const C*)in_dev;
    a.out = (C*)out_dev;
    a.x = nullptr;
    a.m2 = 0.0;
    a.b = nullptr;
    a.rf = nullptr;
    a.sg = nullptr;
    a.g.nd0 = L.nd[0];
    a.g.nd0h = L.nd[0] / 2;
    a.g.nd1 = L.nd[1];
    a.g.nd2 = L.nd[2];
    a.g.nd3 = L.nd[3];
    a.g.sizeh = (int)L.sizeh;
    // t-fastest tiles need whole tiles per t-slice; used for FP64 only (no gain in FP32)
    const long s3 = L.sizeh / L.nd[3];
    a.tmajor = (sizeof(R) == 8 && s3 % (dslash_split<R>() ? kSplitSites : kBlock) == 0) ? 1 : 0;
    a.rev = ctx().dslash_serpentine ? (int)(ctx().dslash_launches++ & 1u) : 0;
    return true;
}

// Launch one Dslash on device pointers.  mode/fin select the fused epilogue.
template <typename R>
bool launch_dslash(int eo, int mode, int fin, const void* u, const void* ph, const void* in, void* out,
                   const void* x, double m2, const SolverCtl& ctl, const unsigned char* sg) {
    DslashArgs<R> a;
    fill_args<R>(a, u, ph, in, out);
    if (sg) a.sg = sg + eo * ctx().lat.sizeh;
    a.x = (const typename Cplx<R>::T*)x;
    a.m2 = m2;
    a.ctl = ctl;
    const int nb = dslash_blocks<R>();
    if (mode == kPlain) {
        if (eo == 0) go<R, 0, kPlain>(a); else go<R, 1, kPlain>(a);
    } else if (mode == kMdagM) {
        if (eo == 0) go<R, 0, kMdagM>(a); else go<R, 1, kMdagM>(a);
    } else {
        if (eo != 0) return fail("fused dot epilogue only on Deo");
        if (fin != kFinNone && fin != kFinStore && fin != kFinMsAlpha && fin != kFinFcgAlpha && fin != kFinMxmAlpha)
            return fail("unsupported dslash finalizer %d", fin);
        go<R, 0, kMdagMDot>(a);
    }
    if (!hip_ok(hipGetLastError(), "k_dslash launch")) return false;
    return mode == kMdagMDot && fin != kFinNone ? launch_finalize(fin, ctl, nb) : true;
}

template bool launch_dslash<double>(int, int, int, const void*, const void*, const void*, void*, const void*,
                                    double, const SolverCtl&, const unsigned char*);
template bool launch_dslash<float>(int, int, int, const void*, const void*, const void*, void*, const void*,
                                   double, const SolverCtl&, const unsigned char*);

// Signs of the hops.  A phase that is +-1 to rounding (its sine within two
// roundings of pi) is taken as its sign: 1 byte a half-site instead of 64 of
// the 928 a hop reads, and a hop without its rotation.  The solvers scan the
// phases once per solve where their hops are the ordinary ones (above
// kHopSplitSizeh, where a solve takes milliseconds against the scan's 30 us; the
// small lattices' iterations are not bound by bytes): 204 iterations with 19
// shifts on 32^4 42.28 -> 41.49 ms, a force of two systems on 32^3 x 8 6.50 -> 6.39.
struct SignArgs {
    const double* ph[8];
    SiteGeom g;
    unsigned char* sg;
    int* bad;
};
template <int EO>
__device__ __forceinline__ unsigned sign_bits(const SignArgs& a, int idx, bool& bad) {
    constexpr int F = EO == 0 ? 0 : 1, B = 1 - F;
    const Nbrs nb = site_neighbours<EO>(a.g, idx);
    unsigned bits = 0;
#pragma unroll
    for (int h = 0; h < 8; h++) {
        const int mu = h & 3;
        double s, c;
        phase_sincos(a.ph[2 * mu + (h < 4 ? B : F)][h < 4 ? nb.im[mu] : idx], &s, &c);
        if (!(fabs(s) <= 2.5e-16) || fabs(c) != 1.0) bad = true;
        bits |= c < 0.0 ? 1u << h : 0u;
    }
    return bits;
}
__global__ __launch_bounds__(kBlock) void k_phase_signs(SignArgs a) {
    const int idx = (int)blockIdx.x * kBlock + (int)threadIdx.x, sh = a.g.sizeh;
    if (idx >= sh) return;
    bool bad = false;
    a.sg[idx] = (unsigned char)sign_bits<0>(a, idx, bad);
    a.sg[sh + idx] = (unsigned char)sign_bits<1>(a, idx, bad);
    if (bad) *a.bad = 1;
}
static Workspace g_signs;
const unsigned char* phase_signs(const void* ph) {
    const Lattice& L = ctx().lat;
    const size_t n = (2 * (size_t)L.sizeh + 255) / 256 * 256;
    char* w = (char*)g_signs.try_get(n + 256);
    if (!w) return nullptr;
    SignArgs a;
    for (int l = 0; l < 8; l++) a.ph[l] = (const double*)((const char*)ph + l * L.dsoa_bytes());
    a.g.nd0 = L.nd[0];
    a.g.nd0h = L.nd[0] / 2;
    a.g.nd1 = L.nd[1];
    a.g.nd2 = L.nd[2];
    a.g.nd3 = L.nd[3];
    a.g.sizeh = (int)L.sizeh;
    a.sg = (unsigned char*)w;
    a.bad = (int*)(w + n);
    int bad = 1;
    if (!hip_ok(hipMemsetAsync(a.bad, 0, sizeof(int), ctx().stream), "phase signs")) return nullptr;
    hipLaunchKernelGGL(k_phase_signs, dim3(blocks_for(L.sizeh)), dim3(kBlock), 0, ctx().stream, a);
    if (!hip_ok(hipGetLastError(), "k_phase_signs") ||
        !hip_ok(hipMemcpyAsync(&bad, a.bad, sizeof(int), hipMemcpyDeviceToHost, ctx().stream), "phase signs") ||
        !hip_ok(hipStreamSynchronize(ctx().stream), "phase signs"))
        return nullptr;
    return bad ? nullptr : a.sg;
}

// The two hops of a reliable update: temp = Doe x, then r_f = (float)(b - M x)
// with the block partials of |r_f|^2.
bool launch_mdagm_resid(const void* u, const void* ph, const void* x, void* temp, const void* b, void* rf, double m2,
                        const SolverCtl& ctl) {
    if (!launch_dslash<double>(1, kPlain, kFinStore, u, ph, x, temp, nullptr, 0.0, ctl)) return false;
    DslashArgs<double> a;
    fill_args<double>(a, u, ph, temp, nullptr);
    a.x = (const double2*)x;
    a.m2 = m2;
    a.b = (const double2*)b;
    a.rf = (float2*)rf;
    a.ctl = ctl;
    go<double, 0, kMdagMResid>(a);
    return hip_ok(hipGetLastError(), "k_dslash launch");
}

// M = (m^2+shift) - Deo Doe on device pointers; temp receives Doe in.
template <typename R>
bool launch_mdagm(const void* u, const void* ph, const void* in, void* temp, void* out, double m2, int mode,
                  int fin, const SolverCtl& ctl) {
    if (!launch_dslash<R>(1, kPlain, kFinStore, u, ph, in, temp, nullptr, 0.0, ctl)) return false;
    return launch_dslash<R>(0, mode, fin, u, ph, temp, out, in, m2, ctl);
}

template bool launch_mdagm<double>(const void*, const void*, const void*, void*, void*, double, int, int,
                                   const SolverCtl&);
template bool launch_mdagm<float>(const void*, const void*, const void*, void*, void*, double, int, int,
                                  const SolverCtl&);

}  // namespace ostp

using namespace ostp;

// ------------------------------------------------------------ C entry points
static bool sync_ok(const char* what) { return entry_done(what); }

extern "C" {

static void dslash_entry(int eo, const void* u, void* out, const void* in, const void* backfield, int single,
                         const char* name) {
    if (!require_init(name)) return;
    const Lattice& L = ctx().lat;
    const size_t vb = single ? L.vec3f_bytes() : L.vec3_bytes();
    const size_t ub = 8 * (single ? L.su3f_bytes() : L.su3_bytes());
    const size_t pb = 8 * (single ? L.fsoa_bytes() : L.dsoa_bytes());
    const void* du = resolve(u, ub, name);
    const void* dp = resolve(backfield, pb, name);
    const void* di = resolve(in, vb, name);
    void* dout = resolve(out, vb, name);
    if (!du || !dp || !di || !dout) return;
    bool ok = single ? launch_dslash<float>(eo, kPlain, kFinStore, du, dp, di, dout, nullptr, 0.0, SolverCtl{})
                     : launch_dslash<double>(eo, kPlain, kFinStore, du, dp, di, dout, nullptr, 0.0, SolverCtl{});
    if (ok) sync_ok(name);
}

void acc_Deo(const su3_soa* u, vec3_soa* out, const vec3_soa* in, const double_soa* backfield) {
    dslash_entry(0, u, out, in, backfield, 0, "acc_Deo");
}
void acc_Doe(const su3_soa* u, vec3_soa* out, const vec3_soa* in, const double_soa* backfield) {
    dslash_entry(1, u, out, in, backfield, 0, "acc_Doe");
}
void acc_Deo_f(const su3_soa_f* u, vec3_soa_f* out, const vec3_soa_f* in, const float_soa* backfield) {
    dslash_entry(0, u, out, in, backfield, 1, "acc_Deo_f");
}
void acc_Doe_f(const su3_soa_f* u, vec3_soa_f* out, const vec3_soa_f* in, const float_soa* backfield) {
    dslash_entry(1, u, out, in, backfield, 1, "acc_Doe_f");
}

static void mdagm_entry(const void* u, void* out, const void* in, void* temp, const ferm_param* pars,
                        double shift, int single, const char* name) {
    if (!require_init(name)) return;
    if (!pars) { fail("%s: null ferm_param", name); return; }
    const Lattice& L = ctx().lat;
    const size_t vb = single ? L.vec3f_bytes() : L.vec3_bytes();
    const size_t ub = 8 * (single ? L.su3f_bytes() : L.su3_bytes());
    const size_t pb = 8 * (single ? L.fsoa_bytes() : L.dsoa_bytes());
    const void* ph = single ? (const void*)pars->phases_f : (const void*)pars->phases;
    const void* du = resolve(u, ub, name);
    const void* dp = resolve(ph, pb, name);
    const void* di = resolve(in, vb, name);
    void* dt = resolve(temp, vb, name);
    void* dout = resolve(out, vb, name);
    if (!du || !dp || !di || !dt || !dout) return;
    const double m2 = single ? pars->ferm_mass * pars->ferm_mass + (double)(float)shift
                             : pars->ferm_mass * pars->ferm_mass + shift;
    bool ok = single ? launch_mdagm<float>(du, dp, di, dt, dout, m2, kMdagM, kFinStore, SolverCtl{})
                     : launch_mdagm<double>(du, dp, di, dt, dout, m2, kMdagM, kFinStore, SolverCtl{});
    if (ok) sync_ok(name);
}

void fermion_matrix_multiplication(const su3_soa* u, vec3_soa* out, const vec3_soa* in, vec3_soa* temp1,
                                   ferm_param* pars) {
    mdagm_entry(u, out, in, temp1, pars, 0.0, 0, "fermion_matrix_multiplication");
}
void fermion_matrix_multiplication_shifted(const su3_soa* u, vec3_soa* out, const vec3_soa* in, vec3_soa* temp1,
                                           ferm_param* pars, double shift) {
    mdagm_entry(u, out, in, temp1, pars, shift, 0, "fermion_matrix_multiplication_shifted");
}
void fermion_matrix_multiplication_shifted_f(const su3_soa_f* u, vec3_soa_f* out, const vec3_soa_f* in,
                                             vec3_soa_f* temp1, ferm_param* pars, double shift) {
    mdagm_entry(u, out, in, temp1, pars, shift, 1, "fermion_matrix_multiplication_shifted_f");
}

double ostp_time_dslash(const void* u, void* out, const void* in, const void* phases, int eo, int single,
                        int reps) {
    if (!require_init("ostp_time_dslash")) return -1.0;
    const Lattice& L = ctx().lat;
    const size_t vb = single ? L.vec3f_bytes() : L.vec3_bytes();
    const void* du = resolve(u, 8 * (single ? L.su3f_bytes() : L.su3_bytes()), "ostp_time_dslash");
    const void* dp = resolve(phases, 8 * (single ? L.fsoa_bytes() : L.dsoa_bytes()), "ostp_time_dslash");
    const void* di = resolve(in, vb, "ostp_time_dslash");
    void* dout = resolve(out, vb, "ostp_time_dslash");
    if (!du || !dp || !di || !dout || reps <= 0) return -1.0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    double us = -1.0;
    if (hip_ok(hipEventCreate(&e0), "event") && hip_ok(hipEventCreate(&e1), "event") &&
        hip_ok(hipEventRecord(e0, ctx().stream), "event record")) {
        bool ok = true;
        for (int r = 0; r < reps && ok; r++)
            ok = single ? launch_dslash<float>(eo, kPlain, kFinStore, du, dp, di, dout, nullptr, 0.0, SolverCtl{})
                        : launch_dslash<double>(eo, kPlain, kFinStore, du, dp, di, dout, nullptr, 0.0, SolverCtl{});
        float ms = 0.f;
        if (ok && hip_ok(hipEventRecord(e1, ctx().stream), "event record") &&
            hip_ok(hipEventSynchronize(e1), "event sync") && hip_ok(hipEventElapsedTime(&ms, e0, e1), "elapsed"))
            us = 1000.0 * (double)ms / reps;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    return us;
}

}  // extern "C"
