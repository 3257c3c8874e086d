// The iteration of CG and CG-M on m^2 - D_eo D_oe in three launches, for one
// system or up to kKrSys that share the operator up to the mass.
//
// The scalar recurrences have no launches of their own: the kernel that needs
// a reduction's result sums the partials in every block (one wave per system,
// the same order in each block, so all blocks hold the same scalars) and
// block 0 alone stores the solver's state.  A state is kept twice: iteration j
// reads the copy j - 1 left and writes the other, so no block reads what
// block 0 of its own kernel writes.
//   k_kr_doe  ends iteration j - 1 (lambda, gamma, exit test, the shifts'
//             gammas and flags, the window's coefficients), then
//             h = D_oe p with p = r + gamma p formed at each neighbour
//   k_kr_deo  stores p = r + gamma p at its own sites, s = m2 p - D_eo h, <p, s>
//   k_kr_r    omega from <p, s>; r and (CG) x, |r|^2; the shifts' omegas, zetas
// (the reference: OpenAcc/inverter_full.c:71-105, inverter_multishift_full.c:
// 100-190; the per-shift expressions are those of finalize_ms_lanes).
//
// The hops of these kernels are split: a block takes 64 sites, one hop per
// wave, so that a small lattice fills the compute units and a site does not
// wait for its eight hops one after the other; the eight results are added in
// k_dslash's order.  Larger lattices form p in a kernel of its own (k_kr_p,
// which ends iteration j - 1 in k_kr_doe's place) between k_kr_r and the
// ordinary hop kernels (k_dslash, k_ms_multi_hop).
//
// Small lattices are bound by the chain of dependent waits inside a launch
// (state, partials, links, LDS: 3 to 5 us each), not by bytes, hence few
// launches with every load issued before the first wait.  41 CG iterations on
// 16^3 x 4: 1107 us with two hop kernels, two vector kernels and two one-block
// finalizers an iteration, 804 us so and 740 to 780 with the streaming kernels'
// sums over whole blocks; 52 CG-M iterations of order 9 on 12x14x10x6: 1855 ->
// 1196 us; a force of two systems on 32^3 x 8: 8.87 -> 8.04 ms; 204 iterations
// on 32^4, bound by the links' bytes: 44.6 -> 43.7 ms.
#pragma once

#include "ostp_dslash.h"

namespace ostp {

constexpr int kKrSys = 4;

// Window of CG-M iterations whose shift updates are applied at once (see
// k_msw_flush)
constexpr int kMsWinMax = 64;
constexpr int kMsWinRows = 40;  // whole passes of k_msw_flush: two of 20 shifts
static_assert(kMaxShifts <= kMsWinRows, "rows of the window coefficients");
struct MsWin {
    int t;                                  // iterations in the current window
    int first;                              // a solve's first: x_k and p_k not stored yet
    int active[kMaxShifts];                 // shift moved in this window
    double a[kMaxShifts], B[kMaxShifts];
    double c[kMsWinRows][kMsWinMax], D[kMsWinRows][kMsWinMax];
};

struct KrArgs {
    const double2* u[8];
    const double* ph[8];
    const unsigned char* sg;     // ordinary hops: signs of the hops, or null (phase_signs)
    SiteGeom g;
    const double2* r[kKrSys];    // residual after iteration j - 1
    double2* rn[kKrSys];         // k_kr_r: after iteration j (CG: the same array)
    double2* p[kKrSys];
    double2* h[kKrSys];
    double2* s[kKrSys];
    double2* x[kKrSys];          // CG
    double m2[kKrSys];
    SolverState* st[kKrSys];     // two copies: iteration j writes st[j & 1]
    double* partA[kKrSys];       // <p, s> per block of k_kr_deo
    double* partB[kKrSys];       // |r|^2 per block of k_kr_r
    MsWin* win[kKrSys];          // CG-M with windows
    double2* xs[kKrSys];         // CG-M without: the shifts' solutions and directions
    double2* ps[kKrSys];
    int nA, nB, sA;              // numbers of partials, stride of partA
    int j;                       // iteration, 1 for the first after a (re)start
    int ms;                      // CG-M
    int close;                   // k_kr_doe with one block: end iteration j - 1 only
    int n, tmajor, rev;
};

// sums of partials (part_sum): kr_wave a wave's total, kr_block the block's
__device__ __forceinline__ double kr_wave(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ double kr_block(double v, double (&lds)[kBlock / 64]) {
    v = kr_wave(v);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; w++) t += lds[w];
    return t;
}

// End of iteration j - 1 of system k by one wave: the new state (stored when
// `store`), *gamma and whether iteration j runs.  The window's coefficients
// are advanced by the storing block (per-shift values through sh).  total: |r|^2
// where the block has summed it already.
//
// The first launch of the next batch ends the iteration that a close has ended
// once more, from the copy that the close read: a running system's step is left
// to it.  A system that has finished takes its step in the close, which stores
// the final state in both copies, so that the launch finds it finished.
__device__ __forceinline__ void kr_end(const KrArgs& a, int k, int lane, bool store, double* gamma, int* running,
                                       double (*sh)[kMaxShifts], int* on, const double* total = nullptr) {
    SolverState* prev = a.st[k] + ((a.j - 1) & 1);
    // every load is issued before the first wait
    double sum = 0.0;
    if (a.j > 1 && !total) sum = part_sum(a.partB[k], a.nB, 1, lane);
    const int status0 = prev->status;
    int status = status0, cg = prev->cg, restarted = prev->cg_restarted, maxiter = prev->maxiter;
    double g = 0.0, delta = prev->delta, lambda = prev->lambda;
    const int order = prev->order;
    double zi = 0.0, zii = 0.0, ziii = 0.0, gk = 0.0, om_k = 0.0;
    int f = 0, moved = 0;
    if (a.ms && lane < order) {
        zi = prev->zeta_i[lane];
        zii = prev->zeta_ii[lane];
        ziii = prev->zeta_iii[lane];
        gk = prev->gammas[lane];
        om_k = prev->omegas[lane];
        f = prev->flags[0][lane];
    }
    if (a.j > 1 && status0 == kRunning) {
        lambda = total ? *total : kr_wave(sum);
        g = lambda / delta;
        cg += 1;
        if (a.ms) {
            const double target = prev->res * prev->safety;
            if (lane < order && f == 1) {
                moved = 1;
                gk = g * ziii * om_k / (zii * prev->omega);
                const double fact = sqrt(delta * zii * zii / prev->source_norm);
                if (fact < target) f = 0;
                zi = zii;
                zii = ziii;
            }
            const unsigned long long act = __ballot(lane < order && f == 1);
            maxiter = act ? 64 - __clzll(act) : 0;
            if (!(maxiter > 0 && cg < prev->max_cg)) status = kDone;
        } else {
            restarted += 1;
            const bool cont = (sqrt(lambda / prev->source_norm) > prev->res * prev->safety) && restarted < prev->restart_every;
            if (!cont) status = kInnerExit;
        }
        delta = lambda;
    }
    if (lane == 0) {
        *gamma = g;
        *running = status == kRunning;
    }
    if (!store) return;
    // the iteration that ended, its window step still to be taken by this block (or by the next launch,
    // when this one only closes a batch of a solver that goes on)
    const int ended = a.j > 1 && status0 == kRunning && !(a.close && status == kRunning);
    if (a.ms && lane < order) {
        sh[0][lane] = om_k;
        sh[1][lane] = gk;
        sh[2][lane] = ziii;
        on[lane] = moved;
    }
    if (lane == 0) on[kMaxShifts] = ended;
    auto put = [&](SolverState* next) {
        if (a.ms && lane < order) {
            next->zeta_i[lane] = zi;
            next->zeta_ii[lane] = zii;
            next->zeta_iii[lane] = ziii;
            next->gammas[lane] = gk;
            next->omegas[lane] = om_k;
            next->flags[0][lane] = f;
            next->flags[1][lane] = moved;  // in the iteration that ended
            next->shifts[lane] = prev->shifts[lane];
        }
        if (lane == 0) {
            next->delta = delta;
            next->lambda = lambda;
            next->gammag = g;
            next->alpha = prev->alpha;
            next->omega = prev->omega;
            next->omega_save = prev->omega_save;
            next->source_norm = prev->source_norm;
            next->res = prev->res;
            next->safety = prev->safety;
            next->cg = cg;
            next->cg_restarted = restarted;
            next->restart_every = prev->restart_every;
            next->max_cg = prev->max_cg;
            next->status = status;
            next->order = order;
            next->maxiter = maxiter;
            next->hold = ended;
        }
    };
    put(a.st[k] + (a.j & 1));
    if (a.close && status != kRunning) put(prev);
}

// window coefficients of the shifts that moved in iteration j - 1 (as k_msw_p)
__device__ __forceinline__ void kr_window(MsWin* w, int order, const double (*sh)[kMaxShifts], const int* on, int tid,
                                          int nt) {
    const int t = w->t;
    if (t >= kMsWinMax) return;  // the flushes come at W <= kMsWinMax: a row is never left
    const int per = t + 2;  // j < t, the new column t, and the scalar pair
    for (int e = tid; e < order * per; e += nt) {
        const int k = e / per, j = e - k * per;
        if (!on[k]) continue;
        const double om = sh[0][k], gk = sh[1][k];
        if (j < t) {
            w->c[k][j] = fma(-om, w->D[k][j], w->c[k][j]);
            w->D[k][j] *= gk;
        } else if (j == t) {
            w->D[k][t] = sh[2][k];
        } else {
            w->a[k] = fma(-om, w->B[k], w->a[k]);
            w->B[k] *= gk;
            w->active[k] = 1;
        }
    }
    __syncthreads();
    if (tid == 0) w->t = t + 1;
}

// The vector expressions below spell their fused multiply-adds out, so that
// the forms for one and for several systems round alike whatever the compiler
// would contract.
__device__ __forceinline__ double2 kr_mul(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ double2 kr_cross(double2 a, double2 b, double2 c, double2 d) {  // a b - c d
    const double2 p = kr_mul(a, b), q = kr_mul(c, d);
    return make_double2(p.x - q.x, p.y - q.y);
}
// one hop's link: rows 0,1 and the U(1) argument
struct KrLink {
    double2 a0, a1, a2, b0, b1, b2;
    double arg;
};
__device__ __forceinline__ void kr_link(const double2* __restrict__ U, const double* __restrict__ P, int sizeh, int iu,
                                        KrLink& l) {
    l.a0 = ld_link(U + iu);
    l.a1 = ld_link(U + sizeh + iu);
    l.a2 = ld_link(U + 2 * sizeh + iu);
    l.b0 = ld_link(U + 3 * sizeh + iu);
    l.b1 = ld_link(U + 4 * sizeh + iu);
    l.b2 = ld_link(U + 5 * sizeh + iu);
    l.arg = ld_link(P + iu);
}
// the link with its third row's conjugate x and phase, and its action (hop<double, DAG>'s arithmetic)
struct KrHop {
    double2 x0, x1, x2, phase;
};
__device__ __forceinline__ void kr_prepare(const KrLink& l, bool dag, KrHop& q) {
    double s, c;
    phase_sincos(l.arg, &s, &c);
    q.phase = make_double2(c, dag ? -s : s);
    q.x0 = kr_cross(l.a1, l.b2, l.a2, l.b1);
    q.x1 = kr_cross(l.a2, l.b0, l.a0, l.b2);
    q.x2 = kr_cross(l.a0, l.b1, l.a1, l.b0);
}
__device__ __forceinline__ void kr_apply(const KrLink& l, const KrHop& q, bool dag, double2 v0, double2 v1, double2 v2,
                                         double2 (&o)[3]) {
    v0 = kr_mul(v0, q.phase);
    v1 = kr_mul(v1, q.phase);
    v2 = kr_mul(v2, q.phase);
    if (!dag) {
        o[0] = cfma(l.a2, v2, cfma(l.a1, v1, kr_mul(l.a0, v0)));
        o[1] = cfma(l.b2, v2, cfma(l.b1, v1, kr_mul(l.b0, v0)));
        o[2] = cfmac(q.x2, v2, cfmac(q.x1, v1, kr_mul(cconj(q.x0), v0)));
    } else {
        o[0] = cfma(q.x0, v2, cfmac(l.b0, v1, kr_mul(cconj(l.a0), v0)));
        o[1] = cfma(q.x1, v2, cfmac(l.b1, v1, kr_mul(cconj(l.a1), v0)));
        o[2] = cfma(q.x2, v2, cfmac(l.b2, v1, kr_mul(cconj(l.a2), v0)));
    }
}
// p = r + gamma p (k_cg_p's expression)
__device__ __forceinline__ double2 kr_p(double2 r, double2 p, double g) {
    return make_double2(fma(p.x, g, r.x), fma(p.y, g, r.y));
}

constexpr int kKrSites = 64, kKrThreads = 512;  // of a block of the split hops

__device__ __forceinline__ int kr_site(const KrArgs& a, int blk, int sites, int lane) {
    if (a.tmajor) {
        const int s3 = a.g.sizeh / a.g.nd3;
        const int tile = blk / a.g.nd3, tt = blk - tile * a.g.nd3;
        return tt * s3 + tile * sites + lane;
    }
    return blk * sites + lane;
}

__device__ __forceinline__ constexpr int kr_owner(int k, int c) { return (3 * k + c) & 7; }

// The eight hops of the block's sites for the active systems: out(k, col, site
// index, value) receives every system's sum of hops, halved.  load(k, iv, v):
// system k's input at half-site iv.
template <int EO, int NR, class Load, class Early, class Ready, class Out>
__device__ __forceinline__ void kr_hops(const KrArgs& a, int blk, Load load, Early early, Ready ready, Out out) {
    constexpr int F = EO == 0 ? 0 : 1, B = 1 - F;
    const int tid = (int)threadIdx.x, sh = a.g.sizeh;
    __shared__ double2 con[NR][8][3][64];
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int idx = kr_site(a, blk, kKrSites, lane);
    const bool live = idx < sh;
    const Nbrs nb = site_neighbours<EO>(a.g, live ? idx : 0);
    const bool dag = w < 4;
    const int mu = w & 3;
    const int im = mu == 0 ? nb.im[0] : mu == 1 ? nb.im[1] : mu == 2 ? nb.im[2] : nb.im[3];
    const int ip = mu == 0 ? nb.ip[0] : mu == 1 ? nb.ip[1] : mu == 2 ? nb.ip[2] : nb.ip[3];
    const int iu = dag ? im : (live ? idx : 0), iv = dag ? im : ip;
    const int arr = 2 * mu + (dag ? B : F);
    KrLink l;
    kr_link(a.u[arr], a.ph[arr], sh, iu, l);
    const auto raw = load.raw(iv);
    // the owners' own-site operands as well
#pragma unroll
    for (int k = 0; k < NR; k++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            if (w == kr_owner(k, c)) early(k, c, live ? idx : 0);
    if (!ready()) return;
    KrHop q;
    kr_prepare(l, dag, q);
#pragma unroll
    for (int k = 0; k < NR; k++) {
        double2 v[3], o[3];
        load.get(raw, k, v);
        kr_apply(l, q, dag, v[0], v[1], v[2], o);
#pragma unroll
        for (int c = 0; c < 3; c++) con[k][w][c][lane] = o[c];
    }
    __syncthreads();
    // one colour of one system per wave (wave kr_owner)
#pragma unroll
    for (int k = 0; k < NR; k++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if (w != kr_owner(k, c)) continue;
            double2 o = make_double2(0.0, 0.0);
#pragma unroll
            for (int i = 0; i < 4; i++) o = csub(o, con[k][i][c][lane]);
#pragma unroll
            for (int i = 4; i < 8; i++) o = cadd(o, con[k][i][c][lane]);
            if (live) out(k, c, idx, make_double2(0.5 * o.x, 0.5 * o.y));
        }
}

template <int NR>
__global__ __launch_bounds__(kKrThreads) void k_kr_doe(KrArgs a) {
    __shared__ double sh_gamma[NR];
    __shared__ int sh_run[NR], sh_on[NR][kMaxShifts + 1];
    __shared__ double sh_k[NR][3][kMaxShifts];
    const int tid = (int)threadIdx.x;
    const bool store = blockIdx.x == 0;
    auto ready = [&]() {
        const int w = tid >> 6;
        if (w < NR && w < a.n) kr_end(a, w, tid & 63, store, &sh_gamma[w], &sh_run[w], sh_k[w], sh_on[w]);
        if (w == 0 && (tid & 63) < NR && (tid & 63) >= a.n) sh_run[tid & 63] = 0;
        __syncthreads();
        if (store && a.ms)
#pragma unroll 1
            for (int k = 0; k < a.n; k++)
                if (sh_on[k][kMaxShifts] && a.win[k]) kr_window(a.win[k], a.st[k][a.j & 1].order, sh_k[k], sh_on[k], tid, kKrThreads);
        bool any = false;
#pragma unroll
        for (int k = 0; k < NR; k++) any = any || sh_run[k];
        return any && !a.close;
    };
    if (a.close) {
        ready();
        return;
    }
    struct Raw {
        double2 r[NR][3], p[NR][3];
    };
    struct Load {
        const KrArgs& a;
        const double* gamma;
        __device__ Raw raw(int iv) const {
            Raw v;
#pragma unroll
            for (int k = 0; k < NR; k++) {
                const int q = k < a.n ? k : 0;
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    v.r[k][c] = a.r[q][(long)c * a.g.sizeh + iv];
                    v.p[k][c] = a.p[q][(long)c * a.g.sizeh + iv];
                }
            }
            return v;
        }
        __device__ void get(const Raw& w, int k, double2 (&v)[3]) const {
#pragma unroll
            for (int c = 0; c < 3; c++) v[c] = kr_p(w.r[k][c], w.p[k][c], gamma[k]);
        }
    };
    const int blk = xcd_block_id_dir(a.rev);
    kr_hops<1, NR>(a, blk, Load{a, sh_gamma}, [](int, int, int) {}, ready, [&](int k, int c, int idx, double2 v) {
        if (!sh_run[k]) return;
        a.h[k][(long)c * a.g.sizeh + idx] = v;
    });
}

template <int NR>
__global__ __launch_bounds__(kKrThreads) void k_kr_deo(KrArgs a) {
    __shared__ double wsum[NR][3];
    const int tid = (int)threadIdx.x, w = tid >> 6, lane = tid & 63;
    double gamma[NR], dot[NR];
    bool run[NR];
    bool any = false;
#pragma unroll
    for (int k = 0; k < NR; k++) {
        const SolverState* st = a.st[k < a.n ? k : 0] + (a.j & 1);
        run[k] = k < a.n && st->status == kRunning;
        gamma[k] = st->gammag;
        any = any || run[k];
        dot[k] = 0.0;
    }
    double2 er[NR], ep[NR];  // the own-site r and p of the colour this wave finishes
    struct Raw {
        double2 h[NR][3];
    };
    struct Load {
        const KrArgs& a;
        __device__ Raw raw(int iv) const {
            Raw v;
#pragma unroll
            for (int k = 0; k < NR; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) v.h[k][c] = a.h[k < a.n ? k : 0][(long)c * a.g.sizeh + iv];
            return v;
        }
        __device__ void get(const Raw& w, int k, double2 (&v)[3]) const {
#pragma unroll
            for (int c = 0; c < 3; c++) v[c] = w.h[k][c];
        }
    };
    const int blk = xcd_block_id_dir(a.rev);
    auto early = [&](int k, int c, int idx) {
        const long i = (long)c * a.g.sizeh + idx;
        const int q = k < a.n ? k : 0;
        er[k] = a.r[q][i];
        ep[k] = a.p[q][i];
    };
    kr_hops<0, NR>(a, blk, Load{a}, early, [&]() { return any; }, [&](int k, int c, int idx, double2 v) {
        if (!run[k]) return;
        const long i = (long)c * a.g.sizeh + idx;
        const double2 p = kr_p(er[k], ep[k], gamma[k]);
        a.p[k][i] = p;
        const double2 s = make_double2(fma(p.x, a.m2[k], -v.x), fma(p.y, a.m2[k], -v.y));
        a.s[k][i] = s;
        dot[k] = fma(p.x, s.x, fma(p.y, s.y, dot[k]));
    });
    if (!any) return;
    // the waves' sums, one colour each
#pragma unroll
    for (int k = 0; k < NR; k++) {
        double v = dot[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
#pragma unroll
        for (int c = 0; c < 3; c++)
            if (lane == 0 && w == kr_owner(k, c)) wsum[k][c] = v;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NR; k++)
        if (tid == k && run[k]) {
            a.partA[k][blk] = wsum[k][0] + wsum[k][1] + wsum[k][2];
        }
}

// The streaming kernels: blockIdx.y = system, blocks over the half-sites in
// strides; the operands of a thread's first two sites (of its one site, where
// the grid covers the lattice) are loaded before the block waits for its scalars.
constexpr int kKrAhead = 2;

// End of iteration j - 1 and p = r + gamma p
__global__ __launch_bounds__(kBlock) void k_kr_p(KrArgs a) {
    __shared__ double sh_gamma, sh_k[3][kMaxShifts], lds[kBlock / 64];
    __shared__ int sh_run, sh_on[kMaxShifts + 1];
    const int k = (int)blockIdx.y, tid = (int)threadIdx.x, sh = a.g.sizeh;
    const bool store = blockIdx.x == 0;
    const int i0 = (int)blockIdx.x * kBlock + tid, step = (int)gridDim.x * kBlock;
    const double2* r = a.r[k];
    double2* p = a.p[k];
    double2 rr[kKrAhead][3], pp[kKrAhead][3];
#pragma unroll
    for (int q = 0; q < kKrAhead; q++) {
        if (q * step >= sh) break;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + (i0 + q * step < sh ? i0 + q * step : 0);
            rr[q][c] = r[e];
            pp[q][c] = p[e];
        }
    }
    const double total = kr_block(a.j > 1 ? part_sum<kBlock>(a.partB[k], a.nB, 1, tid) : 0.0, lds);
    if (tid < 64) kr_end(a, k, tid, store, &sh_gamma, &sh_run, sh_k, sh_on, &total);
    __syncthreads();
    if (store && a.ms && sh_on[kMaxShifts] && a.win[k]) kr_window(a.win[k], a.st[k][a.j & 1].order, sh_k, sh_on, tid, kBlock);
    if (!sh_run || a.close) return;
    const double g = sh_gamma;
#pragma unroll
    for (int q = 0; q < kKrAhead; q++)
        if (i0 + q * step < sh)
#pragma unroll
            for (int c = 0; c < 3; c++) p[(long)c * sh + i0 + q * step] = kr_p(rr[q][c], pp[q][c], g);
    for (int i = i0 + kKrAhead * step; i < sh; i += step)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + i;
            p[e] = kr_p(r[e], p[e], g);
        }
}

// Without windows: the shifts that moved in the iteration that has just ended,
// x_k -= omega_k p_k ; p_k = gamma_k p_k + zeta_k r; blockIdx.y = system.
__global__ __launch_bounds__(kBlock) void k_kr_shifts(KrArgs a, long n3) {
    const int q = (int)blockIdx.y;
    const SolverState* st = a.st[q] + (a.j & 1);
    if (!st->hold) return;
    const long i = (long)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n3) return;
    const double2 rr = a.r[q][i];
    for (int k = 0; k < st->order; k++) {
        if (!st->flags[1][k]) continue;
        const double om = st->omegas[k], gk = st->gammas[k], zk = st->zeta_iii[k];
        double2 *xk = a.xs[q] + k * n3, *pk = a.ps[q] + k * n3;
        const double2 pv = pk[i], xv = xk[i];
        xk[i] = make_double2(xv.x - om * pv.x, xv.y - om * pv.y);
        pk[i] = make_double2(gk * pv.x + zk * rr.x, gk * pv.y + zk * rr.y);
    }
}

// omega and the vectors' step
template <int MS>
__global__ __launch_bounds__(kBlock) void k_kr_r(KrArgs a) {
    const int k = (int)blockIdx.y, tid = (int)threadIdx.x, lane = tid & 63, sh = a.g.sizeh;
    SolverState* st = a.st[k] + (a.j & 1);
    __shared__ double lds[kBlock / 64];
    __shared__ double sh_om;
    __shared__ int sh_run;
    const int i0 = (int)blockIdx.x * kBlock + tid, step = (int)gridDim.x * kBlock;
    const double2 *r = a.r[k], *s = a.s[k], *p = a.p[k];
    double2 *rn = a.rn[k], *x = a.x[k];
    double2 ra[kKrAhead][3], sa[kKrAhead][3], pa[kKrAhead][3], xa[kKrAhead][3];
#pragma unroll
    for (int q = 0; q < kKrAhead; q++) {
        if (q * step >= sh) break;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + (i0 + q * step < sh ? i0 + q * step : 0);
            ra[q][c] = r[e];
            sa[q][c] = s[e];
            if (!MS) {
                pa[q][c] = p[e];
                xa[q][c] = x[e];
            }
        }
    }
    const double tot = kr_block(part_sum<kBlock>(a.partA[k], a.nA, a.sA, tid), lds);
    if (tid < 64) {
        const double delta = st->delta;
        const int running = st->status == kRunning;
        const double om = MS ? -delta / tot : delta / tot;
        if (lane == 0) {
            sh_om = om;
            sh_run = running;
        }
        if (blockIdx.x == 0 && running) {
            const double omega_save = st->omega, gammag = st->gammag;
            if (MS && lane < st->maxiter && st->flags[0][lane] == 1) {
                const double zi = st->zeta_i[lane], zii = st->zeta_ii[lane];
                const double ziii = (zi * zii * omega_save) /
                                    (om * gammag * (zi - zii) + zi * omega_save * (1.0 - (st->shifts[lane]) * om));
                st->zeta_iii[lane] = ziii;
                st->omegas[lane] = om * ziii / zii;
            }
            if (lane == 0) {
                st->alpha = tot;
                st->omega_save = omega_save;
                st->omega = om;
            }
        }
    }
    __syncthreads();
    if (!sh_run) return;
    const double om = sh_om;
    double v = 0.0;
    auto one = [&](long e, double2 rr, double2 ss, double2 pp, double2 xx) {
        double2 n;
        if (MS) {
            n = make_double2(fma(om, ss.x, rr.x), fma(om, ss.y, rr.y));
        } else {
            x[e] = make_double2(fma(pp.x, om, xx.x), fma(pp.y, om, xx.y));
            n = make_double2(fma(ss.x, -om, rr.x), fma(ss.y, -om, rr.y));
        }
        rn[e] = n;
        v = fma(n.x, n.x, fma(n.y, n.y, v));
    };
#pragma unroll
    for (int q = 0; q < kKrAhead; q++)
        if (i0 + q * step < sh)
#pragma unroll
            for (int c = 0; c < 3; c++)
                one((long)c * sh + i0 + q * step, ra[q][c], sa[q][c], MS ? ra[q][c] : pa[q][c], MS ? ra[q][c] : xa[q][c]);
    for (int i = i0 + kKrAhead * step; i < sh; i += step)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + i;
            one(e, r[e], s[e], MS ? r[e] : p[e], MS ? r[e] : x[e]);
        }
    const double t = block_sum<kBlock>(v, lds);  // (the barrier above lies after every read of lds)
    if (tid == 0) a.partB[k][blockIdx.x] = t;
}

// ---- mixed-precision CG with reliable updates (inverter_mixedp.c:54-155) ----
// FP32 iterations in four launches: k_mx_p ends iteration j - 1 and forms p,
// the two ordinary FP32 hops follow, k_mx_xr takes the step.  Whether iteration
// j is a reliable update is known when it starts (delta against the largest
// since the last one), so its k_mx_xr adds the step to x instead and the FP64
// residual comes from two predicated launches, queued after every
// kMxTailEvery-th iteration only: an update that falls between two of them
// pauses the solver (hold) until the next.  79 iterations on 32^3 x 8: 4370
// us with nine launches each, four of them for an update that seldom came, 3747
// so, 3630 to 3650 with sums over whole blocks (21 us an iteration in the FP32
// hops, 10 in these two kernels).
// Every iteration, second, third, fourth: 3.72, 3.66, 3.62, 3.88 ms on 32^3 x 8,
// 2.12, 1.68 to 1.98, 1.90, 2.06 on 16^3 x 8 (predicated launches that do nothing
// against iterations that wait).
constexpr int kMxTailEvery = 2;
struct MxArgs {
    float2 *pf, *rf, *outf;
    const float2* sf;
    double2* x;
    SolverState* st;      // two copies, as KrArgs
    const double* partA;  // <p, s>, two doubles a block
    double* partB;        // |r|^2 of k_mx_xr
    const double* partT;  // |r|^2 of a reliable update, two doubles a block
    int nA, nB, nT, sizeh;
    int j, close;
    int tail;             // the update's launches were queued after iteration j - 1
};

// p = r + gamma p in the precision of k_cg_p<float2>
__device__ __forceinline__ float2 mx_p(float2 r, float2 p, double g) {
    return make_float2((float)((double)p.x * g + (double)r.x), (float)((double)p.y * g + (double)r.y));
}

__global__ __launch_bounds__(kBlock) void k_mx_p(MxArgs a) {
    __shared__ double sh_gamma, lds[kBlock / 64], ldst[kBlock / 64];
    __shared__ int sh_run;
    const int tid = (int)threadIdx.x, sh = a.sizeh;
    const int i0 = (int)blockIdx.x * kBlock + tid, step = (int)gridDim.x * kBlock;
    float2 rr[kKrAhead][3], pp[kKrAhead][3];
#pragma unroll
    for (int q = 0; q < kKrAhead; q++) {
        if (q * step >= sh) break;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + (i0 + q * step < sh ? i0 + q * step : 0);
            rr[q][c] = a.rf[e];
            pp[q][c] = a.pf[e];
        }
    }
    const double sumt = a.tail ? kr_block(part_sum<kBlock>(a.partT, a.nT, 2, tid), ldst) : 0.0;
    const double sum = kr_block(a.j > 1 ? part_sum<kBlock>(a.partB, a.nB, 1, tid) : 0.0, lds);
    if (tid < 64) {
        const SolverState* prev = a.st + ((a.j - 1) & 1);
        SolverState* next = a.st + (a.j & 1);
        double delta = prev->delta, lambda = prev->lambda, g = 0.0, last = prev->last_max_res;
        int status = prev->status, cg = prev->cg, rus = prev->ru_count, ru = prev->ru;
        const bool hold = a.j > 1 && status == kRunning && ru && !a.tail;
        if (a.j > 1 && status == kRunning && !hold) {
            lambda = ru ? sumt : sum;
            g = lambda / delta;
            delta = lambda;
            cg += 1;
            if (ru) {
                last = 0.0;
                rus += 1;
            }
            const bool cont = (sqrt(lambda / prev->source_norm) > prev->res * prev->safety) && cg < prev->max_cg;
            if (!cont) status = kDone;
        }
        if (status == kRunning && !hold) {
            if (last < delta) last = delta;
            ru = (delta < prev->mixed_delta * last) ? 1 : 0;
        }
        if (tid == 0) {
            sh_gamma = g;
            sh_run = status == kRunning && !hold;
            if (blockIdx.x == 0) {
                next->delta = delta;
                next->lambda = lambda;
                next->gammag = g;
                next->alpha = prev->alpha;
                next->omega = prev->omega;
                next->source_norm = prev->source_norm;
                next->res = prev->res;
                next->safety = prev->safety;
                next->last_max_res = last;
                next->mixed_delta = prev->mixed_delta;
                next->cg = cg;
                next->max_cg = prev->max_cg;
                next->status = status;
                next->ru = ru;
                next->hold = hold;
                next->ru_count = rus;
            }
        }
    }
    __syncthreads();
    if (!sh_run || a.close) return;
    const double g = sh_gamma;
#pragma unroll
    for (int q = 0; q < kKrAhead; q++)
        if (i0 + q * step < sh)
#pragma unroll
            for (int c = 0; c < 3; c++) a.pf[(long)c * sh + i0 + q * step] = mx_p(rr[q][c], pp[q][c], g);
    for (int i = i0 + kKrAhead * step; i < sh; i += step)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + i;
            a.pf[e] = mx_p(a.rf[e], a.pf[e], g);
        }
}

// out_f += omega p_f; then either r_f -= omega s_f with |r_f|^2, or (reliable
// update) x += out_f, out_f = 0   (inverter_mixedp.c:107-134)
__global__ __launch_bounds__(kBlock) void k_mx_xr(MxArgs a) {
    SolverState* st = a.st + (a.j & 1);
    __shared__ double lds[kBlock / 64];
    __shared__ double sh_om;
    __shared__ int sh_go, sh_ru;
    const int tid = (int)threadIdx.x, sh = a.sizeh;
    const int i0 = (int)blockIdx.x * kBlock + tid, step = (int)gridDim.x * kBlock;
    float2 pa[kKrAhead][3], oa[kKrAhead][3], ra[kKrAhead][3], sa[kKrAhead][3];
#pragma unroll
    for (int q = 0; q < kKrAhead; q++) {
        if (q * step >= sh) break;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + (i0 + q * step < sh ? i0 + q * step : 0);
            pa[q][c] = a.pf[e];
            oa[q][c] = a.outf[e];
            ra[q][c] = a.rf[e];
            sa[q][c] = a.sf[e];
        }
    }
    const double tot = kr_block(part_sum<kBlock>(a.partA, a.nA, 2, tid), lds);
    if (tid < 64) {
        const int go = st->status == kRunning && !st->hold, ru = st->ru;
        const double om = st->delta / tot;
        if (tid == 0) {
            sh_om = om;
            sh_go = go;
            sh_ru = ru;
            if (blockIdx.x == 0 && go) {
                st->alpha = tot;
                st->omega = om;
            }
        }
    }
    __syncthreads();
    if (!sh_go) return;
    const double om = sh_om;
    const int ru = sh_ru;
    double v = 0.0;
    auto one = [&](long e, float2 pp, float2 oo, float2 rr, float2 ss) {
        const float2 on =
            make_float2((float)((double)pp.x * om + (double)oo.x), (float)((double)pp.y * om + (double)oo.y));
        if (ru) {
            const double2 xx = a.x[e];
            a.x[e] = make_double2(xx.x + (double)on.x, xx.y + (double)on.y);
            a.outf[e] = make_float2(0.f, 0.f);
            return;
        }
        const float2 rn =
            make_float2((float)((double)ss.x * (-om) + (double)rr.x), (float)((double)ss.y * (-om) + (double)rr.y));
        a.outf[e] = on;
        a.rf[e] = rn;
        v += (double)rn.x * rn.x + (double)rn.y * rn.y;
    };
#pragma unroll
    for (int q = 0; q < kKrAhead; q++)
        if (i0 + q * step < sh)
#pragma unroll
            for (int c = 0; c < 3; c++)
                one((long)c * sh + i0 + q * step, pa[q][c], oa[q][c], ra[q][c], sa[q][c]);
    for (int i = i0 + kKrAhead * step; i < sh; i += step)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const long e = (long)c * sh + i;
            one(e, a.pf[e], a.outf[e], a.rf[e], a.sf[e]);
        }
    const double t = block_sum<kBlock>(v, lds);
    if (tid == 0) a.partB[blockIdx.x] = t;
}

}  // namespace ostp
