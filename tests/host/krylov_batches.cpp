// The kernels of ostp_krylov.h on the CPU, launched in the order of kr_iterate
// (solvers.hip): systems of a group with batches that end anywhere against
// each system by itself in one batch.  Prints one line per case:
//   form window stops... : agree   (windows, states and residuals bit for bit)
#include "ostp_krylov.h"

using namespace ostp;

namespace {

constexpr int kN = 4, kSizeh = kN * kN * kN * kN / 2, kN3 = 3 * kSizeh;

struct Rng {
    uint64_t s;
    double next() {  // splitmix64, in (-1, 1)
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return (double)(int64_t)(z ^ (z >> 31)) / 9223372036854775808.0;
    }
};

using Vec = std::vector<double2>;
struct Field {
    Vec u[8];
    std::vector<double> ph[8];
};

// links with orthonormal rows 0 and 1, phases of any size
Field field() {
    Field f;
    Rng r{7};
    for (int l = 0; l < 8; l++) {
        f.u[l].resize(9 * kSizeh);
        f.ph[l].resize(kSizeh);
        for (int i = 0; i < kSizeh; i++) {
            double2 m[2][3];
            for (auto& row : m)
                for (auto& e : row) e = make_double2(r.next(), r.next());
            for (int a = 0; a < 2; a++) {
                if (a) {
                    double2 d = make_double2(0, 0);
                    for (int c = 0; c < 3; c++) d = cadd(d, cmulc(m[0][c], m[1][c]));
                    for (int c = 0; c < 3; c++) m[1][c] = csub(m[1][c], cmul(d, m[0][c]));
                }
                double n = 0;
                for (int c = 0; c < 3; c++) n += m[a][c].x * m[a][c].x + m[a][c].y * m[a][c].y;
                for (int c = 0; c < 3; c++) f.u[l][(size_t)(3 * a + c) * kSizeh + i] = cscale(m[a][c], 1 / sqrt(n));
            }
            f.ph[l][i] = 3 * r.next();
        }
    }
    return f;
}

struct Sys {
    int order, max_cg;
    double m2;
    Vec b;
};

// what a system leaves: every window that was applied to the solutions (the
// last one as it stands), the residuals it read, the state
struct Left {
    std::vector<MsWin> wins;
    std::vector<double2> resid;
    SolverState st;
};

std::vector<Left> solve(const Field& f, const std::vector<Sys>& sy, bool split, int W, const std::vector<int>& batches) {
    const int n = (int)sy.size(), nb = split ? kSizeh / kKrSites : (kSizeh + kBlock - 1) / kBlock, nr = 1;
    std::vector<Vec> r(n), h(n, Vec(kN3)), s(n, Vec(kN3)), p(n), hist(n, Vec((size_t)W * kN3));
    std::vector<SolverState> st(2 * n);
    std::vector<MsWin> win(n);
    std::vector<std::vector<double>> pa(n, std::vector<double>(2 * nb)), pb(n, std::vector<double>(nr));
    std::vector<Left> left(n);
    KrArgs a{};
    for (int l = 0; l < 8; l++) {
        a.u[l] = f.u[l].data();
        a.ph[l] = f.ph[l].data();
    }
    a.g = SiteGeom{kN / 2, kN, kN, kN, kN, kSizeh};
    a.n = n;
    a.ms = 1;
    a.nA = nb;
    a.nB = nr;
    a.sA = split ? 1 : 2;
    memset(win.data(), 0, n * sizeof(MsWin));
    memset(st.data(), 0, 2 * n * sizeof(SolverState));
    auto reset = [&](int k) {
        memset(&win[k], 0, sizeof(MsWin));
        for (int i = 0; i < kMaxShifts; i++) win[k].B[i] = 1.0;
    };
    for (int k = 0; k < n; k++) {
        r[k] = p[k] = sy[k].b;
        reset(k);
        SolverState& q = st[2 * k];
        for (const double2& e : sy[k].b) q.source_norm += e.x * e.x + e.y * e.y;
        q.delta = q.source_norm;
        q.res = 1e-300;  // stopped by max_cg
        q.safety = 0.95;
        q.max_cg = sy[k].max_cg;
        q.omega = 1.0;
        q.order = q.maxiter = sy[k].order;
        for (int i = 0; i < q.order; i++) {
            q.flags[0][i] = 1;
            q.zeta_i[i] = q.zeta_ii[i] = 1.0;
            q.shifts[i] = 0.05 * (i + 1);
        }
        a.p[k] = p[k].data();
        a.h[k] = h[k].data();
        a.s[k] = s[k].data();
        a.m2[k] = sy[k].m2;
        a.st[k] = &st[2 * k];
        a.partA[k] = pa[k].data();
        a.partB[k] = pb[k].data();
        a.win[k] = &win[k];
    }
    auto residual = [&](int k, int j) { return j ? hist[k].data() + (size_t)((j - 1) % W) * kN3 : r[k].data(); };
    auto apply = [&](int k) {  // k_msw_flush: what it reads
        left[k].wins.push_back(win[k]);
        const int t = std::min(win[k].t, W);
        left[k].resid.insert(left[k].resid.end(), hist[k].begin(), hist[k].begin() + (size_t)t * kN3);
    };
    auto first = [&]() {
        const unsigned blocks = a.close ? 1 : split ? nb : nr;
        if (!split) hostblock::launch(dim3(blocks, n), kBlock, [&]() { k_kr_p(a); });
        else if (n == 1) hostblock::launch(dim3(blocks), kKrThreads, [&]() { k_kr_doe<1>(a); });
        else if (n == 2) hostblock::launch(dim3(blocks), kKrThreads, [&]() { k_kr_doe<2>(a); });
        else hostblock::launch(dim3(blocks), kKrThreads, [&]() { k_kr_doe<kKrSys>(a); });
    };
    auto hops = [&]() {
        if (split) {
            if (n == 1) hostblock::launch(dim3(nb), kKrThreads, [&]() { k_kr_deo<1>(a); });
            else if (n == 2) hostblock::launch(dim3(nb), kKrThreads, [&]() { k_kr_deo<2>(a); });
            else hostblock::launch(dim3(nb), kKrThreads, [&]() { k_kr_deo<kKrSys>(a); });
            return;
        }
        // the ordinary hop kernels
        for (int k = 0; k < n; k++) {
            if (a.st[k][a.j & 1].status != kRunning) continue;
            double2 o0, o1, o2;
            for (int i = 0; i < kSizeh; i++) {
                dslash_site<double, 1>(a.u, a.ph, p[k].data(), a.g, i, o0, o1, o2);
                h[k][i] = o0;
                h[k][kSizeh + i] = o1;
                h[k][2 * kSizeh + i] = o2;
            }
            double dot = 0;
            for (int i = 0; i < kSizeh; i++) {
                dslash_site<double, 0>(a.u, a.ph, h[k].data(), a.g, i, o0, o1, o2);
                const double2 o[3] = {o0, o1, o2};
                for (int c = 0; c < 3; c++) {
                    const double2 x = p[k][c * kSizeh + i];
                    const double2 v = csub(cscale(x, sy[k].m2), o[c]);
                    s[k][c * kSizeh + i] = v;
                    dot += x.x * v.x + x.y * v.y;
                }
            }
            pa[k][0] = dot;
        }
    };
    int j = 0;
    for (size_t batch = 0;; batch++) {
        for (int i = 0; i < batches[std::min(batch, batches.size() - 1)]; i++) {
            a.j = ++j;
            a.close = 0;
            for (int k = 0; k < n; k++) {
                a.r[k] = residual(k, j - 1);
                a.rn[k] = residual(k, j);
            }
            first();
            if (j > 1 && (j - 1) % W == 0)
                for (int k = 0; k < n; k++) {
                    if (win[k].t < W) continue;
                    apply(k);
                    reset(k);
                }
            hops();
            hostblock::launch(dim3(nr, n), kBlock, [&]() { k_kr_r<1>(a); });
        }
        a.j = j + 1;
        a.close = 1;
        for (int k = 0; k < n; k++) a.r[k] = residual(k, j);
        first();
        bool running = false;
        for (int k = 0; k < n; k++) running = running || st[2 * k + (a.j & 1)].status == kRunning;
        if (!running) break;
    }
    for (int k = 0; k < n; k++) {
        if (win[k].t) apply(k);
        left[k].st = st[2 * k + (a.j & 1)];
    }
    return left;
}

bool same(const Left& a, const Left& b, int order) {
    if (a.wins.size() != b.wins.size() || a.resid.size() != b.resid.size() || a.st.cg != b.st.cg ||
        a.st.delta != b.st.delta || a.st.status != b.st.status)
        return false;
    for (size_t i = 0; i < a.wins.size(); i++) {
        const MsWin &x = a.wins[i], &y = b.wins[i];
        if (x.t != y.t) return false;
        for (int k = 0; k < order; k++)
            if (x.active[k] != y.active[k] || x.a[k] != y.a[k] || x.B[k] != y.B[k] || memcmp(x.c[k], y.c[k], sizeof x.c[k]) ||
                memcmp(x.D[k], y.D[k], sizeof x.D[k]))
                return false;
    }
    return !memcmp(a.resid.data(), b.resid.data(), a.resid.size() * sizeof(double2));
}

}  // namespace

int main() {
    const Field f = field();
    Rng r{3};
    std::vector<Sys> all;
    for (int k = 0; k < 4; k++) {
        Sys s{2 + k % 2, 0, 0.3 + 0.1 * k, Vec(kN3)};
        for (double2& e : s.b) e = make_double2(r.next(), r.next());
        all.push_back(s);
    }
    const std::vector<int> batches = {8, 4, 16};  // ends at 8, 12, 28, 44
    const int sets[][5] = {{2, 7, 20},  {2, 8, 20},  {2, 9, 20},  {2, 12, 13},     {2, 12, 40},     {2, 28, 44},
                           {2, 16, 30}, {2, 20, 8},  {2, 12, 12}, {3, 8, 12, 20},  {3, 28, 12, 29}, {4, 8, 8, 12, 30},
                           {4, 1, 28, 44, 45}};
    for (int split = 0; split < 2; split++)
        for (int W : {4, 5, 64})
            for (const auto& stops : sets) {
                const int n = stops[0];
                std::vector<Sys> sy(all.begin(), all.begin() + n);
                for (int k = 0; k < n; k++) sy[k].max_cg = stops[1 + k];
                const std::vector<Left> got = solve(f, sy, split, W, batches);
                bool ok = true;
                for (int k = 0; k < n; k++) {
                    const Left one = solve(f, {sy[k]}, split, W, {sy[k].max_cg})[0];
                    ok = ok && one.st.cg == stops[1 + k] && same(got[k], one, sy[k].order);
                }
                printf("%s %d", split ? "split" : "plain", W);
                for (int k = 0; k < n; k++) printf(" %d", stops[1 + k]);
                printf(" : %s\n", ok ? "agree" : "differ");
                fflush(stdout);
            }
    // a window that is full takes no further step
    static MsWin full, kept;
    static double v[3][kMaxShifts];
    static int on[kMaxShifts + 1];
    full.t = kMsWinMax;
    for (int k = 0; k < 4; k++) on[k] = 1, full.D[k][0] = full.B[k] = v[0][k] = v[1][k] = v[2][k] = 1.5;
    kept = full;
    hostblock::launch(dim3(1), 64, [&]() { kr_window(&full, 4, v, on, (int)threadIdx.x, 64); });
    printf("full : %s\n", memcmp(&full, &kept, sizeof full) ? "differ" : "agree");
    return 0;
}
