// Calls of the library on the fake device of fake_device.cpp: what they do
// when memory runs out, and what a solve that fails leaves.  Prints one line
// per check, "name : ok" or what went wrong.
#include "ostp_krylov.h"

#include <string>

using namespace ostp;

extern "C" {
extern size_t fake_capacity, fake_used;
int fake_is_live(const void* p);
void on_launch(const char* kernel, void** args);
}

namespace {
bool solves_end = true;
int stop, iterations;        // (not 0) a CG converges in that many; launched
std::string gone;            // kernels that were given memory that is no longer there
int tiles, links;            // launches of the gauge force's plane and per-link kernels
int with_qa, with_hops;      // launches that took a kept QA; that formed D_oe of solutions

void* arg(void** args, int i) {
    void* p;
    memcpy(&p, args[i], sizeof p);
    return p;
}
void used(const char* kernel, const void* p) {
    if (!fake_is_live(p)) gone += std::string(" ") + kernel;
}
}  // namespace

extern "C" void on_launch(const char* kernel, void** args) {
    const std::string k = kernel;
    auto is = [&](const char* s) { return k.find(s) != std::string::npos; };
    if (is("k_kr_doe") || is("k_kr_p")) {
        const KrArgs& a = *(const KrArgs*)args[0];
        for (int q = 0; q < a.n; q++) {
            used("k_kr", a.p[q]);
            if (a.win[q]) used("k_kr_win", a.rn[q] ? a.rn[q] : a.r[q]);
            if (stop) {
                const SolverState& prev = a.st[q][(a.j - 1) & 1];
                SolverState next = prev;
                if (prev.status == kRunning && a.j > 1) {
                    next.cg = a.j - 1;
                    next.delta = next.lambda = prev.source_norm * pow(prev.res * prev.safety, 2.0 * next.cg / stop);
                    if (next.cg >= stop) next.status = kInnerExit;
                }
                a.st[q][a.j & 1] = next;
                iterations += !a.close;
                continue;
            }
            if (!solves_end) a.st[q][a.j & 1] = a.st[q][(a.j - 1) & 1];
            for (int c = 0; c < 2 && a.close && solves_end; c++) {
                a.st[q][c].status = kDone;
                a.st[q][c].cg = 1;
            }
        }
    } else if (is("k_finalize")) {
        ((const SolverCtl*)args[0])->st->sum = 1.0;
    } else if (is("k_direct_product_sites")) {  // aux, stride, xs, hs
        used("k_direct_product", arg(args, 0));
        used("k_direct_product", arg(args, 2));
        used("k_direct_product", arg(args, 3));
    } else if (is("k_qa_lambda")) {  // links, S', stride, QA, Lambda
        used("k_qa_lambda", arg(args, 3));
        used("k_qa_lambda", arg(args, 4));
        with_qa += is("ILb1E") ? 1 : 0;
    } else if (is("k_sigma")) {
        used("k_sigma", arg(args, 1));
        used("k_sigma", arg(args, 2));
    } else if (is("k_gf_tile")) {  // records, links, parts
        tiles++;
        used("k_gf_tile", arg(args, 0));
        used("k_gf_tile", arg(args, 2));
    } else if (is("k_gauge_force")) {
        links++;
    } else if (is("k_ms_verifyILi1E")) {
        // u[8], ph[8], x[8], m2[8], n, h
        const char* v = (const char*)args[0];
        void* h;
        memcpy(&h, v + 32 * 8 + 8, sizeof h);
        used("k_ms_verify", h);
        with_hops++;
    }
}

namespace {

constexpr int kShape[4] = {8, 8, 8, 8};
constexpr size_t kSh = 2048, kGauge = 8 * 144 * kSh, kVec = 48 * kSh, kIp = 8 * 64 * kSh;
constexpr int kOrder = 4;

struct Fields {
    char *u, *arr, *gl3, *ip, *taux, *mom, *chi, *xs, *sf, *ph;
    vec3_soa* w[4];
    ferm_param fp[2] = {};
    Fields() {
        ostp_set_abort_on_error(0);
        ostp_init(kShape[0], kShape[1], kShape[2], kShape[3], 0);
        ostp_set_stout(0.15, 2, 0.0, 0, 0, 1);
        auto get = [](size_t n) { return (char*)ostp_malloc(n); };
        u = get(kGauge), arr = get(2 * kGauge), gl3 = get(kGauge), taux = get(kGauge);
        ip = get(kIp), mom = get(kIp), chi = get(2 * kVec), xs = get(kOrder * kVec), sf = get(kOrder * kVec);
        ph = get(64 * kSh);
        for (auto& p : w) p = (vec3_soa*)get(kVec);
        for (int f = 0; f < 2; f++) {
            fp[f].ferm_mass = 0.1 + f;
            fp[f].number_of_ps = 1;
            fp[f].index_of_the_first_ps = f;
            fp[f].phases = (double_soa*)ph;
            fp[f].approx_md.approx_order = kOrder;
            for (int k = 0; k < kOrder; k++) fp[f].approx_md.RA_b[k] = 0.1 * (k + 1);
        }
    }
    void gauge_force() {
        ostp_set_gauge_force_kernel(2);  // whose work space this is about
        ostp_time_gauge_force((su3_soa*)u, nullptr, (tamat_soa*)ip, (thmat_soa*)mom, 0.1, 1);
    }
    void force() {
        inverter_package p = {};
        p.u = (su3_soa*)u;
        p.ferm_shift_temp = (vec3_soa*)sf;
        p.nshifts = kOrder;
        p.loc_r = w[0], p.loc_h = w[1], p.loc_s = w[2], p.loc_p = w[3];
        fermion_force_soloopenacc((su3_soa*)u, (su3_soa*)arr, (su3_soa*)gl3, (tamat_soa*)ip, fp, 2, (vec3_soa*)chi, 1e-9,
                                  (su3_soa*)taux, (vec3_soa*)xs, p, 100);
    }
    int multishift() {
        int cg = 0;
        return multishift_invert((su3_soa*)u, &fp[0], &fp[0].approx_md, (vec3_soa*)xs, (vec3_soa*)chi, 1e-9, w[0], w[1],
                                 w[2], w[3], (vec3_soa*)sf, 100, &cg);
    }
};

// what went wrong since the last call, or "ok"
const char* verdict() {
    static std::string s;
    s = ostp_last_error();
    if (s.empty()) s = gone.empty() ? "ok" : "gone:" + gone;
    ostp_clear_error();
    gone.clear();
    return s.c_str();
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argv[1];
    Fields f;
    const size_t base = fake_used;
    if (what == "given_back") {
        // The gauge force's work space first; the memory that is left beside it is too little for the call.
        f.gauge_force();
        const size_t held = fake_used - base;
        printf("work space : %s\n", held == 288 * 8 * kSh ? "ok" : "none");
        auto tight = [&](const char* name, auto call) {
            f.gauge_force();  // holds its work space again
            fake_capacity = fake_used + 64;
            call();
            fake_capacity = (size_t)1 << 40;
            printf("%s : %s\n", name, verdict());
        };
        tight("caller", [&] { ostp_free(ostp_malloc(held / 2)); });
        tight("tables", [&] {
            std::vector<int> a(8 * kSh), b(8 * kSh);
            ostp_compute_nnp_and_nnm(a.data(), b.data());
        });
        ostp_set_multishift_window(16);
        tight("window", [&] { f.multishift(); });
        ostp_set_multishift_window(0);
        tight("again", [&] { f.gauge_force(); });
    } else if (what == "refused") {
        // Free memory of four times the links' records and a little less than four times the force's parts on
        // top: the parts are refused, the per-link kernel takes the call, and nothing stays allocated.
        const size_t rec = 96 * 8 * kSh, part = 2 * rec;
        fake_capacity = fake_used + rec + 4 * part - 64;
        f.gauge_force();
        printf("refused : %s\n", fake_used == base ? verdict() : "kept");
        fake_capacity += 64;
        f.gauge_force();
        printf("taken : %s\n", fake_used == base + rec + part ? verdict() : "not kept");
    } else if (what == "force") {
        // A gauge force, then a fermion force, in the memory given: the bytes it took, whether the levels' QA and
        // the solutions' D_oe were kept to the end, and whether all went well.
        fake_capacity = base + strtoull(argv[2], nullptr, 0);
        ostp_set_multishift_window(8);
        if (argc > 3) f.gauge_force();
        f.force();
        printf("force %zu %d %d : %s\n", fake_used - base, with_qa == 2, with_hops == 2, verdict());
    } else if (what == "failed_solve") {
        solves_end = false;  // the state does not advance: an error
        for (int w : {0, 1}) {
            ostp_set_multishift_window(w);
            ostp_memset(f.xs, 1, kOrder * kVec);
            const int st = f.multishift();
            bool zero = st == 0 && *ostp_last_error();
            ostp_clear_error();
            for (size_t i = 0; i < kOrder * kVec; i++) zero = zero && !f.xs[i];
            printf("window %d : %s\n", w, zero ? "ok" : "old solutions");
        }
    } else if (what == "gauge") {
        // launches of the two kernels: a force with its staples, one without, the integrator's
        ostp_init(atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), atoi(argv[5]), 0);
        ostp_set_stout(0.15, 2, 0.0, 0, 0, atoi(argv[6]));
        ostp_set_gauge_force_kernel(atoi(argv[7]));
        const size_t sh = ostp_sizeh();
        su3_soa *u = (su3_soa*)ostp_malloc(8 * 144 * sh), *s = (su3_soa*)ostp_malloc(8 * 144 * sh);
        tamat_soa* ip = (tamat_soa*)ostp_malloc(512 * sh);
        thmat_soa* mom = (thmat_soa*)ostp_malloc(512 * sh);
        md_param md = {};
        md.no_md = 1, md.gauge_scale = 5, md.t = 1.0;
        md_parameters = md;
        initialize_md_global_variables(md);
        auto count = [&](const char* name, auto call) {
            tiles = links = 0;
            call();
            printf("%s : %d %d %s\n", name, tiles, links, verdict());
        };
        count("staples", [&] { calc_ipdot_gauge_soloopenacc(u, s, ip); });
        count("force", [&] { ostp_time_gauge_force(u, nullptr, ip, nullptr, 0.0, 1); });
        count("moves", [&] { multistep_2MN_gauge(u, s, ip, mom); });
    } else if (what == "short") {
        // CG solves that take few iterations: how many were queued
        ostp_init(16, 16, 16, 2 * strtol(argv[2], nullptr, 0), 0);  // half-sites: 4096 each
        const size_t sh = ostp_sizeh();
        char* big[7];
        for (auto& p : big) p = (char*)ostp_malloc(48 * sh);
        const su3_soa* u = (su3_soa*)ostp_malloc(8 * 144 * sh);
        ferm_param fp = f.fp[0];
        fp.phases = (double_soa*)ostp_malloc(64 * sh);
        for (stop = 1; stop <= 12; stop++) {
            int cg = 0;
            iterations = 0;
            auto v = [&](int k) { return (vec3_soa*)big[k]; };
            ker_invert_openacc(u, &fp, v(0), v(1), 1e-9, v(2), v(3), v(4), v(5), 100, 0.0, &cg);
            printf("%d %d : %d\n", stop, iterations, cg);
        }
    }
    return 0;
}
