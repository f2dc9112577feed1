// layout_check.hip -- host checks of the sizes and indices that the host plans
// launches by against what the device reads and writes by them
// (cusr_amd/csrc/program.h, launch_plan.h). Built and run by tests/test_layout.py with the
// check's name; prints "layout ok".
#include <malloc.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <thread>
#include <vector>

#include "../cusr_amd/csrc/launch_plan.h"
#include "../cusr_amd/csrc/program.h"

using namespace cusr;

#define CHECK(c)                                        \
    do {                                                \
        if (!(c)) {                                     \
            printf("%s fails at line %d\n", #c, __LINE__); \
            exit(1);                                    \
        }                                               \
    } while (0)

// A population built tree by tree; operators and leaves in prefix order.
struct Pop {
    std::vector<int32_t> nt, ci;
    std::vector<float> nv;
    std::vector<TreeMeta> metas;
    PopHeader h = {};
    std::vector<uint64_t> prog;
    std::vector<ExprDesc> desc;
    Plan plan = {};

    void op(int f, bool binary) {
        nt.push_back(binary ? NODE_BFUNC : NODE_UFUNC);
        nv.push_back((float)f);
        ci.push_back(-1);
        metas.back().n_nodes++;
    }
    void var(int v) {
        nt.push_back(NODE_VAR);
        nv.push_back((float)v);
        ci.push_back(-1);
        metas.back().n_nodes++;
    }
    void con() {
        nt.push_back(NODE_CONST);
        nv.push_back(0.0f);
        ci.push_back(metas.back().K++);
        metas.back().n_nodes++;
        h.total_c++;
    }
    void tree() { metas.push_back({(int32_t)nt.size(), 0, h.total_c, 0}); }
    int decode(int N, int D, int k_max) {
        h.magic = POP_MAGIC;
        h.version = POP_VERSION;
        h.M_prob = (int)metas.size();
        h.total_nodes = (int)nt.size();
        h.N = N;
        h.n_vars = D;
        h.K_max = k_max;
        prog.assign(staged_words_max(h.total_nodes, D), 0);
        desc.assign(metas.size(), ExprDesc{});
        const int rc = check_header(&h, nt.data(), nv.data(), ci.data(), metas.data());
        return rc != CO_OK ? rc
                           : decode_range(&h, nt.data(), nv.data(), ci.data(), metas.data(), 0,
                                          h.M_prob, 0, prog.data(), desc.data(), &plan);
    }
};

// sin(c) * x with k constants summed under the sine: a C program of k operators
static void sine_of_constants(Pop &p, int k) {
    p.tree();
    p.op(OP_MUL, true);
    p.op(OP_SIN, false);
    for (int i = 1; i < k; i++) p.op(OP_ADD, true);
    for (int i = 0; i < k; i++) p.con();
    p.var(0);
}

// An evaluation's scalar area holds every expression's constants and slots, with
// a header that claims fewer constants than the expressions have, or none.
static void check_eval() {
    for (int k_max : {0, 1, 8, 20})
        for (int D : {1, 12}) {
            Pop p;
            sine_of_constants(p, 3);
            sine_of_constants(p, 20);
            p.tree();
            p.var(0);
            CHECK(p.decode(1024, D, k_max) == CO_OK);
            const int room = eval_uni_doubles(p.plan);
            bool any = false;
            for (const ExprDesc &d : p.desc) {
                if (d.n_c == 0) continue;
                any = true;
                CHECK(uni_at(d.K, 0, d.cslots, 0).size <= room);
            }
            CHECK(any);
        }
    Pop none;
    none.tree();
    none.op(OP_MUL, true);
    none.con();
    none.var(0);
    CHECK(none.decode(1024, 1, 1) == CO_OK);
    CHECK(eval_uni_doubles(none.plan) == 0);
}

// The damped solve's loads stay within its sums and the kSolveBefore entries that
// every kernel holds before them: at every K of the kernel whose K is
// known at run time only (the sums laid out by it), and for every group of K
// bins in a padded kernel (laid out by the kernel's K).
static void check_solve() {
    auto loads = [](int KM, int KL, int Kr) {
        for (int g = 0; g * kSolveCols < Kr; g++)
            for (int j = g * kSolveCols; j < (g + 1) * kSolveCols && j < KM; j++)
                for (int i = 0; i < Kr; i++) {
                    const int at = sums_row(KL, j) + i;
                    CHECK(at >= -kSolveBefore && at < sums_width(KL));
                    // a column that is used holds its own entries
                    if (j < Kr && i >= j) {
                        int q = 1 + KL;
                        for (int a = 0; a < j; a++) q += KL - a;
                        CHECK(at == q + i - j);
                    }
                }
        for (int i = 0; i < Kr; i++) CHECK(sums_row(KL, i) + i < sums_width(KL));
    };
    for (int K = 1; K <= CO_MAX_K; K++) loads(CO_MAX_K, K, K);
    for (int top = 1; top <= CO_FAST_MAX_K; top++)
        for (int K = 1; K <= top; K++) loads(top, top, K);
}

// Plans the decoded population's launches at the default options of its N.
static int plan(const Pop &p, bool rev, bool mixed, int parts, std::vector<LaunchPlan> &lp,
                bool group = true) {
    PlanArgs a = {};
    a.rev = rev;
    a.mixed = mixed;
    a.split = parts > CO_MAX_PARTITIONS;
    a.group = group;
    a.N = p.h.N;
    a.parts = a.seg_parts[0] = parts;
    a.nseg = 1;
    a.lds_per_block = 160 << 10;
    lp.resize(CO_BINS);
    int nl = 0, kmax = 0;
    const int rc = plan_launches(p.desc.data(), 0, p.h.M_prob, a, lp.data(), &nl, &kmax);
    lp.resize(rc == CO_OK ? nl : 0);
    return rc;
}

// Every launch's scalar area holds its expressions' constants, the tangents that
// its kernel reads (its own K of them, padded and general kernels too), the
// slots and the tape; rows of one point for the rest of the launch's LDS.
static void check_scalars() {
    for (int N : {60, 1024, 70000})
        for (int D : {1, 12})
            for (bool vars : {false, true}) {
                Pop p;
                for (int k : {1, 1, 2, 3, 4, 5, 7, 9, 11, 12, 13, 15, 16, 20, 32}) {
                    if (vars) {
                        sine_of_constants(p, k);
                        continue;
                    }
                    // constants alone: a scalar area and no rows beside it
                    p.tree();
                    p.op(OP_SIN, false);
                    for (int i = 1; i < k; i++) p.op(OP_ADD, true);
                    for (int i = 0; i < k; i++) p.con();
                }
                CHECK(p.decode(N, D, 32) == CO_OK);
                for (int parts : {1, 4, 8})
                    for (int mode = 0; mode < 8; mode++) {
                        const bool rev = mode & 1, mixed = mode & 2, group = mode & 4;
                        std::vector<LaunchPlan> lp;
                        CHECK(plan(p, rev, mixed, parts, lp, group) == CO_OK);
                        int n = 0;
                        for (const LaunchPlan &b : lp) {
                            for (int q = b.pos; q < b.pos + b.cnt; q++, n++) {
                                const ExprDesc &d = p.desc[q];
                                CHECK(b.bin == CO_GENERAL_BIN ? d.gen : !d.gen && d.K <= b.bin);
                                if (d.n_c == 0) continue;
                                const int t0 = rev ? 0 : kernel_k(b);
                                const UniAt at = uni_at(d.K, t0, d.cslots, rev ? d.ctape : 0);
                                CHECK(at.t0 >= d.K && at.slot - at.t0 >= t0);
                                const int ub = b.bin == CO_GENERAL_BIN
                                                   ? uni_bytes_of(d, rev, kGenK) : uni_bytes(b);
                                CHECK(at.size * (int)sizeof(double) <= ub);
                                CHECK(ub + (rev ? d.rows_rev : d.rows) * 256 <= (int)b.wave_bytes);
                            }
                        }
                        CHECK(n == p.h.M_prob);
                    }
            }
}

// Rows (variables and spill slots) and reverse-AD tape of the plain programs, the
// largest of each over the population.
static void plain_lds(const Pop &p, int *rows, int *tape) {
    std::vector<uint64_t> w(2 * p.nt.size());
    std::vector<int32_t> off(p.metas.size());
    CHECK(decode_population(&p.h, p.nt.data(), p.nv.data(), p.ci.data(), p.metas.data(), w.data(),
                            nullptr, nullptr, nullptr, off.data(), nullptr) == CO_OK);
    int slots = 0;
    *tape = 0;
    for (size_t m = 0; m < p.metas.size(); m++) {
        int t = 0;
        for (int k = 0; k < p.metas[m].n_nodes; k++) {
            const uint64_t a = w[off[m] + 2 * k];
            t += (int)(a >> 39 & 1) + (int)(a >> 40 & 1);
            if (a >> 27 & 1 && (int)(a >> 28 & 255) + 1 > slots) slots = (int)(a >> 28 & 255) + 1;
        }
        if (t > *tape) *tape = t;
    }
    *rows = p.h.n_vars + slots;
}

// A sum of K constants times functions of x, some of them subtrees of variables
// alone (v of them), and one subtree of constants alone.
static void sum_with_subtrees(Pop &p, int K, int v, int D) {
    p.tree();
    for (int i = 0; i < K; i++) p.op(OP_ADD, true);
    p.op(OP_MUL, true);
    p.op(OP_EXP, false);
    p.op(OP_SIN, false);
    p.op(OP_MUL, true);
    p.con();
    p.con();
    p.var(0);
    for (int i = 2; i < K + 2; i++) {
        if (i < K) {
            p.op(OP_MUL, true);
            p.con();
        }
        if (i - 2 < v) {
            p.op(i & 1 ? OP_SIN : OP_COS, false);
            p.op(OP_SQUARE, false);
        }
        p.var(i % D);
    }
}

// A population of the general kernel whose plain programs fit the LDS is planned,
// whatever staging adds to one expression's rows beside another's tape; the
// planned bytes hold every expression.
static void check_limit() {
    const size_t limit = 160 << 10;
    int at_limit = 0;
    for (int D : {1, 2, 12, 60})
        for (int parts : {1, 2, 4, 8})
            for (int mode = 0; mode < 4; mode++)
                for (int v : {0, 3, 12})
                    for (int slack = 0; slack < 6; slack++) {
                        const bool rev = mode & 1, mixed = mode & 2;
                        const size_t row = 64 * (mixed ? 4 : 8);
                        const int sp = parts > CO_MAX_PARTITIONS ? 1 : parts;
                        const size_t fixed = fit_static_lds(CO_GENERAL_BIN) + kGenJtBytes +
                                             (sp > 1 ? sp * sums_width(20) * 8 : 0);
                        Pop p;
                        sum_with_subtrees(p, 20, v, D);
                        sum_with_subtrees(p, 17, v / 2, D);
                        // a chain whose tape takes what is left, down to a slot of slack
                        p.h.N = 1000;
                        p.h.n_vars = D;
                        const int rows0 = D + 1;
                        const int chain = (int)((limit - fixed) / row) - rows0 - slack;
                        p.tree();
                        for (int i = 0; i < chain; i++) p.op(i & 1 ? OP_SIN : OP_COS, false);
                        p.op(OP_MUL, true);
                        p.con();
                        p.var(0);
                        CHECK(p.decode(1000, D, 20) == CO_OK);
                        int rows, tape;
                        plain_lds(p, &rows, &tape);
                        if (!rev) tape = 0;
                        size_t was = (size_t)(rows + tape) * row;
                        if (mixed && was < (size_t)rows * 512) was = (size_t)rows * 512;
                        was += fixed;
                        std::vector<LaunchPlan> lp;
                        const int rc = plan(p, rev, mixed, parts, lp);
                        CHECK(was > limit || rc == CO_OK);
                        at_limit += rev && was <= limit && was + 8 * row > limit;
                        if (rc != CO_OK) continue;
                        CHECK(lp[0].bin == CO_GENERAL_BIN && lp[0].cnt >= 2);
                        CHECK(lp[0].lds[0] + fit_static_lds(CO_GENERAL_BIN) <= limit);
                        for (const ExprDesc &d : p.desc) {
                            if (!d.gen) continue;   // a chain of at most 255 nodes
                            const size_t r = rev ? d.rows_rev : d.rows, t = rev ? d.tape : 0;
                            const size_t need = uni_bytes_of(d, rev, kGenK) + kGenJtBytes;
                            CHECK(need + (r + t) * row <= lp[0].wave_bytes);
                            CHECK(!mixed || need + r * 512 <= lp[0].wave_bytes);
                        }
                    }
    CHECK(at_limit > 50);
}

// Staging is linear in the nodes: a sum of n sines of variables, far more values than
// the rows hold, and the same over 40 of 100 variables, which M reads itself too.
static void check_long() {
    auto seconds = [](Pop &p, int D) {
        const auto t0 = std::chrono::steady_clock::now();
        CHECK(p.decode(1024, D, 1) == CO_OK);
        return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    };
    for (int D : {1, 100}) {
        const int used = D == 1 ? 1 : 40;
        double s[2];
        for (int big = 0; big < 2; big++) {
            Pop p;
            p.tree();
            const int n = big ? 64000 : 2000;
            for (int i = 0; i < n; i++) {
                p.op(OP_ADD, true);
                p.op(OP_SIN, false);
                p.var(i % used);
                if (i % 50 == 49) {
                    p.op(OP_ADD, true);
                    p.var(i / 50 % used);
                }
            }
            p.con();
            s[big] = std::min(seconds(p, D), std::min(seconds(p, D), seconds(p, D)));
            CHECK(p.desc[0].vrows > 0 && p.desc[0].rows <= std::max(D + 1, 8));
        }
        printf("D %d: %.1f ms for 32 times %.2f ms\n", D, 1e3 * s[1], 1e3 * s[0]);
        CHECK(s[1] < 32 * 5 * s[0] + 0.02);   // quadratic: 1,024 times
    }
}

// Kernel, launch order and columns of a population around the fast kernels' bounds:
// chains right and left of a stack depth of 16 (31 and 33 nodes), K 0 to 20.
static void check_order() {
    Pop p;
    srand(7);
    for (int m = 0; m < 6000; m++) {
        p.tree();
        const int depth = 14 + rand() % 5, K = rand() % 21;
        for (int i = 1; i < depth; i++) p.op(OP_ADD, true);   // depth leaves stack up
        for (int i = 0; i < depth; i++) {
            const bool sine = rand() % 4 == 0;
            if (sine) p.op(OP_SIN, false);
            if (i < K) p.con();
            else p.var(0);
        }
    }
    CHECK(p.decode(1000, 1, 32) == CO_OK);
    std::vector<int32_t> route(p.metas.size()), v_col(p.metas.size()), vrows(p.metas.size());
    CHECK(decode_population(&p.h, p.nt.data(), p.nv.data(), p.ci.data(), p.metas.data(), nullptr,
                            nullptr, nullptr, nullptr, nullptr, route.data()) == CO_OK);
    int gen = 0;
    for (int32_t r : route) gen += r;
    CHECK(gen == p.plan.n_gen && gen > 500 && gen < 5500);
    int rows = 0, ck = 0;
    for (size_t q = 0; q < p.desc.size(); q++) {
        const ExprDesc &d = p.desc[q];
        CHECK(d.gen == route[d.y_row] && d.gen == (q < (size_t)gen));
        if (q > 0 && d.gen == p.desc[q - 1].gen) CHECK(d.K <= p.desc[q - 1].K);
        CHECK(d.K == p.metas[d.y_row].K && d.c_off == p.metas[d.y_row].c_offset);
        v_col[d.y_row] = d.v_col;
        vrows[d.y_row] = d.vrows;
        rows = std::max(rows, d.rows);
        if (d.n_c > 0) ck = std::max(ck, d.K);
    }
    CHECK(rows == p.plan.max_rows && ck == p.plan.max_ck);
    int64_t cols = 0;
    for (size_t m = 0; m < v_col.size(); m++) {
        CHECK(v_col[m] == cols);
        cols += vrows[m];
    }
    CHECK(cols == p.plan.vcols && cols > 0);
}

// What a thread keeps of its decodes is bounded: the working arrays of 400,000
// expressions (48 MB) are given back.
static void check_kept() {
    Pop p;
    for (int m = 0; m < 400000; m++) {
        p.tree();
        p.op(OP_ADD, true);
        p.con();
        p.var(0);
    }
    CHECK(p.decode(100, 1, 1) == CO_OK);   // the pool's threads, the outputs' arrays
    const auto used = [] {
        const struct mallinfo2 i = mallinfo2();
        return (double)(i.uordblks + i.hblkhd);
    };
    double kept = 0.0;
    std::thread([&] {
        const double before = used();
        Plan plan = {};
        CHECK(decode_range(&p.h, p.nt.data(), p.nv.data(), p.ci.data(), p.metas.data(), 0,
                           p.h.M_prob, 0, p.prog.data(), p.desc.data(), &plan) == CO_OK);
        kept = used() - before;
    }).join();
    printf("kept %.1f MB\n", kept / 1e6);
    CHECK(kept < 4e6);
}

int main(int argc, char **argv) {
    CHECK(argc == 2);
    if (!strcmp(argv[1], "eval")) check_eval();
    else if (!strcmp(argv[1], "solve")) check_solve();
    else if (!strcmp(argv[1], "scalars")) check_scalars();
    else if (!strcmp(argv[1], "limit")) check_limit();
    else if (!strcmp(argv[1], "long")) check_long();
    else if (!strcmp(argv[1], "order")) check_order();
    else if (!strcmp(argv[1], "kept")) check_kept();
    else CHECK(!"check's name");
    puts("layout ok");
    return 0;
}
