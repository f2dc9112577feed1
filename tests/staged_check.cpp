// staged_check.cpp -- host check of the staged programs (cusr_amd/csrc/program.h)
// against the plain ones: random expressions of both formats are decoded both
// ways, and a scalar interpreter with the device's rules runs each program.
// Value, tangents and adjoints must be bit-identical, every index a word holds
// must lie within the descriptor's rows, slots and tapes (which size the
// device's LDS), every row must be written before it is read, and no operator
// may be lost or run twice. Built and run by tests/test_staged.py; prints
// "staged ok".
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <random>
#include <vector>

#include "../cusr_amd/csrc/program.h"

using namespace cusr;

#define CHECK(c)                                                             \
    do {                                                                     \
        if (!(c)) {                                                          \
            printf("seed %d: %s fails at line %d\n", g_seed, #c, __LINE__);  \
            exit(1);                                                         \
        }                                                                    \
    } while (0)
static int g_seed = 0;

struct Ins {
    int fid, bin, ak, ai, bk, bi, toslot, di, lo, mid, hi, tape, sel, sa, sb, ta, tb, root, cidx;
};

static Ins plain_word(const uint64_t *p, bool wide, int k) {
    Ins w = {};
    const uint64_t a = wide ? p[2 * k] : p[k], b = wide ? p[2 * k + 1] : 0;
    w.fid = a & 63;
    w.bin = a >> 6 & 1;
    w.ak = a >> 7 & 3;
    if (wide) {
        w.ai = a >> 9 & 255, w.bk = a >> 17 & 3, w.bi = a >> 19 & 255, w.toslot = a >> 27 & 1;
        w.di = a >> 28 & 255, w.sel = a >> 36 & 1, w.sa = a >> 37 & 1, w.sb = a >> 38 & 1;
        w.ta = a >> 39 & 1, w.tb = a >> 40 & 1, w.lo = b & 255, w.mid = b >> 8 & 255;
        w.hi = b >> 16 & 255, w.tape = b >> 24 & 0xffffffff;
    } else {
        w.ai = ins_aidx(a), w.bk = ins_bkind(a), w.bi = ins_bidx(a), w.toslot = ins_toslot(a);
        w.di = ins_didx(a), w.sel = ins_sel(a), w.sa = ins_scale_a(a), w.sb = ins_scale_b(a);
        w.ta = ins_tape_a(a), w.tb = ins_tape_b(a), w.lo = ins_lo(a), w.mid = ins_mid(a);
        w.hi = ins_hi(a), w.tape = ins_tape(a);
    }
    return w;
}

static Ins staged_word(const uint64_t *p, bool wide, int k) {
    if (!wide) {
        Ins w = plain_word(p, false, k);
        w.root = p[k] >> 52 & 1;
        w.cidx = p[k] >> 53 & 255;
        return w;
    }
    const uint64_t a = p[2 * k], b = p[2 * k + 1];
    Ins w = {};
    w.fid = wst_fid(a), w.bin = wst_bit(a, 6), w.ak = wst_akind(a), w.ai = wst_aidx(a);
    w.bk = wst_bkind(a), w.bi = wst_bidx(a), w.sel = wst_bit(a, 21), w.sa = wst_bit(a, 22);
    w.sb = wst_bit(a, 23), w.ta = wst_bit(a, 24), w.tb = wst_bit(a, 25), w.toslot = wst_bit(a, 26);
    w.root = wst_bit(a, 27), w.cidx = wst_cidx(a), w.di = wst_didx(b), w.lo = wst_lo(b);
    w.mid = wst_mid(b), w.hi = wst_hi(b), w.tape = wst_tape(b);
    return w;
}

// value and partials; any smooth-enough rule will do, the two programs share it
static void apply(const Ins &w, double a, double b, double *o, double *d1, double *d2, bool *z1,
                  bool *z2) {
    *z1 = *z2 = false;
    *d1 = *d2 = 1.0;
    switch (w.fid) {
    case OP_IDENT: *o = a; return;
    case OP_ADD: *o = a + b; return;
    case OP_SUB: *o = a - b; *d2 = -1.0; return;
    case OP_MUL: *o = a * b; *d1 = b; *d2 = a; return;
    case OP_MAX: *o = fmax(a, b); *z1 = !(a >= b); *z2 = a >= b; *d1 = !*z1; *d2 = !*z2; return;
    case OP_PDIV:
        *z1 = *z2 = fabs(b) < 1e-9;
        *o = *z1 ? 1.0 : a / b;
        *d1 = *z1 ? 0.0 : 1.0 / b;
        *d2 = *z1 ? 0.0 : -(*o * *d1);
        return;
    case OP_SIN: *o = sin(a); *d1 = cos(a); return;
    case OP_CEXP: *z1 = a > 20.0; *o = exp(fmin(a, 20.0)); *d1 = *z1 ? 0.0 : *o; return;
    case OP_SQUARE: *o = a * a; *d1 = a + a; return;
    case OP_INV: *o = 1.0 / a; *d1 = -(*o * *o); return;
    default: CHECK(!"operator");
    }
}
static double safe_mul(double a, double b) { return (a == 0.0 || b == 0.0) ? 0.0 : a * b; }
static bool same(double a, double b) { return memcmp(&a, &b, 8) == 0 || (a != a && b != b); }

static void scale(std::vector<double> &T, int lo, int hi, double d, bool z) {
    for (int j = lo; j < hi; j++) T[j] = z ? 0.0 : T[j] * d;
}

struct Result {
    double value = 0.0;
    std::vector<double> fwd, rev;
    int ops = 0;
};

static Result run_plain(const uint64_t *prog, bool wide, int n, int K, const double *x,
                        const double *c) {
    Result r;
    std::vector<double> slot(64, NAN), tape(4096, NAN), T(K, 1.0), G(K, 0.0);
    double acc = NAN;
    auto get = [&](int kind, int idx) {
        return kind == OPD_ACC ? acc : kind == OPD_VAR ? x[idx] : kind == OPD_CONST ? c[idx] : slot[idx];
    };
    for (int k = 0; k < n; k++) {
        const Ins w = plain_word(prog, wide, k);
        const double a = get(w.ak, w.ai), b = w.bin ? get(w.bk, w.bi) : 0.0;
        double o, d1, d2;
        bool z1, z2;
        apply(w, a, b, &o, &d1, &d2, &z1, &z2);
        if (w.sa) scale(T, w.lo, w.mid, d1, z1 && w.sel);
        if (w.sb) scale(T, w.mid, w.hi, d2, z2 && w.sel);
        if (w.ta) tape[w.tape] = d1;
        if (w.tb) tape[w.tape + w.ta] = d2;
        if (w.toslot) slot[w.di] = o;
        acc = o;
        r.ops += w.fid != OP_IDENT;
    }
    r.value = acc;
    r.fwd = T;
    double adjacc = 1.0;
    for (int k = n - 1; k >= 0; k--) {
        const Ins w = plain_word(prog, wide, k);
        const double adj = w.toslot ? slot[w.di] : adjacc;
        for (int side = 0; side <= w.bin; side++) {
            const int kind = side ? w.bk : w.ak, idx = side ? w.bi : w.ai;
            if (kind == OPD_VAR) continue;
            const bool kept = side ? w.tb : w.ta;
            const double p = kept ? tape[w.tape + (side ? w.ta : 0)]
                             : side && w.fid == OP_SUB ? -1.0 : 1.0;
            const double g = safe_mul(adj, p);
            if (kind == OPD_ACC) adjacc = g;
            else if (kind == OPD_SLOT) slot[idx] = g;
            else G[idx] = G[idx] + g;
        }
    }
    r.rev = G;
    return r;
}

// The staged program as the device runs it: C once, V into rows (kept: from an
// earlier pass, then not run), M.
static Result run_staged(const uint64_t *base, const ExprDesc &d, const double *x,
                         const double *c, std::vector<double> &kept, bool load) {
    const bool wide = d.gen != 0;
    const int W = wide ? 2 : 1, K = d.K;
    Result r;
    std::vector<double> row(d.rows_rev, NAN), cslot(d.cslots, NAN), ctape(d.ctape, NAN),
        tape(d.tape, NAN), cm(c, c + K), T(K, 1.0), G(K, 0.0);
    std::vector<char> live(d.rows_rev, 0), clive(d.cslots, 0);
    const uint64_t *pc = base + d.prog_off, *pv = pc + W * d.n_c, *pm = pv + W * d.n_v,
                   *map = pm + W * d.n_m;
    // C
    double acc = NAN;
    for (int k = 0; k < d.n_c; k++) {
        const Ins w = staged_word(pc, wide, k);
        auto get = [&](int kind, int idx) {
            CHECK(kind == OPD_ACC || kind == OPD_CONST || kind == OPD_SLOT);
            if (kind == OPD_CONST) { CHECK(idx < K); return c[idx]; }
            if (kind == OPD_SLOT) { CHECK(idx < d.cslots && clive[idx]); return cslot[idx]; }
            return acc;
        };
        const double a = get(w.ak, w.ai), b = w.bin ? get(w.bk, w.bi) : 0.0;
        double o, d1, d2;
        bool z1, z2;
        apply(w, a, b, &o, &d1, &d2, &z1, &z2);
        if (w.sa) scale(T, w.lo, w.mid, d1, z1 && w.sel);
        if (w.sb) scale(T, w.mid, w.hi, d2, z2 && w.sel);
        if (w.ta) { CHECK(w.tape < d.ctape); ctape[w.tape] = d1; }
        if (w.tb) { CHECK(w.tape + w.ta < d.ctape); ctape[w.tape + w.ta] = d2; }
        CHECK(!(w.toslot && w.root));
        if (w.toslot) { CHECK(w.di < d.cslots); cslot[w.di] = o; clive[w.di] = 1; }
        if (w.root) { CHECK(w.lo < K); cm[w.lo] = o; }
        acc = o;
        r.ops++;
    }
    // rows
    const int nvars = d.mvars + d.ovars;
    auto var = [&](int i) { return wide ? (int)map[i] : (int)(d.map >> (4 * i) & 15); };
    for (int i = 0; i < nvars; i++) {
        if (load && i >= d.mvars) break;
        const int at = i < d.mvars ? i : i + d.vrows;
        CHECK(at < d.rows);
        row[at] = x[var(i)];
        live[at] = 1;
    }
    if (load)
        for (int j = 0; j < d.vrows; j++) {
            row[d.mvars + j] = kept[j];
            live[d.mvars + j] = 1;
        }
    // V, then M
    acc = NAN;
    for (int k = load ? d.n_v : 0; k < d.n_v + d.n_m; k++) {
        const bool in_v = k < d.n_v;
        const Ins w = staged_word(pv, wide, k);
        auto get = [&](int kind, int idx) {
            if (kind == OPD_CONST) { CHECK(!in_v && idx < K); return cm[idx]; }
            if (kind == OPD_ACC) return acc;
            CHECK(idx < d.rows && live[idx]);
            return row[idx];
        };
        const double a = get(w.ak, w.ai), b = w.bin ? get(w.bk, w.bi) : 0.0;
        double o, d1, d2;
        bool z1, z2;
        apply(w, a, b, &o, &d1, &d2, &z1, &z2);
        CHECK(!in_v || (!w.sa && !w.sb));
        if (w.sa) scale(T, w.lo, w.mid, d1, z1 && w.sel);
        if (w.sb) scale(T, w.mid, w.hi, d2, z2 && w.sel);
        if (!in_v && w.ta) { CHECK(w.tape < d.tape); tape[w.tape] = d1; }
        if (!in_v && w.tb) { CHECK(w.tape + w.ta < d.tape); tape[w.tape + w.ta] = d2; }
        if (w.toslot) { CHECK(w.di < d.rows); row[w.di] = o; live[w.di] = 1; }
        acc = o;
        r.ops += w.fid != OP_IDENT;
    }
    r.value = acc;
    r.fwd = T;
    kept.assign(row.begin() + d.mvars, row.begin() + d.mvars + d.vrows);
    // reverse sweep
    double adjacc = 1.0;
    for (int k = d.n_m - 1; k >= 0; k--) {
        const Ins w = staged_word(pm, wide, k);
        const double adj = w.toslot ? row[w.di] : adjacc;
        int at = -1;
        double gc = 0.0;
        for (int side = 0; side <= w.bin; side++) {
            const int kind = side ? w.bk : w.ak, idx = side ? w.bi : w.ai;
            if (kind == OPD_VAR) continue;
            const bool kpt = side ? w.tb : w.ta;
            const double p = kpt ? tape[w.tape + (side ? w.ta : 0)]
                             : side && w.fid == OP_SUB ? -1.0 : 1.0;
            const double g = safe_mul(adj, p);
            if (kind == OPD_ACC) adjacc = g;
            else if (kind == OPD_SLOT) row[idx] = g;
            else if (w.root) { CHECK(at < 0); at = w.cidx; gc = g; }
            else G[idx] = G[idx] + g;
        }
        if (at < 0) continue;
        CHECK(at < d.n_c);
        const Ins root = staged_word(pc, wide, at);
        CHECK(root.root && root.cidx <= at + 1);
        double ca = gc;
        for (int q = at; q > at - root.cidx; q--) {
            const Ins v = staged_word(pc, wide, q);
            if (v.toslot) CHECK(d.crow + v.di < d.rows_rev);
            const double cadj = v.toslot ? row[d.crow + v.di] : ca;
            for (int side = 0; side <= v.bin; side++) {
                const int kind = side ? v.bk : v.ak, idx = side ? v.bi : v.ai;
                const bool kpt = side ? v.tb : v.ta;
                const double p = kpt ? ctape[v.tape + (side ? v.ta : 0)]
                                 : side && v.fid == OP_SUB ? -1.0 : 1.0;
                const double g = safe_mul(cadj, p);
                if (kind == OPD_ACC) ca = g;
                else if (kind == OPD_SLOT) { CHECK(d.crow + idx < d.rows_rev); row[d.crow + idx] = g; }
                else G[idx] = G[idx] + g;
            }
        }
    }
    r.rev = G;
    return r;
}

int main(int argc, char **argv) {
    const int seeds = argc > 1 ? atoi(argv[1]) : 300;
    const int bins[] = {OP_ADD, OP_SUB, OP_MUL, OP_MAX, OP_PDIV};
    const int unas[] = {OP_SIN, OP_CEXP, OP_SQUARE, OP_INV};
    long exprs = 0, hoisted_c = 0, hoisted_v = 0, wides = 0;
    for (int seed = 0; seed < seeds; seed++) {
        g_seed = seed;
        std::mt19937 g(seed);
        auto rnd = [&](int n) { return (int)(g() % (unsigned)n); };
        // few to many variables, trees up to the formats' limits
        const int D = seed % 7 == 6 ? 1 + rnd(250) : seed % 5 == 4 ? rnd(2) : 1 + rnd(8);
        const int most = (const int[]){3, 15, 31, 63, 127, 255, 700}[rnd(7)];
        const double pconst = (const double[]){0.0, 0.2, 0.5, 0.8, 1.0}[rnd(5)];
        std::vector<int32_t> nt, ci;
        std::vector<float> nv;
        std::vector<TreeMeta> metas;
        int total_c = 0, kmax = 0;
        for (int m = 0; m < 40; m++) {
            for (;;) {
                std::vector<int32_t> t, c;
                std::vector<float> v;
                int K = 0, todo = 1, used = 1;
                while (todo > 0) {
                    const bool leaf = used + 1 > most || rnd(10) < 3;
                    --todo;
                    if (leaf) {
                        const bool con = D == 0 || (K < CO_MAX_K && rnd(1000) < 1000 * pconst);
                        t.push_back(con ? NODE_CONST : NODE_VAR);
                        v.push_back(con ? 0.0f : (float)rnd(D));
                        c.push_back(con ? K++ : -1);
                    } else if (rnd(10) < 6 && used + 2 <= most) {
                        t.push_back(NODE_BFUNC);
                        v.push_back((float)bins[rnd(5)]);
                        c.push_back(-1);
                        todo += 2;
                        used += 2;
                    } else {
                        t.push_back(NODE_UFUNC);
                        v.push_back((float)unas[rnd(4)]);
                        c.push_back(-1);
                        todo += 1;
                        used += 1;
                    }
                }
                int sp = 0, depth = 0;
                for (int i = (int)t.size() - 1; i >= 0; i--) {
                    sp += t[i] == NODE_BFUNC ? -1 : t[i] == NODE_UFUNC ? 0 : 1;
                    if (sp > depth) depth = sp;
                }
                if (K > CO_MAX_K || depth > CO_MAX_STACK) continue;
                metas.push_back({(int32_t)nt.size(), (int32_t)t.size(), total_c, K});
                nt.insert(nt.end(), t.begin(), t.end());
                nv.insert(nv.end(), v.begin(), v.end());
                ci.insert(ci.end(), c.begin(), c.end());
                total_c += K;
                if (K > kmax) kmax = K;
                break;
            }
        }
        const int M = (int)metas.size();
        PopHeader h = {};
        h.magic = POP_MAGIC;
        h.version = POP_VERSION;
        h.M_prob = M;
        h.total_nodes = (int)nt.size();
        h.total_c = total_c;
        h.N = seed % 4 == 3 ? 64 : 4096;   // without and with C
        h.n_vars = D;
        h.K_max = kmax;
        h.max_stack = CO_MAX_STACK;
        std::vector<uint64_t> plain(2 * nt.size()), staged(staged_words_max((int)nt.size(), D) + 4, 0xabababababababab);
        std::vector<int32_t> poff(M), route(M);
        std::vector<ExprDesc> descs(M);
        CHECK(decode_population(&h, nt.data(), nv.data(), ci.data(), metas.data(), plain.data(),
                                nullptr, nullptr, nullptr, poff.data(), route.data()) == CO_OK);
        // the population in two ranges, as an upload of a large one takes it
        Plan p0 = {}, p1 = {};
        const int cut = seed % 3 ? rnd(M + 1) : 0;
        CHECK(decode_range(&h, nt.data(), nv.data(), ci.data(), metas.data(), 0, cut, 0,
                           staged.data(), descs.data(), &p0) == CO_OK);
        CHECK(decode_range(&h, nt.data(), nv.data(), ci.data(), metas.data(), cut, M, p0.words,
                           staged.data(), descs.data(), &p1) == CO_OK);
        for (int i = 0; i < 4; i++) CHECK(staged[staged.size() - 4 + i] == 0xabababababababab);
        std::vector<char> seen(M, 0);
        int64_t vcols = 0;
        std::vector<double> x(D > 0 ? D : 1), c(total_c > 0 ? total_c : 1);
        for (double &v : c) v = (rnd(2001) - 1000) / 250.0;
        for (int pos = 0; pos < M; pos++) {
            const ExprDesc &d = descs[pos];
            const int m = d.y_row;
            CHECK(m >= 0 && m < M && !seen[m]);
            seen[m] = 1;
            const TreeMeta &t = metas[m];
            CHECK(d.gen == route[m] && d.K == t.K && d.c_off == t.c_offset);
            const Plan &p = pos < cut ? p0 : p1;
            CHECK(d.v_col >= 0 && d.v_col + d.vrows <= p.vcols);
            vcols += d.vrows;
            const int words = (d.gen ? 2 : 1) * (d.n_c + d.n_v + d.n_m) +
                              (d.gen ? d.mvars + d.ovars : 0);
            CHECK(words <= (d.gen ? 2 : 1) * t.n_nodes || (d.gen && t.n_nodes == 1 && words <= 3));
            int n = 0;
            for (int i = 0; i < t.n_nodes; i++) n += nt[t.node_offset + i] >= NODE_UFUNC;
            // LDS: no more rows than the budget or the plain program's
            CHECK(d.rows <= p.max_rows && d.cslots <= p.max_cslots);
            if (!d.gen) CHECK(d.rows <= kFastRows);
            // every operator once; C, V and M as the subtrees say
            CHECK(d.n_c + d.n_v + d.n_m == n || (d.n_m == 1 && d.n_c + d.n_v + 1 == n + 1));
            std::vector<double> kept(d.vrows, NAN);
            for (int pt = 0; pt < 3; pt++) {
                for (double &v : x) v = pt == 2 ? 0.0 : (rnd(2001) - 1000) / 300.0;
                const Result a = run_plain(plain.data() + poff[m], d.gen != 0,
                                           n == 0 ? 1 : n, t.K, x.data(), c.data() + t.c_offset);
                for (int load = 0; load < 2; load++) {
                    const Result b = run_staged(staged.data(), d, x.data(), c.data() + t.c_offset,
                                                kept, load);
                    CHECK(same(a.value, b.value));
                    CHECK(a.ops == b.ops + (load ? d.n_v : 0));
                    for (int j = 0; j < t.K; j++) {
                        CHECK(same(a.fwd[j], b.fwd[j]));
                        CHECK(same(a.rev[j], b.rev[j]));
                    }
                }
            }
            exprs++;
            hoisted_c += d.n_c;
            hoisted_v += d.n_v;
            wides += d.gen;
        }
        CHECK(vcols == p0.vcols + p1.vcols);
    }
    printf("%ld expressions, %ld wide, %ld C and %ld V operators\n", exprs, wides, hoisted_c,
           hoisted_v);
    puts("staged ok");
    return 0;
}
