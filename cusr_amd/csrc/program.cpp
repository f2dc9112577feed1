// program.cpp -- population checks and decode into device programs.
//
// Check order follows co_optimize (cusr/kernel/co_lib.cu:208-220): device
// bounds on the header, then the sum checks of cusr/kernel/loader.c:58-68,
// then per-expression validation, all before any device memory is touched.
// The per-expression checks go further than the reference, which trusts its
// input: every node type, operator id, variable index, constant rank and stack
// move is validated, so the device interpreter never indexes out of bounds.
#include <string.h>

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "program.h"

namespace cusr {

// Per operator id: arity (0: unknown), the relative device cost of one
// instruction per interpreter pass (VALU instructions per 64 lanes x 4 points,
// measured with SQ_INSTS_VALU on single-operator expressions; only the launch
// order within a K bin uses it), and whether its partials have flat branches.
struct OpInfo {
    uint8_t arity;
    bool sel;
    int16_t cost;
};
struct OpTable {
    OpInfo op[64] = {};
    constexpr OpTable() {
        for (int f : {OP_SIN, OP_COS, OP_TAN, OP_SINH, OP_COSH, OP_TANH, OP_LOG, OP_LOOSE_LOG,
                      OP_EXP, OP_INV, OP_LOOSE_INV, OP_NEG, OP_ABS, OP_SQRT, OP_LOOSE_SQRT,
                      OP_CEXP, OP_SQUARE, OP_PLOG})
            op[f].arity = 1;
        for (int f : {OP_ADD, OP_SUB, OP_MUL, OP_DIV, OP_LOOSE_DIV, OP_POW, OP_LOOSE_POW, OP_MAX,
                      OP_MIN, OP_LT, OP_GT, OP_LE, OP_GE, OP_PDIV})
            op[f].arity = 2;
        for (int f : {OP_MAX, OP_MIN, OP_LT, OP_GT, OP_LE, OP_GE, OP_PDIV, OP_CEXP}) op[f].sel = true;
        for (OpInfo &o : op) o.cost = 100;
        for (int f : {OP_ADD, OP_SUB}) op[f].cost = 12;
        op[OP_MUL].cost = 23;
        op[OP_SQUARE].cost = 83;
        for (int f : {OP_DIV, OP_LOOSE_DIV, OP_PDIV, OP_SQRT, OP_LOOSE_SQRT}) op[f].cost = 224;
        for (int f : {OP_EXP, OP_CEXP}) op[f].cost = 284;
        for (int f : {OP_SIN, OP_COS}) op[f].cost = 333;
        for (int f : {OP_LOG, OP_LOOSE_LOG, OP_PLOG}) op[f].cost = 391;
        for (int f : {OP_TAN, OP_POW, OP_LOOSE_POW}) op[f].cost = 450;
    }
};
static constexpr OpTable kOps;
static inline bool unary_op(int f) { return f >= 0 && kOps.op[f].arity == 1; }
static inline bool binary_op(int f) { return f >= 0 && kOps.op[f].arity == 2; }
static inline int op_cost(int f) { return kOps.op[f].cost; }

// Forward-AD and reverse-AD flags of an instruction: flat-branch select
// rule, which of its rank ranges get scaled (ADD's partials and SUB's left
// one are exactly 1; the identity has no partial to apply), and which partials
// keep a reverse-AD tape slot (read, and not exactly +-1).
struct Ins {
    int fid, bin, ak, ai, bk, bi, lo, mid, hi, tape, cidx;
    bool sel, sa, sb, ta, tb, root;
};

static void set_flags(Ins &w) {
    const int f = w.fid;
    w.sel = kOps.op[f].sel;
    const bool unit_a = w.bin ? (f == OP_ADD || f == OP_SUB) : (f == OP_IDENT);
    const bool unit_b = !w.bin || f == OP_ADD;
    w.sa = !unit_a && w.mid > w.lo;
    w.sb = !unit_b && w.hi > w.mid;
}

// program.h bit layouts
static uint64_t encode_fast(const Ins &w) {
    uint64_t x = (uint64_t)w.fid | (uint64_t)w.bin << 6;
    x |= (uint64_t)w.ak << 7 | (uint64_t)(w.ai & 15) << 9;
    x |= (uint64_t)w.bk << 13 | (uint64_t)(w.bi & 15) << 15;
    x |= (uint64_t)w.lo << 24 | (uint64_t)w.mid << 29 | (uint64_t)w.hi << 34;
    x |= (uint64_t)w.tape << 39;
    x |= (uint64_t)w.sel << 47 | (uint64_t)w.sa << 48 | (uint64_t)w.sb << 49;
    x |= (uint64_t)w.ta << 50 | (uint64_t)w.tb << 51;
    return x;
}

static void encode_wide(const Ins &w, uint64_t *out) {
    uint64_t a = (uint64_t)w.fid | (uint64_t)w.bin << 6;
    a |= (uint64_t)w.ak << 7 | (uint64_t)(w.ai & 255) << 9;
    a |= (uint64_t)w.bk << 17 | (uint64_t)(w.bi & 255) << 19;
    a |= (uint64_t)w.sel << 36 | (uint64_t)w.sa << 37 | (uint64_t)w.sb << 38;
    a |= (uint64_t)w.ta << 39 | (uint64_t)w.tb << 40;
    uint64_t b = (uint64_t)w.lo | (uint64_t)w.mid << 8 | (uint64_t)w.hi << 16;
    b |= (uint64_t)(uint32_t)w.tape << 24;
    out[0] = a;
    out[1] = b;
}

// program.h layouts of the staged program; at most `tape` bits of a tape slot
// are kept (a longer tape fits no LDS and is refused before any launch)
static void encode_staged(const Ins &w, bool wide, uint64_t *out) {
    if (!wide) {
        out[0] = encode_fast(w) | (uint64_t)w.root << 52 | (uint64_t)(w.cidx & 255) << 53;
        return;
    }
    uint64_t a = (uint64_t)w.fid | (uint64_t)w.bin << 6;
    a |= (uint64_t)w.ak << 7 | (uint64_t)(w.ai & 4095) << 9;
    a |= (uint64_t)w.sel << 21 | (uint64_t)w.sa << 22 | (uint64_t)w.sb << 23;
    a |= (uint64_t)w.ta << 24 | (uint64_t)w.tb << 25 | (uint64_t)w.root << 27;
    a |= (uint64_t)w.bk << 28 | (uint64_t)(w.bi & 4095) << 32;
    a |= (uint64_t)(w.cidx & kWideCidxMax) << 44;
    uint64_t b = (uint64_t)w.lo | (uint64_t)w.mid << 8 | (uint64_t)w.hi << 16;
    b |= (uint64_t)(w.tape & 0xfffff) << 44;
    out[0] = a;
    out[1] = b;
}

// Integral node value in [0, limit) or -1.
static int node_int(float v, int limit) {
    if (!(v >= 0.0f) || v >= (float)limit) return -1;
    int i = (int)v;
    return ((float)i == v) ? i : -1;
}

struct Operand {
    int kind;      // OPD_*
    int idx;       // var / const rank / slot
    int producer;  // instruction that produced an ACC value, else -1
};

struct Visit {
    int node;   // subtree root (prefix index)
    int stage;  // 0: nothing evaluated, 1: first operand done, 2: both done
};

// A node of a staged program. Operators of its subtree in all (ops) and in M
// (mops, with every one-class subtree of operators an operand); then, top
// down: its program, the first instruction of its subtree there, the slots
// live while it runs, and the slot or row its value goes to (-1: ACC, -2: a C
// subtree's value).
struct StagedNode {
    int ops, mops, start, dest;
    uint8_t prog, live;
};

// Sets of an expression's nodes, a bit each, in words of 64: the staging goes
// through them instead of through the nodes, whose types and classes a branch
// predictor cannot follow (its share of the decode of 60,000 expressions of 27
// nodes, one thread: 32 -> 15 of 107 ms).
struct NodeSets {
    std::vector<uint64_t> bits;
    int words = 0;
    uint64_t *var, *op, *m;           // variable leaves, operators, M's operators
    uint64_t *mvar, *vroot, *croot;   // variables M reads, the maximal V and C subtrees
    void reserve(int n) { bits.resize(6 * (size_t)((n + 63) / 64)); }
    void clear(int n) {
        words = (n + 63) / 64;
        uint64_t **const sets[6] = {&var, &op, &m, &mvar, &vroot, &croot};
        for (int k = 0; k < 6; k++) *sets[k] = bits.data() + (size_t)k * words;
        memset(bits.data(), 0, sizeof(uint64_t) * 6 * words);
    }
    static void mark(uint64_t *set, int i, bool on) { set[i >> 6] |= (uint64_t)on << (i & 63); }
    // fn(i) for the members, ascending, until it returns false
    template <typename Fn>
    static void each(const uint64_t *set, int words, const uint64_t *but, const Fn &fn) {
        for (int w = 0; w < words; w++)
            for (uint64_t b = but ? set[w] & ~but[w] : set[w]; b; b &= b - 1)
                if (!fn(w * 64 + __builtin_ctzll(b))) return;
    }
    // the operators of [i, end) go to M, and their variables
    void to_m(int i, int end) {
        for (int w = i >> 6; w < words && w * 64 < end; w++) {
            uint64_t r = ~(uint64_t)0;
            if (w * 64 < i) r &= ~(uint64_t)0 << (i & 63);
            if (end - w * 64 < 64) r &= ~(~(uint64_t)0 << (end - w * 64));
            m[w] |= op[w] & r;
            mvar[w] |= var[w] & r;
            vroot[w] &= ~r;
            croot[w] &= ~r;
        }
    }
};

// The largest rows, constants beside a C program and scalar slots of the
// expressions emitted (Plan).
struct Most {
    int rows = 0, ck = 0, cslots = 0;
    void add(const Most &o) {
        rows = std::max(rows, o.rows);
        ck = std::max(ck, o.ck);
        cslots = std::max(cslots, o.cslots);
    }
};

// Per-thread working arrays, grown to the largest expression seen and not
// cleared between expressions (every entry read is written first).
struct TreeScratch {
    std::vector<int> size, left, cc, need, depth_stack;
    // staged programs: bit 0 variables, bit 1 constants in the subtree; slots of
    // M; and what the emission hands down
    std::vector<int> cls, needm;
    std::vector<StagedNode> st;
    NodeSets set;
    Most most;
    int rows[CO_MAX_VARS + 1];
    std::vector<Operand> res;
    std::vector<Visit> work;
    void reserve(int n) {
        if ((int)size.size() >= n + 1) return;
        cls.resize(n + 1);
        needm.resize(n + 1);
        st.resize(n + 1);
        set.reserve(n);
        size.resize(n + 1);
        left.resize(n + 1);
        cc.resize(n + 1);
        need.resize(n + 1);
        depth_stack.resize(n + 1);
        res.resize(n + 1);
        work.resize(n + 1);
    }
};

static inline bool is_leaf(int t) { return t == NODE_VAR || t == NODE_CONST; }

// Validate one expression (n nodes, K constants, D variables): node types,
// operator ids, variable indices, prefix-order constant ranks and stack moves.
// Returns CO_OK, CO_ERR_BOUNDS (value stack beyond CO_MAX_STACK) or
// CO_ERR_PROGRAM, and its value-stack depth. Fills s.size / s.left / s.cc / s.cls,
// s.needm, s.set, the counts of s.st and s.need (the spill slots of each subtree in the
// emission's order) for the emission. stage_c: operators over constants alone
// are class 2, to go to C; else class 3, to stay in M.
static int check_tree(const int32_t *nt, const float *nv, const int32_t *ci, int n, int K,
                      int D, bool stage_c, int *stack_depth, TreeScratch &s) {
    if (n <= 0) return CO_ERR_PROGRAM;
    s.reserve(n);
    int *size = s.size.data(), *left = s.left.data(), *cc = s.cc.data(), *need = s.need.data();
    int *st = s.depth_stack.data(), *cls = s.cls.data(), *needm = s.needm.data();
    StagedNode *sn = s.st.data();
    NodeSets &set = s.set;
    set.clear(n);
    // prefix pass: constant ranks must be 0..K-1 in prefix order
    cc[0] = 0;
    for (int i = 0; i < n; i++) {
        const int c = nt[i] == NODE_CONST;
        if (c && ci[i] != cc[i]) return CO_ERR_PROGRAM;
        cc[i + 1] = cc[i] + c;
    }
    if (cc[n] != K) return CO_ERR_PROGRAM;
    // execution pass (last node first): validation, stack depth, subtree sizes;
    // the stack holds subtree roots (a subtree's size is known when it is pushed)
    int sp = 0, depth = 0;
    for (int i = n - 1; i >= 0; i--) {
        const int t = nt[i];
        if (t == NODE_VAR || t == NODE_CONST) {
            if (t == NODE_VAR && node_int(nv[i], D) < 0) return CO_ERR_PROGRAM;
            cls[i] = t == NODE_VAR ? 1 : 2;
            NodeSets::mark(set.var, i, t == NODE_VAR);
            size[i] = 1;
            need[i] = needm[i] = 0;
            sn[i].ops = sn[i].mops = 0;
            st[sp++] = i;
        } else if (t == NODE_UFUNC) {
            if (!unary_op(node_int(nv[i], 64))) return CO_ERR_PROGRAM;
            if (sp < 1) return CO_ERR_PROGRAM;
            const int c = st[sp - 1];
            size[i] = size[c] + 1;
            cls[i] = cls[c] == 2 && !stage_c ? 3 : cls[c];
            need[i] = need[c];
            needm[i] = cls[c] == 3 ? needm[c] : 0;
            sn[i].ops = sn[c].ops + 1;
            sn[i].mops = cls[c] == 3 ? sn[c].mops + 1 : 1;
            NodeSets::mark(set.op, i, true);
            NodeSets::mark(set.m, i, cls[i] == 3);
            st[sp - 1] = i;
        } else if (t == NODE_BFUNC) {
            if (!binary_op(node_int(nv[i], 64))) return CO_ERR_PROGRAM;
            if (sp < 2) return CO_ERR_PROGRAM;
            const int l = st[sp - 1], r = st[sp - 2];   // left operand = top of stack
            --sp;
            left[i] = size[l];
            size[i] = size[l] + size[r] + 1;
            cls[i] = cls[l] | cls[r];
            if (cls[i] == 2 && !stage_c) cls[i] = 3;
            // the operand that needs more slots runs first; two that both need
            // instructions hold one value in a slot while the other runs
            const int nl = need[l], nr = need[r];
            const int hi = nl > nr ? nl : nr;
            need[i] = (!is_leaf(nt[l]) && !is_leaf(nt[r]) && nl == nr) ? nl + 1 : hi;
            // the same within M, where subtrees of one class are operands
            const bool ml = cls[l] == 3, mr = cls[r] == 3;
            const int a = ml ? needm[l] : 0, b = mr ? needm[r] : 0;
            needm[i] = (ml && mr && a == b) ? a + 1 : (a > b ? a : b);
            sn[i].ops = sn[l].ops + sn[r].ops + 1;
            sn[i].mops = (ml ? sn[l].mops : 0) + (mr ? sn[r].mops : 0) + 1;
            NodeSets::mark(set.op, i, true);
            const bool m = cls[i] == 3;
            NodeSets::mark(set.m, i, m);
            for (int c : {l, r}) {
                const bool leaf = sn[c].ops == 0;
                NodeSets::mark(set.mvar, c, m & leaf & (cls[c] == 1));
                NodeSets::mark(set.vroot, c, m & !leaf & (cls[c] == 1));
                NodeSets::mark(set.croot, c, m & !leaf & (cls[c] == 2));
            }
            st[sp - 1] = i;
        } else {
            return CO_ERR_PROGRAM;
        }
        if (sp > depth) depth = sp;
    }
    if (sp != 1) return CO_ERR_PROGRAM;
    NodeSets::mark(set.mvar, 0, is_leaf(nt[0]) && cls[0] == 1);
    NodeSets::mark(set.vroot, 0, !is_leaf(nt[0]) && cls[0] == 1);
    NodeSets::mark(set.croot, 0, !is_leaf(nt[0]) && cls[0] == 2);
    *stack_depth = depth;
    if (depth > CO_MAX_STACK) return CO_ERR_BOUNDS;
    return CO_OK;
}

// Instruction k of a plain program, and the later mark that sends its result to
// slot di.
static inline void put_ins(uint64_t *out, bool wide, int k, Ins &w) {
    set_flags(w);
    if (wide) encode_wide(w, out + 2 * k);
    else out[k] = encode_fast(w);
}
static inline void put_spill(uint64_t *out, bool wide, int k, int di) {
    if (wide) out[2 * k] |= (uint64_t)1 << 27 | (uint64_t)(di & 255) << 28;
    else out[k] |= (uint64_t)1 << 19 | (uint64_t)(di & 15) << 20;
}
// Emit the plain program of a checked expression (program.h), encoded, into out
// in execution order (out holds zeros on entry). Returns CO_OK, CO_ERR_BOUNDS or
// CO_ERR_PROGRAM.
//
// Operands are evaluated in Sethi-Ullman order: when both operands of a binary
// operator need instructions, the one whose subtree needs more spill slots runs
// first (the right one on a tie, as the reference's last-node-first order
// does) and its value waits in a slot while the other runs. A subtree's value
// and its constants' tangents and adjoints do not depend on which sibling runs
// first, and the order keeps the slot count at the minimum (at most
// log2(nodes + 1)), which is what sizes each wavefront's LDS.
static int emit_plain(const int32_t *nt, const float *nv, const int32_t *ci, int n, int D,
                      bool wide, uint64_t *out, TreeScratch &s) {
    const int *left = s.left.data(), *cc = s.cc.data(), *need = s.need.data(),
              *size = s.size.data();
    Operand *res = s.res.data();
    Visit *work = s.work.data();
    auto leaf_opd = [&](int i) -> Operand {
        return nt[i] == NODE_VAR ? Operand{OPD_VAR, node_int(nv[i], D), -1}
                                 : Operand{OPD_CONST, ci[i], -1};
    };
    int k = 0, tape = 0, live_slots = 0;
    if (is_leaf(nt[0])) {
        // the expression is one leaf: its value is the identity of that leaf
        const Operand a = leaf_opd(0);
        Ins w = {};
        w.fid = OP_IDENT;
        w.ak = a.kind;
        w.ai = a.idx;
        w.lo = cc[0];
        w.mid = w.hi = cc[n];
        put_ins(out, wide, k++, w);   // the identity's partial is +1: no tape slot
        return CO_OK;
    }
    int sp = 0;
    work[sp++] = {0, 0};
    while (sp > 0) {
        Visit &fr = work[sp - 1];
        const int i = fr.node;
        const bool bin = nt[i] == NODE_BFUNC;
        const int l = i + 1, r = bin ? i + 1 + left[i] : -1;
        const bool both = bin && !is_leaf(nt[l]) && !is_leaf(nt[r]);
        const int first = (!bin || (both && need[l] > need[r])) ? l : r;
        const int second = !bin ? -1 : (first == l ? r : l);
        if (fr.stage == 0) {
            fr.stage = 1;
            if (!is_leaf(nt[first])) {
                work[sp++] = {first, 0};
                continue;
            }
            res[first] = leaf_opd(first);
        }
        if (fr.stage == 1 && bin) {
            fr.stage = 2;
            if (both) {
                // the first operand's value waits in the next free slot
                if (live_slots >= (wide ? kMaxSlotsWide : kMaxSlots)) return CO_ERR_BOUNDS;
                const int slot = live_slots++;
                Operand &o = res[first];
                if (o.kind != OPD_ACC || o.producer < 0) return CO_ERR_PROGRAM;
                put_spill(out, wide, o.producer, slot);
                o = {OPD_SLOT, slot, -1};
            }
            if (!is_leaf(nt[second])) {
                work[sp++] = {second, 0};
                continue;
            }
            res[second] = leaf_opd(second);
        }
        --sp;
        const Operand a = res[l];
        const Operand b = bin ? res[r] : Operand{OPD_ACC, 0, -1};
        // spill slots are used last in, first out
        if (a.kind == OPD_SLOT) {
            if (a.idx != live_slots - 1) return CO_ERR_PROGRAM;
            live_slots--;
        }
        if (bin && b.kind == OPD_SLOT) {
            if (b.idx != live_slots - 1) return CO_ERR_PROGRAM;
            live_slots--;
        }
        Ins w = {};
        w.fid = (int)nv[i];
        w.bin = bin ? 1 : 0;
        w.ak = a.kind;
        w.ai = a.idx;
        if (bin) {
            w.bk = b.kind;
            w.bi = b.idx;
        }
        w.lo = cc[i + 1];
        w.hi = cc[i + size[i]];
        w.mid = bin ? cc[i + 1 + left[i]] : w.hi;
        w.tape = tape;
        // reverse-AD tape slots only for partials that are read and not exactly +-1
        const bool unit = bin && (w.fid == OP_ADD || w.fid == OP_SUB);
        w.ta = a.kind != OPD_VAR && !unit;
        w.tb = bin && b.kind != OPD_VAR && !unit;
        tape += (w.ta ? 1 : 0) + (w.tb ? 1 : 0);
        res[i] = {OPD_ACC, 0, k};
        put_ins(out, wide, k++, w);
    }
    if (live_slots != 0) return CO_ERR_PROGRAM;
    return !wide && tape > 255 ? CO_ERR_BOUNDS : CO_OK;   // never: n <= 255 keeps it below
}

static int64_t program_words(int n_nodes, bool wide, bool staged);

// Rows of a wavefront's LDS that an expression may use (variables, V values,
// slots): what its plain program takes, n_vars and its slots, or this many.
// V subtrees beyond stay in M, the last ones first. A row of the fp64 forward
// kernels to K = 8 is 2 KB (four points per lane), and their registers let three
// wavefronts on a SIMD at K = 1 to 3, two beyond: as many as these rows leave room
// for in a CU's 160 KB. Measured at K = 1, 4 rows -> 6 -> 8: 16,384 x 1,024 2.09 ->
// 1.68 -> 2.12 ms, 60,000 x 300 3.37 -> 2.73 -> 3.11, reverse AD 5.90 -> 4.11 -> 3.46;
// 6 -> 8 at K = 2 and 3: 16,384 x 1,024 2.48 -> 3.34 and 2.99 -> 4.06 ms. Elsewhere a
// row is 512 bytes or 1 KB (from N = 16,384 on two points per lane); more than eight
// rows cost reverse AD wavefronts (twelve: C3 67.9 -> 70.4 ms).
static int row_budget(int K, int N) { return K > 3 || N >= 16384 ? 8 : 6; }
// A wide expression with more variable rows than this is not staged: its plain
// rows may fill the LDS, which then has no room for C's scalars.
constexpr int kStageVarsMax = 128;
constexpr int kRowsMax = 160;   // likewise for the rows of a staged one

// Whether C pays at N points: a step of C takes about as long as a step of M
// (one point per lane against up to four, but both wait mostly on their own
// chains: 1,300 and 1,400 cycles on the benchmark operators at K = 8), so a
// pass of one batch of four points per lane has nothing to gain. Measured, 60,000
// expressions of K 1-5, ten iterations, N = 60: 5.95 ms of device time with C,
// 5.38 without; N = 1,024 (two batches) with C is faster (16,384 expressions,
// K 1-8: 9.10 -> 7.67 ms with C and V).
static bool stage_constants(int N) {
    const int granules = (N + 63) / 64, parts = co_partitions_for_n(N);
    return (granules + parts - 1) / parts > 4;
}

// The staged program of a checked expression (program.h) and its descriptor's
// counts; out holds zeros on entry. Operands run in emit_plain's order, in one
// pass over the nodes, parents first: a subtree's instructions are contiguous,
// its root's last, so each node's place follows from the operator counts.
static int emit_staged(const int32_t *nt, const float *nv, const int32_t *ci, int n, int K, int D,
                       int N, bool wide, bool staged, uint64_t *out, ExprDesc &d, int64_t *cost,
                       TreeScratch &s) {
    const int *size = s.size.data(), *left = s.left.data(), *cc = s.cc.data(),
              *need = s.need.data();
    int *cls = s.cls.data(), *needm = s.needm.data(), *rows = s.rows;
    StagedNode *sn = s.st.data();
    NodeSets &set = s.set;
    int vars[CO_MAX_VARS + 1];         // variable rows: M's, then V's others
    const int plain_rows = D + need[0];
    const int budget = std::min(wide ? 4096 : kFastRows,
                                std::max(std::min(plain_rows, kRowsMax), row_budget(K, N)));
    bool stage = staged && K > 0;
    // class 3 to every operator of [i, end), so that it stays in M
    auto into_m = [&](int i, int end) {
        set.to_m(i, end);
        for (; i < end; ++i) cls[i] = sn[i].ops > 0 ? 3 : cls[i];
    };
    // slots and operators of M after such changes below end, last node first
    auto recount = [&](int end) {
        for (int w = (end - 1) >> 6; w >= 0; w--)
            for (uint64_t b = set.m[w]; b;) {
                const int k = 63 - __builtin_clzll(b), i = w * 64 + k;
                b ^= (uint64_t)1 << k;
                const bool bin = nt[i] == NODE_BFUNC;
                const int l = i + 1, r = bin ? l + left[i] : l;
                const bool ml = cls[l] == 3, mr = bin && cls[r] == 3;
                const int x = ml ? needm[l] : 0, y = mr ? needm[r] : 0;
                needm[i] = ml && mr && x == y ? x + 1 : std::max(x, y);
                sn[i].mops = (ml ? sn[l].mops : 0) + (mr ? sn[r].mops : 0) + 1;
            }
    };
    if (!stage) {
        into_m(0, n);
        recount(n);
    }
    int mv = 0, nvars = 0, nvr = 0, vslots = 0, cslots = 0, n_c = 0, n_v = 0, tail = 0;
    int *vroot = s.depth_stack.data();   // roots of the V subtrees
    const auto row = [&](int i) {
        int &r = rows[(int)nv[i]];
        if (r < 0) {
            vars[nvars] = (int)nv[i];
            r = nvars++;
        }
        return nvars < D;   // until every variable has its row
    };
    for (;;) {
        for (int v = 0; v < D; v++) rows[v] = -1;
        nvars = nvr = vslots = cslots = n_c = n_v = 0;
        // the variables M reads itself, and the maximal subtrees of operators
        // over constants or variables alone
        NodeSets::each(set.mvar, set.words, nullptr, row);
        mv = nvars;
        NodeSets::each(set.croot, set.words, nullptr, [&](int i) {
            n_c += sn[i].ops;
            cslots = std::max(cslots, need[i]);
            return true;
        });
        NodeSets::each(set.vroot, set.words, nullptr, [&](int i) {
            n_v += sn[i].ops;
            vslots = std::max(vslots, need[i]);
            vroot[nvr++] = i;
            return true;
        });
        if (nvr > 0 && mv < D) NodeSets::each(set.var, set.words, set.mvar, row);
        tail = mv + nvr;
        if (stage && (n_c > kWideCidxMax || (wide && nvars > kStageVarsMax))) {
            stage = false;
            into_m(0, n);
            recount(n);
            continue;
        }
        if (nvr == 0 || tail + std::max(nvars - mv + vslots, cls[0] == 3 ? needm[0] : 0) <= budget)
            break;
        // the last V subtrees go to M, one more each time round, but at once as many
        // as the rows of the values, the variables and V's slots alone refuse: M's
        // slots then ask for at most need[0] more rounds (one by one, the decode of a
        // sum of 64,000 sines took 57 s, now 22 ms)
        int keep = 0;
        for (int slots = 0; keep < nvr - 1; ++keep) {
            slots = std::max(slots, need[vroot[keep]]);
            if (keep + 1 + nvars + slots > budget) break;
        }
        for (int k = keep; k < nvr; ++k) into_m(vroot[k], vroot[k] + size[vroot[k]]);
        recount(vroot[nvr - 1] + size[vroot[nvr - 1]]);
    }
    // rows: M's variables, V's values, then V's other variables and slots over
    // M's slots
    for (int r = mv; r < nvars; r++) rows[vars[r]] = r + nvr;
    enum { C = 0, V = 1, M = 2, kCRoot = -2 };
    const int words = wide ? 2 : 1;
    const bool ident = is_leaf(nt[0]) || cls[0] != 3;
    const int n_m = ident ? 1 : sn[0].mops;
    uint64_t *base[3] = {out, out + (size_t)words * n_c, out + (size_t)words * (n_c + n_v)};
    const int slot0[3] = {0, tail + nvars - mv, tail};
    int at_c = 0, at_v = 0, at_row = mv;     // next C and V subtree's place
    int tape[3] = {0, 0, 0};
    int64_t op_costs[3] = {0, 0, 0};
    struct Opd {
        int kind, idx, cidx;   // cidx: C instruction of a C subtree's root, -1
    };
    // a leaf or, in M, a hoisted subtree, whose program gets its place
    auto operand = [&](int i) -> Opd {
        if (nt[i] == NODE_VAR) return {OPD_VAR, rows[(int)nv[i]], -1};
        if (nt[i] == NODE_CONST) return {OPD_CONST, ci[i], -1};
        StagedNode &t = sn[i];
        t.live = 0;
        if (cls[i] == 2) {
            t.prog = C;
            t.start = at_c;
            t.dest = kCRoot;
            at_c += t.ops;
            return {OPD_CONST, cc[i], at_c - 1};
        }
        t.prog = V;
        t.start = at_v;
        t.dest = at_row;
        at_v += t.ops;
        return {OPD_VAR, at_row++, -1};
    };
    auto put = [&](int prog, int k, Ins &w, int dest) {
        set_flags(w);
        encode_staged(w, wide, base[prog] + (size_t)words * k);
        if (dest < 0) return;
        uint64_t *q = base[prog] + (size_t)words * k;
        if (!wide) {
            q[0] |= (uint64_t)1 << 19 | (uint64_t)(dest & 15) << 20;
        } else {
            q[0] |= (uint64_t)1 << 26;
            q[1] |= (uint64_t)(dest & 4095) << 32;
        }
    };
    if (ident) {
        // one operand: its identity, whose partial is +1 (no tape slot)
        const Opd a = operand(0);
        Ins w = {};
        w.fid = OP_IDENT;
        w.ak = a.kind;
        w.ai = a.idx;
        w.mid = w.hi = cc[n];
        w.root = a.cidx >= 0;
        w.cidx = w.root ? a.cidx : 0;
        op_costs[M] += op_cost(OP_IDENT);
        put(M, 0, w, -1);
    } else {
        sn[0].prog = M;
        sn[0].start = 0;
        sn[0].live = 0;
        sn[0].dest = -1;
    }
    NodeSets::each(set.op, set.words, nullptr, [&](int i) {
        const StagedNode t = sn[i];
        const bool bin = nt[i] == NODE_BFUNC;
        const int l = i + 1, r = bin ? l + left[i] : l;
        // an operand that needs instructions of this program
        const bool il = !is_leaf(nt[l]) && (t.prog != M || cls[l] == 3);
        const bool ir = bin && !is_leaf(nt[r]) && (t.prog != M || cls[r] == 3);
        const int *nd = t.prog == M ? needm : need;
        auto count = [&](int c) { return t.prog == M ? sn[c].mops : sn[c].ops; };
        const bool both = il && ir, left_first = both && nd[l] > nd[r];
        const int slot = slot0[t.prog] + t.live;   // where the first of two waits
        auto place = [&](int c, bool first, int start) {
            StagedNode &k = sn[c];
            k.prog = t.prog;
            k.start = start;
            k.live = (uint8_t)(t.live + (both && !first));
            k.dest = both && first ? slot : -1;
        };
        Opd a, b = {OPD_ACC, 0, -1};
        if (il) {
            place(l, left_first || !both, t.start + (both && !left_first ? count(r) : 0));
            a = left_first ? Opd{OPD_SLOT, slot, -1} : Opd{OPD_ACC, 0, -1};
        } else {
            a = operand(l);
        }
        if (ir) {
            place(r, !left_first, t.start + (left_first ? count(l) : 0));
            if (both && !left_first) b = {OPD_SLOT, slot, -1};
        } else if (bin) {
            b = operand(r);
        }
        Ins w = {};
        w.fid = (int)nv[i];
        w.bin = bin;
        w.ak = a.kind;
        w.ai = a.idx;
        w.bk = bin ? b.kind : 0;
        w.bi = bin ? b.idx : 0;
        w.lo = cc[l];
        w.hi = cc[i + size[i]];
        w.mid = bin ? cc[r] : w.hi;
        w.tape = tape[t.prog];
        const bool unit = bin && (w.fid == OP_ADD || w.fid == OP_SUB);
        w.ta = a.kind != OPD_VAR && !unit;
        w.tb = bin && b.kind != OPD_VAR && !unit;
        tape[t.prog] += w.ta + w.tb;
        op_costs[t.prog] += op_cost(w.fid);
        // M: the operand that is a C subtree; C: a subtree's last instruction
        const int k = t.start + count(i) - 1;
        const bool c_root = t.dest == kCRoot;
        w.root = c_root || a.cidx >= 0 || b.cidx >= 0;
        w.cidx = c_root ? t.ops : a.cidx >= 0 ? a.cidx : b.cidx >= 0 ? b.cidx : 0;
        put(t.prog, k, w, t.dest);
        return true;
    });
    if (!wide && tape[M] > 255) return CO_ERR_BOUNDS;   // never: n <= 255 keeps it below
    d.map = 0;
    if (wide) {
        uint64_t *vm = base[M] + 2 * (size_t)n_m;
        for (int r = 0; r < nvars; r++) vm[r] = (uint64_t)vars[r];
    } else {
        for (int r = 0; r < nvars; r++) d.map |= (uint64_t)vars[r] << (4 * r);
    }
    const int mslots = ident ? 0 : needm[0];
    d.n_c = n_c;
    d.n_v = n_v;
    d.n_m = n_m;
    d.K = K;
    d.mvars = mv;
    d.vrows = nvr;
    d.ovars = nvars - mv;
    d.crow = tail + mslots;
    d.rows = tail + std::max(nvars - mv + vslots, mslots);
    d.rows_rev = std::max(d.rows, d.crow + cslots);
    d.cslots = cslots;
    d.ctape = tape[C];
    d.tape = tape[M];
    // V runs once in a fit and C once per pass, by one point per lane
    *cost = 229 + op_costs[M] + op_costs[C] / 4;
    if (wide && stage) {
        // what the general kernel's wavefront takes for it in reverse AD must not
        // pass what the plain program took where that may have been the device's
        // limit (at 512 bytes a row and tape slot in fp64; measured by the 256 of
        // fp32, which hold for both)
        int plain_tape = 0;
        for (int i = 0; i < n; i++) {
            if (is_leaf(nt[i])) continue;
            const bool bin = nt[i] == NODE_BFUNC;
            const int f = (int)nv[i];
            if (bin && (f == OP_ADD || f == OP_SUB)) continue;
            plain_tape += nt[i + 1] != NODE_VAR;
            if (bin) plain_tape += nt[i + 1 + left[i]] != NODE_VAR;
        }
        const size_t row = 64 * sizeof(float), rows = (size_t)d.rows_rev + d.tape;
        const size_t uni = (size_t)uni_bytes_of(d, true, K);
        if (2 * rows * row + uni > (64u << 10) &&
            rows * row + uni > (plain_rows + (size_t)plain_tape) * row) {
            memset(out, 0, sizeof(uint64_t) * program_words(n, true, true));
            return emit_staged(nt, nv, ci, n, K, D, N, wide, false, out, d, cost, s);
        }
    }
    return CO_OK;
}

// Worker threads for the decode, started on first use and kept for the
// process: a decode phase hands its chunks to them instead of starting threads
// (starting 15 threads twice per decode cost about 1.5 ms of C5's 6 ms). One
// job at a time; a caller that finds the pool busy, or runs in a process
// forked after the pool started, does its chunks itself.
class DecodePool {
  public:
    static DecodePool &get() {
        static DecodePool pool;
        return pool;
    }
    // fn(i) for every i in [0, n) on the workers and this thread; false (and
    // nothing run) when the pool cannot take the job
    bool run(int n, const std::function<void(int)> &fn) {
        if (workers_.empty() || getpid() != pid_) return false;
        std::unique_lock<std::mutex> job(job_mu_, std::try_to_lock);
        if (!job.owns_lock()) return false;
        {
            std::lock_guard<std::mutex> g(mu_);
            fn_ = &fn;
            n_ = n;
            next_.store(0);
            busy_ = (int)workers_.size();
            ++gen_;
        }
        cv_.notify_all();
        work();
        std::unique_lock<std::mutex> g(mu_);
        done_cv_.wait(g, [&] { return busy_ == 0; });
        fn_ = nullptr;
        return true;
    }

  private:
    DecodePool() : pid_(getpid()) {
        const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
        const int n = (int)std::min(15u, hw - 1);
        try {
            for (int i = 0; i < n; i++) workers_.emplace_back([this] { loop(); });
        } catch (...) {
            // fewer workers than asked: the ones started serve
        }
    }
    ~DecodePool() {
        {
            std::lock_guard<std::mutex> g(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (std::thread &t : workers_) t.join();
    }
    void work() {
        for (int i = next_.fetch_add(1); i < n_; i = next_.fetch_add(1)) (*fn_)(i);
    }
    void loop() {
        uint64_t seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> g(mu_);
                cv_.wait(g, [&] { return stop_ || gen_ != seen; });
                if (stop_) return;
                seen = gen_;
            }
            work();
            std::lock_guard<std::mutex> g(mu_);
            if (--busy_ == 0) done_cv_.notify_one();
        }
    }
    std::vector<std::thread> workers_;
    std::mutex job_mu_, mu_;
    std::condition_variable cv_, done_cv_;
    const std::function<void(int)> *fn_ = nullptr;
    int n_ = 0, busy_ = 0;
    std::atomic<int> next_{0};
    uint64_t gen_ = 0;
    bool stop_ = false;
    const pid_t pid_;
};

// Runs fn(m0, m1) over so many contiguous pieces of [0, M) on the decode pool and
// this thread; without the pool, redo(0, M) runs on this thread.
template <typename Fn, typename Redo>
static void chunked(int M, int pieces, const Fn &fn, const Redo &redo) {
    if (pieces > 1 && M > 0) {
        const int chunk = (M + pieces - 1) / pieces;
        const int n = (M + chunk - 1) / chunk;
        const std::function<void(int)> job = [&](int i) {
            fn(i * chunk, std::min(M, (i + 1) * chunk));
        };
        if (DecodePool::get().run(n, job)) return;
    }
    redo(0, M);
}

int check_header(const PopHeader *h, const int32_t *nt, const float *nv, const int32_t *ci,
                 const TreeMeta *metas) {
    if (!h || !metas) return CO_ERR_NULLARG;
    if (h->total_nodes > 0 && (!nt || !nv || !ci)) return CO_ERR_NULLARG;
    if (h->M_prob < 0 || h->N < 0 || h->n_vars < 0 || h->total_nodes < 0 || h->total_c < 0)
        return CO_ERR_NULLARG;
    if (h->K_max > CO_MAX_K || h->max_stack > CO_MAX_STACK || h->n_vars > CO_MAX_VARS)
        return CO_ERR_BOUNDS;
    long ksum = 0, nsum = 0;
    for (int m = 0; m < h->M_prob; m++) { ksum += metas[m].K; nsum += metas[m].n_nodes; }
    if (ksum != (long)h->total_c) return CO_ERR_SUM_C;
    if (nsum != (long)h->total_nodes) return CO_ERR_SUM_NODES;
    return CO_OK;
}

// Per-expression bounds of the M expressions at metas, then their kernel by a
// count over the node types (the stack depth check_tree finds for a valid tree;
// the full check runs with the emission, before anything is used), and their
// program offsets: expression after expression, n_nodes words in the fast
// format, 2 * n_nodes in the wide one (node_offset order would let overlapping
// metas alias each other's instructions); a wide staged program of one leaf
// takes a third word for its variable.
static int64_t program_words(int n_nodes, bool wide, bool staged) {
    if (!wide) return n_nodes;
    return staged && n_nodes == 1 ? 3 : 2 * (int64_t)n_nodes;
}

struct Layout {
    std::vector<int32_t> depth, gen, poff, rcs;
    int64_t words = 0;
    int n_gen = 0, pieces = 1;   // pieces that the pool's threads take
    std::mutex mu;   // over most, which the ranges of emit_all add to
    Most most;
};

static int lay_out(const PopHeader *h, const int32_t *nt, const TreeMeta *metas, int M,
                   bool staged, Layout &lo) {
    const int D = h->n_vars;
    long nsum = 0;
    for (int m = 0; m < M; m++) {
        const TreeMeta &t = metas[m];
        nsum += t.n_nodes;
        if (t.K < 0 || t.n_nodes < 0 || t.node_offset < 0 || t.c_offset < 0 ||
            (long)t.node_offset + t.n_nodes > (long)h->total_nodes ||
            (long)t.c_offset + t.K > (long)h->total_c)
            return CO_ERR_PROGRAM;
        if (t.K > CO_MAX_K) return CO_ERR_BOUNDS;
    }
    lo.words = 0;
    lo.n_gen = 0;
    lo.most = Most();
    lo.depth.resize(M);
    lo.gen.resize(M);
    lo.poff.resize(M);
    lo.rcs.assign(M, CO_OK);
    const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
    // four pieces a thread, so that none waits for the slowest (with the shallow trees
    // not counted and the launch order by key, calls of one iteration on 60,000
    // expressions x 300 of 12, 20 and 27 nodes: 4.4 -> 3.8, 6.3 -> 5.6, 8.1 -> 6.7 ms)
    lo.pieces = (int)std::min<int64_t>(4 * std::min(16u, hw), nsum / kDecodeNodes + 1);
    // a valid tree of n nodes stacks at most (n + 1) / 2 values: below twice the fast
    // kernels' depth the count decides nothing
    const auto shallow = [&](const TreeMeta &t) {
        return staged && t.n_nodes < 2 * CO_FAST_MAX_STACK;
    };
    auto depth_range = [&](int m0, int m1) {
        for (int m = m0; m < m1; m++) {
            const TreeMeta &t = metas[m];
            if (shallow(t)) continue;
            const int32_t *tnt = nt + t.node_offset;
            int sp = 0, dmax = 0;
            for (int i = t.n_nodes - 1; i >= 0; i--) {
                // a leaf pushes one; a binary takes two and gives one
                sp += (tnt[i] != NODE_UFUNC) - 2 * (tnt[i] == NODE_BFUNC);
                dmax = sp > dmax ? sp : dmax;
            }
            lo.depth[m] = dmax;
            lo.gen[m] = co_fast_path(t.K, dmax, t.n_nodes, D) ? 0 : 1;
        }
    };
    int count = 0;
    for (int m = 0; m < M; m++)
        if (shallow(metas[m])) {
            lo.depth[m] = -1;
            lo.gen[m] = co_fast_path(metas[m].K, 0, metas[m].n_nodes, D) ? 0 : 1;
        } else {
            ++count;
        }
    if (count) chunked(M, lo.pieces, depth_range, depth_range);
    for (int m = 0; m < M; m++) {
        lo.poff[m] = (int32_t)lo.words;
        lo.words += program_words(metas[m].n_nodes, lo.gen[m] != 0, staged);
        lo.n_gen += lo.gen[m];
    }
    return CO_OK;
}

// Check and emit every expression: emit(m, out, scratch) returns its code.
// Expressions decode independently (C5's 1.7 M nodes take 32 ms on one thread).
template <typename Emit>
static int emit_all(const int32_t *nt, const float *nv, const int32_t *ci, const TreeMeta *metas,
                    int M, int D, bool staged, bool stage_c, uint64_t *prog, Layout &lo,
                    const Emit &emit) {
    auto range = [&](int m0, int m1) {
        TreeScratch s;
        for (int m = m0; m < m1; m++) {
            const TreeMeta &t = metas[m];
            uint64_t *out = prog + lo.poff[m];
            const int64_t words = program_words(t.n_nodes, lo.gen[m] != 0, staged);
            if (words > 0) memset(out, 0, sizeof(uint64_t) * words);
            int dd = 0;
            int rc = check_tree(nt + t.node_offset, nv + t.node_offset, ci + t.node_offset,
                                t.n_nodes, t.K, D, stage_c, &dd, s);
            if (rc == CO_OK && lo.depth[m] >= 0 && dd != lo.depth[m]) rc = CO_ERR_PROGRAM;   // never, for a valid tree
            if (rc == CO_OK) rc = emit(m, out, s);
            lo.rcs[m] = rc;
            if (rc != CO_OK) return;
        }
        std::lock_guard<std::mutex> g(lo.mu);
        lo.most.add(s.most);
    };
    auto redo = [&](int m0, int m1) {
        std::fill(lo.rcs.begin(), lo.rcs.end(), CO_OK);
        range(m0, m1);
    };
    chunked(M, lo.pieces, range, redo);
    for (int m = 0; m < M; m++)
        if (lo.rcs[m] != CO_OK) return lo.rcs[m];
    return CO_OK;
}

// Stable K bins, ascending.
static void k_bins(const TreeMeta *metas, int M, std::vector<int32_t> &start,
                   std::vector<int32_t> &ord) {
    start.assign(CO_MAX_K + 2, 0);
    for (int m = 0; m < M; m++) start[metas[m].K + 1]++;
    for (int k = 0; k <= CO_MAX_K; k++) start[k + 1] += start[k];
    std::vector<int32_t> fill(start.begin(), start.end() - 1);
    ord.resize(M);
    for (int m = 0; m < M; m++) ord[fill[metas[m].K]++] = m;
}

int decode_population(const PopHeader *h, const int32_t *nt, const float *nv,
                      const int32_t *ci, const TreeMeta *metas, uint64_t *prog,
                      int32_t *order, int32_t *bin_start, int32_t *stack, int32_t *prog_off,
                      int32_t *route) {
    int rc = check_header(h, nt, nv, ci, metas);
    if (rc != CO_OK) return rc;
    const int M = h->M_prob, D = h->n_vars;
    std::vector<uint64_t> tmp;
    if (!prog) {
        tmp.assign(h->total_nodes > 0 ? 2 * (size_t)h->total_nodes : 1, 0);
        prog = tmp.data();
    }
    Layout lo;
    rc = lay_out(h, nt, metas, M, false, lo);
    if (rc != CO_OK) return rc;
    rc = emit_all(nt, nv, ci, metas, M, D, false, true, prog, lo,
                  [&](int m, uint64_t *out, TreeScratch &s) {
        const TreeMeta &t = metas[m];
        return emit_plain(nt + t.node_offset, nv + t.node_offset, ci + t.node_offset, t.n_nodes, D,
                          lo.gen[m] != 0, out, s);
    });
    if (rc != CO_OK) return rc;
    std::vector<int32_t> start, ord;
    k_bins(metas, M, start, ord);
    if (order) memcpy(order, ord.data(), sizeof(int32_t) * M);
    if (bin_start) memcpy(bin_start, start.data(), sizeof(int32_t) * (CO_MAX_K + 2));
    if (stack) memcpy(stack, lo.depth.data(), sizeof(int32_t) * M);
    if (prog_off) memcpy(prog_off, lo.poff.data(), sizeof(int32_t) * M);
    if (route) memcpy(route, lo.gen.data(), sizeof(int32_t) * M);
    return CO_OK;
}

// The arrays of decode_range: descriptors by expression, and what their order and
// columns follow from, apart from them (a descriptor is 80 bytes, in another core's
// cache).
struct RangeScratch {
    Layout lo;
    std::vector<ExprDesc> desc;
    std::vector<uint32_t> key;
    std::vector<int32_t> vrows, v_col, launch;
    std::vector<uint64_t> a;
    // those of at most kKept expressions (31 MB) stay with the thread
    static constexpr size_t kKept = 1 << 18;
    void trim() {
        if (desc.size() <= kKept && lo.depth.size() <= kKept) return;
        std::vector<ExprDesc>().swap(desc);
        std::vector<uint32_t>().swap(key);
        std::vector<uint64_t>().swap(a);
        for (std::vector<int32_t> *v : {&vrows, &v_col, &launch, &lo.depth, &lo.gen, &lo.poff, &lo.rcs})
            std::vector<int32_t>().swap(*v);
    }
};

// Launch order by a key that sorts ascending: the general kernel's bin first, then
// the fast K bins, largest K first; within a bin by K descending (the general bin)
// and the costliest programs first (clamped to kCostBuckets).
constexpr int kCostBits = 15, kCostBuckets = 1 << kCostBits;
constexpr int kKeyBits = 1 + 6 + kCostBits, kHalfBits = kKeyBits / 2;
static_assert(CO_MAX_K < 64 && kKeyBits == 2 * kHalfBits, "two digits of the launch key");
static uint32_t launch_key(bool gen, int K, int64_t cost) {
    const uint32_t c = (uint32_t)std::min<int64_t>(cost, kCostBuckets - 1);
    return (uint32_t)!gen << (6 + kCostBits) | (uint32_t)(CO_MAX_K - K) << kCostBits |
           (kCostBuckets - 1 - c);
}

int decode_range(const PopHeader *h, const int32_t *nt, const float *nv, const int32_t *ci,
                 const TreeMeta *all_metas, int m0, int m1, int64_t word_base, uint64_t *all_prog,
                 ExprDesc *all_descs, Plan *plan) {
    const TreeMeta *metas = all_metas + m0;
    const int M = m1 - m0, D = h->n_vars;
    uint64_t *prog = all_prog + word_base;
    ExprDesc *descs = all_descs + m0;
    // working arrays kept per calling thread: for large populations fresh pages
    // cost a tenth of the decode
    static thread_local RangeScratch rs;
    struct Trim {
        RangeScratch &of;
        ~Trim() { of.trim(); }
    } trim{rs};
    Layout &lo = rs.lo;
    int rc = lay_out(h, nt, metas, M, true, lo);
    if (rc != CO_OK) return rc;
    if ((int)rs.desc.size() < M) {
        rs.desc.resize(M);
        rs.key.resize(M);
        rs.vrows.resize(M);
        rs.v_col.resize(M);
        rs.launch.resize(M);
        rs.a.resize(M);
    }
    // by pointer: on another thread `rs` names that thread's own
    ExprDesc *desc = rs.desc.data();
    uint32_t *key = rs.key.data();
    int32_t *vrows = rs.vrows.data(), *v_col = rs.v_col.data(), *launch = rs.launch.data();
    uint64_t *a = rs.a.data();
    rc = emit_all(nt, nv, ci, metas, M, D, true, stage_constants(h->N), prog, lo,
                  [&](int m, uint64_t *out, TreeScratch &s) {
        const TreeMeta &t = metas[m];
        ExprDesc &d = desc[m];
        d.prog_off = (int32_t)(word_base + lo.poff[m]);
        d.c_off = t.c_offset;
        d.y_row = m0 + m;
        d.gen = lo.gen[m];
        int64_t cost = 0;
        const int e = emit_staged(nt + t.node_offset, nv + t.node_offset, ci + t.node_offset,
                                  t.n_nodes, t.K, D, h->N, lo.gen[m] != 0, true, out, d, &cost, s);
        key[m] = launch_key(d.gen, t.K, cost);
        vrows[m] = d.vrows;
        s.most.add({d.rows, d.n_c > 0 ? d.K : 0, d.cslots});
        return e;
    });
    if (rc != CO_OK) return rc;
    // Columns by expression, and the launch order: two stable counting sorts from
    // the last expression on, by the lower and the upper half of the key.
    int64_t vcols = 0;
    int32_t next[2][(1 << kHalfBits) + 1] = {};
    constexpr uint32_t kHalf = (1u << kHalfBits) - 1;
    for (int m = 0; m < M; m++) {
        v_col[m] = (int32_t)vcols;
        vcols += vrows[m];
        next[0][(key[m] & kHalf) + 1]++;
        next[1][(key[m] >> kHalfBits) + 1]++;
    }
    for (uint32_t i = 0; i < kHalf; i++)
        for (int d = 0; d < 2; d++) next[d][i + 1] += next[d][i];
    for (int m = M - 1; m >= 0; m--)
        a[next[0][key[m] & kHalf]++] = (uint64_t)key[m] << 32 | (uint32_t)m;
    for (int p = 0; p < M; p++)
        launch[next[1][a[p] >> (32 + kHalfBits)]++] = (int32_t)a[p];
    const auto put = [&](int p0, int p1) {
        for (int p = p0; p < p1; p++) {
            const int m = launch[p];
            descs[p] = desc[m];
            descs[p].v_col = v_col[m];
        }
    };
    chunked(M, M >= 4096 ? lo.pieces : 1, put, put);
    plan->M = M;
    plan->N = h->N;
    plan->D = D;
    plan->total_nodes = h->total_nodes;
    plan->total_c = h->total_c;
    plan->max_rows = lo.most.rows;
    plan->max_ck = lo.most.ck;
    plan->max_cslots = lo.most.cslots;
    plan->words = lo.words;
    plan->vcols = vcols;
    plan->n_gen = lo.n_gen;
    return CO_OK;
}

}  // namespace cusr
