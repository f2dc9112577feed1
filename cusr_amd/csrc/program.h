// program.h -- decoded expression programs shared by the host planner and
// the device interpreter.
//
// An expression (pop.bin nt/nv/ci, cusr/kernel/pop_format.h:6-16, prefix
// order) is a tree the reference evaluates last node first
// (cusr/kernel/lm_core.cuh:67), right operand before left. Here each operator
// runs after its operands, and when both operands need instructions the one
// whose subtree needs more spill slots runs first (Sethi-Ullman order; the
// right one on a tie): values, tangents and adjoints do not depend on which
// sibling runs first, and the spill slots (the LDS a wavefront reserves) stay
// at the tree's minimum. The decoded program is a list of operator
// instructions over three kinds of operand:
//   ACC   the running value, i.e. the result of the previous instruction;
//   SLOT  a spill slot holding the operand computed first while the other
//         operand's instructions run (slots are used last-in first-out);
//   VAR / CONST  a leaf, folded into the instruction that consumes it.
// Leaves therefore cost no instruction; an expression that is a single leaf
// becomes one OP_IDENT instruction.
//
// One 64-bit instruction per operator node, in execution order:
//   bits  0..5   fid     operator id (include/pop_format.h), OP_IDENT = 63
//   bit   6      binary
//   bits  7..8   a_kind  left / only operand: OPD_ACC, OPD_VAR, OPD_CONST, OPD_SLOT
//   bits  9..12  a_idx   variable index, constant rank or slot
//   bits 13..14  b_kind  right operand (binary only)
//   bits 15..18  b_idx
//   bit  19      to_slot result goes to slot d_idx instead of ACC
//   bits 20..23  d_idx
//   bits 24..28  lo      constant ranks of the left / only operand: [lo, mid)
//   bits 29..33  mid     constant ranks of the right operand: [mid, hi)
//   bits 34..38  hi      (unary: mid == hi)
//   bits 39..46  tape    first reverse-AD tape slot of this instruction
//   bit  47      sel     the partials have flat branches: where a point's
//                        partial is a structural zero its tangents become 0
//   bit  48      scale_a forward AD scales ranks [lo, mid) by the partial of
//                        the left / only operand (set when that range is
//                        non-empty and the partial is not exactly 1)
//   bit  49      scale_b forward AD scales ranks [mid, hi) by the right partial
//   bit  50      tape_a  reverse AD keeps the left / only partial in tape slot
//                        `tape`; without it the partial is never read (a
//                        variable operand) or exactly +1 (ADD, SUB's left)
//   bit  51      tape_b  the right partial is kept, in slot tape + tape_a;
//                        without it it is never read or exactly +1 (ADD) / -1
//                        (SUB)
// Constants are ranked in prefix order (cusr/benchmark/popio.py:87-91), so the
// constants of a subtree form one contiguous rank range; forward AD scales
// only those ranks.
//
// The general kernel (expressions outside co_fast_path: K up to 32, a value
// stack up to 64, any number of nodes, up to 255 variables) reads the same
// fields from two 64-bit words per instruction, wide enough for its ranges:
//   word 0: bits  0..5   fid         bit 6 binary
//           bits  7..8   a_kind      bits  9..16 a_idx
//           bits 17..18  b_kind      bits 19..26 b_idx
//           bit  27      to_slot     bits 28..35 d_idx
//           bits 36..40  sel, scale_a, scale_b, tape_a, tape_b
//   word 1: bits  0..7   lo          bits  8..15 mid      bits 16..23 hi
//           bits 24..55  tape
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../../include/cusr_co.h"

namespace cusr {

enum { OPD_ACC = 0, OPD_VAR = 1, OPD_CONST = 2, OPD_SLOT = 3 };
constexpr int OP_IDENT = 63;
constexpr int kMaxSlots = 16;                    // fast format (4-bit slot index)
constexpr int kMaxSlotsWide = CO_MAX_STACK;      // wide format

// The staged program, which the device runs. Of an expression's operators, those
// over constants alone give the same value at every point, and those over
// variables alone the same value at every iteration. On the benchmark
// populations they are a quarter to a third of the operators each (a fifth to
// 40 % of their cost each), so neither is evaluated per point and pass:
//   C  the maximal constant-only subtrees, run once per pass with one value per
//      wavefront: each leaves its value in place of its first constant (rank
//      lo) and, in forward AD, the tangents of its constants, from which the
//      per-point rows start instead of from 1;
//   V  the maximal variable-only subtrees, run in the first pass of a fit:
//      each value goes to a row of LDS and to a column of the fit's workspace,
//      which later passes load like an input variable;
//   M  everything else, run per point and pass; a C subtree is a CONST operand
//      of it, a V subtree a VAR operand.
// Every value, tangent and adjoint goes through the operations it went through
// before, in the same order, so results are bit-identical to the plain program.
// An expression without constants is one M program.
//
// The instructions are the words above with these differences: VAR and SLOT
// operands and the destination index a row of the wavefront's LDS (variables of
// M, V values, then a shared tail: V's other variables and slots, M's slots);
// in C, SLOT operands and destinations index the wavefront's scalar slots, and
// tape slots the scalar tape. The fast word adds
//   bit  52      root   C: the subtree's last instruction; M: an operand is a C
//                       subtree
//   bits 53..60  cidx   C root: the subtree's instructions; M with root: the C
//                       instruction of that subtree's root (at most one operand
//                       of an M operator is a C subtree: with two it were in C)
// and the wide words are laid out as
//   word 0: bits  0..5   fid          bit  6 binary
//           bits  7..8   a_kind       bits  9..20 a_idx
//           bits 21..27  sel, scale_a, scale_b, tape_a, tape_b, to_slot, root
//           bits 28..29  b_kind       bits 32..43 b_idx      bits 44..63 cidx
//   word 1: bits  0..7   lo           bits  8..15 mid        bits 16..23 hi
//           bits 32..43  d_idx        bits 44..63 tape
// A wide program is followed by one word per variable row, the variable's index;
// a fast one has them in ExprDesc.map, four bits each.
struct ExprDesc {          // one per expression, device-resident
    int32_t prog_off;      // first program word: C, then V, then M
    int32_t n_c, n_v, n_m; // instructions of each
    int32_t c_off;         // constants offset
    int32_t K;             // constants
    int32_t y_row;         // row of ym / output index (original expression index)
    int32_t v_col;         // first workspace column of its V values
    int32_t mvars;         // rows of variables that M reads
    int32_t vrows;         // rows of V values
    int32_t ovars;         // rows of the other variables, that V reads
    int32_t rows;          // rows in all; forward AD and values
    int32_t rows_rev;      // rows in all; reverse AD
    int32_t crow;          // reverse AD: first row of C's adjoint slots
    int32_t cslots;        // scalar slots of C
    int32_t ctape;         // scalar reverse-AD tape slots of C
    int32_t tape;          // reverse-mode tape slots of M
    int32_t gen;           // 1: wide program, general kernel
    uint64_t map;          // fast: variable index of each variable row
};

static inline __host__ __device__ int ins_fid(uint64_t w) { return (int)(w & 63u); }
static inline __host__ __device__ int ins_binary(uint64_t w) { return (int)((w >> 6) & 1u); }
static inline __host__ __device__ int ins_akind(uint64_t w) { return (int)((w >> 7) & 3u); }
static inline __host__ __device__ int ins_aidx(uint64_t w) { return (int)((w >> 9) & 15u); }
static inline __host__ __device__ int ins_bkind(uint64_t w) { return (int)((w >> 13) & 3u); }
static inline __host__ __device__ int ins_bidx(uint64_t w) { return (int)((w >> 15) & 15u); }
static inline __host__ __device__ int ins_toslot(uint64_t w) { return (int)((w >> 19) & 1u); }
static inline __host__ __device__ int ins_didx(uint64_t w) { return (int)((w >> 20) & 15u); }
static inline __host__ __device__ int ins_lo(uint64_t w) { return (int)((w >> 24) & 31u); }
static inline __host__ __device__ int ins_mid(uint64_t w) { return (int)((w >> 29) & 31u); }
// fields above bit 31 are read from the high half alone: a 64-bit mask test
// costs the device an extra scalar compare per field
static inline __host__ __device__ uint32_t ins_w1(uint64_t w) { return (uint32_t)(w >> 32); }
static inline __host__ __device__ int ins_hi(uint64_t w) { return (int)((ins_w1(w) >> 2) & 31u); }
static inline __host__ __device__ int ins_tape(uint64_t w) { return (int)((ins_w1(w) >> 7) & 255u); }
static inline __host__ __device__ int ins_sel(uint64_t w) { return (int)((ins_w1(w) >> 15) & 1u); }
static inline __host__ __device__ int ins_scale_a(uint64_t w) { return (int)((ins_w1(w) >> 16) & 1u); }
static inline __host__ __device__ int ins_scale_b(uint64_t w) { return (int)((ins_w1(w) >> 17) & 1u); }
static inline __host__ __device__ int ins_tape_a(uint64_t w) { return (int)((ins_w1(w) >> 18) & 1u); }
static inline __host__ __device__ int ins_tape_b(uint64_t w) { return (int)((ins_w1(w) >> 19) & 1u); }

// wide staged fields (word 0 a, word 1 b), each within one 32-bit half
struct Wide {
    uint64_t a, b;
};
static inline __host__ __device__ int wst_fid(uint64_t a) { return (int)(a & 63u); }
static inline __host__ __device__ int wst_bit(uint64_t a, int i) { return (int)(((uint32_t)a >> i) & 1u); }
static inline __host__ __device__ int wst_akind(uint64_t a) { return (int)(((uint32_t)a >> 7) & 3u); }
static inline __host__ __device__ int wst_aidx(uint64_t a) { return (int)(((uint32_t)a >> 9) & 4095u); }
static inline __host__ __device__ int wst_bkind(uint64_t a) { return (int)(((uint32_t)a >> 28) & 3u); }
static inline __host__ __device__ int wst_bidx(uint64_t a) { return (int)(ins_w1(a) & 4095u); }
static inline __host__ __device__ int wst_cidx(uint64_t a) { return (int)(ins_w1(a) >> 12); }
static inline __host__ __device__ int wst_lo(uint64_t b) { return (int)((uint32_t)b & 255u); }
static inline __host__ __device__ int wst_mid(uint64_t b) { return (int)(((uint32_t)b >> 8) & 255u); }
static inline __host__ __device__ int wst_hi(uint64_t b) { return (int)(((uint32_t)b >> 16) & 255u); }
static inline __host__ __device__ int wst_didx(uint64_t b) { return (int)(ins_w1(b) & 4095u); }
static inline __host__ __device__ int wst_tape(uint64_t b) { return (int)(ins_w1(b) >> 12); }
// A wavefront's scalar area (LDS), in doubles: the constants with C's values in
// place, the tangents C leaves (forward AD: t0 of them, the kernel's own K, which a
// padded or the general kernel reads whatever the expression's), C's slots and its
// reverse-AD tape.
struct UniAt {
    int t0, slot, tape, size;
};
static inline constexpr __host__ __device__ UniAt uni_at(int K, int t0, int cslots, int ctape) {
    return {K, K + t0, K + t0 + cslots, K + t0 + cslots + ctape};
}
// Bytes of the scalar area that an expression takes in a kernel of K kernel_k.
static inline __host__ __device__ int uni_bytes_of(const ExprDesc &d, bool rev, int kernel_k) {
    if (d.n_c == 0) return 0;
    const UniAt at = uni_at(d.K, rev ? 0 : kernel_k, d.cslots, rev ? d.ctape : 0);
    return (at.size * (int)sizeof(double) + 15) & ~15;
}
constexpr int kWideCidxMax = (1 << 20) - 1;   // C instructions a wide word can address
constexpr int kFastRows = 16;                 // rows a fast word can address

// The sums vector of a Jacobian pass over K constants: r^2, J^T r, then the upper
// triangle of J^T J row by row; entry (j, i), i >= j, is at sums_row(K, j) + i.
static inline constexpr __host__ __device__ int sums_width(int K) { return 1 + K + K * (K + 1) / 2; }
static inline constexpr __host__ __device__ int sums_row(int K, int j) {
    return 1 + K + j * K - (j * (j + 1)) / 2;
}
// The damped solve takes columns in fours (kSolveCols), so up to three past a
// runtime K are loaded from sums_row and not used. They lie within the vector but
// for column 3 at K = 1, which starts kSolveBefore entries before it: the kernels
// keep the constants there, in one array with the sums, and test no column.
constexpr int kSolveCols = 4, kSolveBefore = 1;

struct Plan {
    int32_t M, N, D, total_nodes, total_c;
    int32_t max_rows;      // LDS rows of a value pass
    int32_t max_ck;        // most constants of an expression with a C program (0: none)
    int32_t max_cslots;    // most scalar slots of one
    int64_t words;         // program words (fast: n_nodes per expression, wide: 2 n_nodes)
    int64_t vcols;         // workspace columns of the V values
    int32_t n_gen;         // expressions of the general kernel
};
// Doubles of the scalar area of a launch that evaluates a whole plan: sized by the
// decoded expressions, not by the header's K_max, which no check holds to them.
static inline int eval_uni_doubles(const Plan &p) {
    return p.max_ck > 0 ? uni_at(p.max_ck, 0, p.max_cslots, 0).size : 0;
}

// Check a population and decode it into plain programs (co_decode). Returns a
// CO_* code. On success fills prog[2 * total_nodes] (expression m's program
// starts at word prog_off[m]: programs are laid out expression after
// expression, n_nodes words for the fast format and 2 * n_nodes for the wide
// one; words past its instructions are 0), order[M] (stable K bins, ascending),
// bin_start[CO_MAX_K+2], stack[M] (value-stack depth, by expression),
// prog_off[M], route[M] (1: general kernel). Any output pointer may be null.
int decode_population(const PopHeader *h, const int32_t *nt, const float *nv,
                      const int32_t *ci, const TreeMeta *metas, uint64_t *prog,
                      int32_t *order, int32_t *bin_start, int32_t *stack, int32_t *prog_off,
                      int32_t *route);

// The header-level checks every decode makes first: null inputs, device
// bounds on K_max / max_stack / n_vars, and the sums of K and of n_nodes.
int check_header(const PopHeader *h, const int32_t *nt, const float *nv, const int32_t *ci,
                 const TreeMeta *metas);

// Decode expressions [m0, m1) of a population whose header passed
// check_header into staged programs, for an upload of the population as a
// whole or in pieces: the programs go to prog from word word_base on (laid out
// expression after expression as above, the descriptors' prog_off counting
// from word 0 of prog), the descriptors to descs[m0..m1) by launch position
// within the range (the general kernel's bin first, then the fast K bins,
// largest K first; y_row the population row, v_col counting from the range's
// first column). plan describes the range. The same per-expression checks and error codes as
// decode_population.
int decode_range(const PopHeader *h, const int32_t *nt, const float *nv, const int32_t *ci,
                 const TreeMeta *metas, int m0, int m1, int64_t word_base, uint64_t *prog,
                 ExprDesc *descs, Plan *plan);

// Words that the staged programs of total_nodes nodes take at most.
static inline size_t staged_words_max(int total_nodes, int n_vars) {
    return total_nodes > 0 ? (size_t)total_nodes * (n_vars > CO_FAST_MAX_VARS ? 3 : 2) : 1;
}

// Nodes a decode thread takes at least: waking the pool's threads costs about
// what one thread decodes in 20 us.
constexpr int64_t kDecodeNodes = 4096;

}  // namespace cusr
