// launch_plan.h -- the launches of one fit, planned on the host from the decoded
// descriptors: bins of K, groups of bins, streams, workgroups and their LDS.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "lm_device.h"

namespace cusr {

// K bins run concurrently on the handle's stream and kExtraStreams more. HIP maps
// each stream of a process to one of GPU_MAX_HW_QUEUES (4) hardware queues,
// and two streams that share a queue run one after the other: a fifth stream
// was measured sharing a queue and serialising its bins behind another's
// (C2: 20.5 ms, the sum of the two streams' bins). So four streams in all.
constexpr int kExtraStreams = 3;
constexpr int kStreams = kExtraStreams + 1;
// wavefronts of a K bin below which bins are grouped (in-workgroup, split path)
constexpr int kGroupWaves = 1024, kGroupWavesSplit = 4096;

// the launcher's choice of instance (fit_kernels.hip): the large-N one from
// kLargeN points where its tables differ
template <typename R, int AD>
static inline size_t lds_for_k(int K, int N, int rows, int tape) {
    switch (K) {
#define CUSR_LDS_CASE(k)                                                        \
    case k:                                                                     \
        return (large_n_variant<R, k, AD>() && N >= kLargeN)                    \
                   ? fit_lds_bytes_t<R, k, AD, 1>(rows, tape)                   \
                   : fit_lds_bytes_t<R, k, AD, 0>(rows, tape);
    CUSR_LDS_CASE(0) CUSR_LDS_CASE(1) CUSR_LDS_CASE(2) CUSR_LDS_CASE(3) CUSR_LDS_CASE(4)
    CUSR_LDS_CASE(5) CUSR_LDS_CASE(6) CUSR_LDS_CASE(7) CUSR_LDS_CASE(8) CUSR_LDS_CASE(9)
    CUSR_LDS_CASE(10) CUSR_LDS_CASE(11) CUSR_LDS_CASE(12) CUSR_LDS_CASE(13)
    CUSR_LDS_CASE(14) CUSR_LDS_CASE(15) CUSR_LDS_CASE(16)
#undef CUSR_LDS_CASE
    default: return 0;
    }
}

static inline size_t fit_lds_bytes(bool mixed, bool rev, int K, int N, int rows, int tape) {
    if (K == CO_GENERAL_BIN)
        return mixed ? fit_lds_bytes_gen<float>(rows, tape)
                     : fit_lds_bytes_gen<double>(rows, tape);
    if (mixed)
        return rev ? lds_for_k<float, CO_AD_REVERSE>(K, N, rows, tape)
                   : lds_for_k<float, CO_AD_FORWARD>(K, N, rows, tape);
    return rev ? lds_for_k<double, CO_AD_REVERSE>(K, N, rows, tape)
               : lds_for_k<double, CO_AD_FORWARD>(K, N, rows, tape);
}

// dynamic LDS a workgroup of a bin's fit kernel may use: the device's LDS per
// workgroup less the kernel's static arrays (constants and pass sums)
static inline size_t max_dyn_lds(size_t lds_per_block, int bin) {
    const size_t st = fit_static_lds(bin);
    return lds_per_block > st ? lds_per_block - st : 0;
}

// One launch of a fit: its bin, workgroups, LDS and stream (planned before
// anything is launched, so a launch that cannot fit is refused up front).
struct LaunchPlan {
    int bin, pos, cnt, rows, tape, uni, kmax, stream;   // uni: doubles of the scalar area
    size_t gen_bytes;   // general bin: the LDS of its largest expression's wavefront
    uint32_t bins;   // the bins it covers, bit by bit (a group: several)
    bool group;      // run by the padded kernel of group_top
    size_t wave_bytes;
    int pwaves[2];
    size_t lds[2];
};

// The K of a launch's kernel, by which it holds tangents (sums: by the expression's
// own in the general kernel).
static inline int kernel_k(const LaunchPlan &b) { return b.bin == CO_GENERAL_BIN ? kGenK : b.bin; }

// Bytes of a launch's per-wavefront scalar area.
static inline int uni_bytes(const LaunchPlan &b) { return (b.uni * (int)sizeof(double) + 15) & ~15; }

// What a plan depends on beside the descriptors.
struct PlanArgs {
    bool rev, mixed, split, group;   // group: small bins may be launched in groups
    int N, parts;                    // points, partitions
    int nseg, seg_parts[2];          // segments of the iteration loop, their partitions
    size_t lds_per_block;
};

// The bins of descriptors [p0, p1) in launch order: the general kernel's
// bin, then the fast K bins, largest K first. The streams are dealt
// round-robin in that order (stream kExtraStreams is the handle's own).
// The kernel launched first on a stream takes the machine first and so
// ends first, so each stream's next bin is the next largest; this beats
// balancing estimated costs over the streams (C2 12.15 -> 11.66 ms, C4
// 173 -> 170 ms, C3 139.7 -> 137.8 ms on an MI355X). A general bin of at
// least a sixteenth of the range's expressions is the exception: one
// wavefront per expression at one point per lane, it outlasts any fast bin
// many times over, so it gets stream 0 to itself and the fast bins are
// dealt over the other three (a GP-generation population, a fifth of it
// general: the fast bins dealt behind it on stream 0 had waited for it,
// 74.6 ms per fit against the general bin's 45 ms).
// Bins too small to fill the chip four at a time are launched in groups
// (group_top), by the padded kernel of the group's largest K: queued behind
// each other, every bin waits for the slowest expression of the one before.
// Measured, one launch per bin -> groups: 700 x 777 reverse AD, K 2-14: 14.2
// -> 5.0 ms; 24 x 1,000,003: 12.3 -> 5.0 ms; 1,000 x 1,000, K 0-8: 2.67 -> 1.77
// ms; 4,000 x 1,000, K 1-28: 35.9 -> 29.6 ms. Larger bins keep their own
// kernels, with fewer registers and no padded sums: at 2,000 wavefronts a bin
// 4.24 ms against 4.60 grouped (K 1-8, N = 1,024), at 1,000 equal. On the split
// path every launch waits for all of the one before, pass and step in turn, so
// groups pay for longer: 1,024 x 100,000 (2,048 a bin) 27.2 -> 22.0 ms, 3,000 x
// 2,048 reverse AD (1,850) 26.5 -> 24.8 ms, 8,192 x 2,048 (5,040) 66.9 against
// 68.6 grouped.
static inline int plan_launches(const ExprDesc *desc, int p0, int p1, const PlanArgs &a, LaunchPlan *lp,
                                int *nl_out, int *kmax_out) {
    const bool rev = a.rev, mixed = a.mixed, split = a.split;
    int nl = 0, kmax = 0, pos = p0, fast = 0, fast_bins = 0;
    for (int i = 0; i < CO_BINS; ++i) {
        const int bin = i == 0 ? CO_GENERAL_BIN : CO_FAST_MAX_K - (i - 1);
        const bool gen = bin == CO_GENERAL_BIN;
        LaunchPlan b = {};
        b.bin = bin;
        b.bins = 1u << bin;
        b.pos = pos;
        while (pos < p1 && (gen ? desc[pos].gen != 0
                                : (!desc[pos].gen && desc[pos].K == bin))) {
            const ExprDesc &d = desc[pos];
            const int rows = rev ? d.rows_rev : d.rows;
            const int uni = d.n_c ? uni_at(d.K, 0, d.cslots, rev ? d.ctape : 0).size : 0;
            if (rows > b.rows) b.rows = rows;
            if (uni > b.uni) b.uni = uni;
            if (d.tape > b.tape) b.tape = d.tape;
            if (gen) {
                const size_t own = (size_t)uni_bytes_of(d, rev, kGenK) +
                                   fit_lds_bytes(mixed, rev, bin, a.N, rows, rev ? d.tape : 0);
                if (own > b.gen_bytes) b.gen_bytes = own;
            }
            if (d.K > b.kmax) b.kmax = d.K;
            ++b.cnt;
            ++pos;
        }
        if (b.cnt == 0) continue;
        if (!rev) b.tape = 0;
        if (!gen) {
            fast += b.cnt;
            ++fast_bins;
        }
        lp[nl++] = b;
    }
    if (pos != p1) return CO_ERR_PROGRAM;   // descriptors out of launch order: never
    if (a.group && a.nseg == 1 &&
        (long)fast * a.parts < (long)fast_bins * (split ? kGroupWavesSplit : kGroupWaves)) {
        int n = 0;
        for (int i = 0; i < nl; ++i) {
            const LaunchPlan b = lp[i];
            const int top = b.bin == CO_GENERAL_BIN ? -1 : group_top(b.bin, rev);
            if (n > 0 && top >= 0 && lp[n - 1].bin != CO_GENERAL_BIN &&
                group_top(lp[n - 1].bin, rev) == top) {
                LaunchPlan &g = lp[n - 1];
                g.bin = top;
                g.group = true;
                g.bins |= b.bins;
                g.cnt += b.cnt;
                g.rows = g.rows > b.rows ? g.rows : b.rows;
                g.tape = g.tape > b.tape ? g.tape : b.tape;
                g.uni = g.uni > b.uni ? g.uni : b.uni;
                g.kmax = top;
            } else {
                lp[n++] = b;
            }
        }
        nl = n;
    }
    bool gen_alone = false;
    for (int i = 0; i < nl; ++i) {
        LaunchPlan &b = lp[i];
        const bool gen = b.bin == CO_GENERAL_BIN;
        if (b.kmax > kmax) kmax = b.kmax;
        if (gen) gen_alone = (long)b.cnt * 16 >= (long)(p1 - p0) && b.cnt < p1 - p0;
        // the handle's own stream first: a fit of one launch waits for no other
        const int lane = !gen_alone ? i % kStreams : (gen ? 0 : 1 + (i - 1) % (kStreams - 1));
        b.stream = (lane + kExtraStreams) % kStreams;
        // forward AD: the tangents that C leaves, to the kernel's K
        if (b.uni > 0 && !rev) b.uni += kernel_k(b);
        // per-wavefront areas, then the partition sums; fewer wavefronts per
        // workgroup (each summing several partitions) when LDS is short. The
        // split path's pass workgroups are one wavefront with no partition
        // sums in LDS.
        const int N = b.group ? 0 : a.N;   // a group has no large-N instance
        const size_t own = gen ? b.gen_bytes
                               : uni_bytes(b) + fit_lds_bytes(mixed, rev, b.bin, N, b.rows, b.tape);
        b.wave_bytes = (own + 15) & ~(size_t)15;
        const size_t cap = max_dyn_lds(a.lds_per_block, b.bin);
        const int ks = gen ? b.kmax : b.bin;
        for (int g = 0; g < (b.kmax == 0 || split ? 1 : a.nseg); ++g) {
            const int sp = split ? 1 : a.seg_parts[g];
            const size_t part_bytes = sp > 1 ? (size_t)sp * sums_width(ks) * 8 : 0;
            int pw = sp;
            while (pw > 1 && pw * b.wave_bytes + part_bytes > cap) pw /= 2;
            b.pwaves[g] = pw;
            b.lds[g] = pw * b.wave_bytes + part_bytes;
            if (b.lds[g] > cap) return CO_ERR_BOUNDS;   // before any launch
        }
    }
    *nl_out = nl;
    *kmax_out = kmax;
    return CO_OK;
}

}  // namespace cusr
