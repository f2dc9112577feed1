// fit_kernels.hip -- instantiates the fit kernels or the pass kernels of the
// split path (lm_split.h) for one (precision, AD mode) variant and one part of
// the bins: K = 0..4, K = 5..8, K = 9..CO_FAST_MAX_K with the general kernel, or
// the groups of bins (group_top).
// Built once for each combination, so that they compile in parallel, with
//   -DCUSR_FIT_R=double|float -DCUSR_FIT_AD=0|1 -DCUSR_PART=0|1|2|3
//   -DCUSR_FIT_LAUNCH=<name> or -DCUSR_PASS_LAUNCH=<name>
#include "lm_device.h"
#include "lm_split.h"

#if !defined(CUSR_FIT_R) || !defined(CUSR_FIT_AD) || !defined(CUSR_PART) || \
    (!defined(CUSR_FIT_LAUNCH) && !defined(CUSR_PASS_LAUNCH))
#error "fit_kernels.hip needs CUSR_FIT_R, CUSR_FIT_AD, CUSR_PART and a launcher's name"
#endif

namespace cusr {

#if CUSR_PART == 0
#define CUSR_CASES CUSR_CASE(0) CUSR_CASE(1) CUSR_CASE(2) CUSR_CASE(3) CUSR_CASE(4)
#elif CUSR_PART == 1
#define CUSR_CASES CUSR_CASE(5) CUSR_CASE(6) CUSR_CASE(7) CUSR_CASE(8)
#elif CUSR_PART == 3
#define CUSR_CASES                                                                     \
    CUSR_CASE(4) CUSR_CASE(8) CUSR_CASE(group_top(9, CUSR_FIT_AD == CO_AD_REVERSE)) CUSR_CASE(15)
#else
#define CUSR_CASES                                                                    \
    CUSR_CASE(9) CUSR_CASE(10) CUSR_CASE(11) CUSR_CASE(12) CUSR_CASE(13) CUSR_CASE(14) \
    CUSR_CASE(15) CUSR_CASE(16)
#endif

#ifdef CUSR_FIT_LAUNCH
hipError_t CUSR_FIT_LAUNCH(int bin, unsigned grid, size_t lds, hipStream_t s, const FitArgs &fa) {
    if (fa.pwaves < 1 || fa.pwaves > CO_MAX_PARTITIONS || fa.parts % fa.pwaves != 0)
        return hipErrorInvalidValue;
    // a segment that can pause or resume needs the state buffer
    if (fa.it_end < 0 || fa.it_end > fa.max_iter ||
        ((fa.resume || fa.it_end < fa.max_iter) && !fa.state))
        return hipErrorInvalidValue;
    switch (bin) {
#if CUSR_PART == 3
#define CUSR_CASE(k)                                                                        \
    case k:                                                                                 \
        lm_fit_kernel<k, CUSR_FIT_R, CUSR_FIT_AD, 0, true>                                  \
            <<<grid, kLanes * fa.pwaves, lds, s>>>(fa);                                     \
        break;
#else
// the large-N instance where its tables differ (large_n_variant), chosen by N
#define CUSR_CASE(k)                                                                        \
    case k:                                                                                 \
        if constexpr (large_n_variant<CUSR_FIT_R, k, CUSR_FIT_AD>()) {                      \
            if (fa.N >= kLargeN) {                                                          \
                lm_fit_kernel<k, CUSR_FIT_R, CUSR_FIT_AD, 1>                                \
                    <<<grid, kLanes * fa.pwaves, lds, s>>>(fa);                             \
                break;                                                                      \
            }                                                                               \
        }                                                                                   \
        lm_fit_kernel<k, CUSR_FIT_R, CUSR_FIT_AD, 0><<<grid, kLanes * fa.pwaves, lds, s>>>(fa); \
        break;
#endif
        CUSR_CASES
#undef CUSR_CASE
#if CUSR_PART == 2
    case CO_GENERAL_BIN:
        lm_fit_gen_kernel<CUSR_FIT_R, CUSR_FIT_AD><<<grid, kLanes * fa.pwaves, lds, s>>>(fa);
        break;
#endif
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

#endif  // CUSR_FIT_LAUNCH

#ifdef CUSR_PASS_LAUNCH
hipError_t CUSR_PASS_LAUNCH(int bin, unsigned grid, size_t lds, hipStream_t s, const FitArgs &fa) {
    if (fa.parts < 1 || !fa.psum || !fa.state) return hipErrorInvalidValue;
    switch (bin) {
#if CUSR_PART == 3
#define CUSR_CASE(k)                                                                        \
    case k:                                                                                 \
        lm_pass_kernel<k, CUSR_FIT_R, CUSR_FIT_AD, 0, false, true>                          \
            <<<grid, kLanes, lds, s>>>(fa);                                                 \
        break;
#else
#define CUSR_CASE(k)                                                                        \
    case k:                                                                                 \
        if constexpr (large_n_variant<CUSR_FIT_R, k, CUSR_FIT_AD>()) {                      \
            if (fa.N >= kLargeN) {                                                          \
                lm_pass_kernel<k, CUSR_FIT_R, CUSR_FIT_AD, 1, false>                        \
                    <<<grid, kLanes, lds, s>>>(fa);                                         \
                break;                                                                      \
            }                                                                               \
        }                                                                                   \
        lm_pass_kernel<k, CUSR_FIT_R, CUSR_FIT_AD, 0, false><<<grid, kLanes, lds, s>>>(fa);  \
        break;
#endif
        CUSR_CASES
#undef CUSR_CASE
#if CUSR_PART == 2
    case CO_GENERAL_BIN:
        lm_pass_kernel<kGenK, CUSR_FIT_R, CUSR_FIT_AD, 0, true><<<grid, kLanes, lds, s>>>(fa);
        break;
#endif
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

#endif  // CUSR_PASS_LAUNCH

}  // namespace cusr
