// range_arith.h -- the page ranges of a page-range plan without divisions, for the kernels and (compiled
// by the host compiler) for tests. Range g of ngroups holds the pages [nnz g / ngroups,
// nnz (g + 1) / ngroups) of the batch's page sequence.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define PD_RANGE_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define PD_RANGE_FN inline
#endif

namespace pdattn {

// floor((2^32 - 1) / d), d > 0
PD_RANGE_FN uint32_t div_multiplier(uint32_t d) { return 0xFFFFFFFFu / d; }

// x / d for x < 2^32 without a division, m = div_multiplier(d): the high product is the quotient or one
// less.
PD_RANGE_FN uint32_t div_by(uint32_t x, uint32_t d, uint32_t m) {
    const uint32_t t = (uint32_t)(((uint64_t)x * m) >> 32);
    return t + ((t + 1) * (uint64_t)d <= x ? 1u : 0u);
}

// What a launch passes along: nnz / ngroups, nnz % ngroups and the multipliers of ngroups and Hkv.
struct RangeConsts {
    uint32_t q = 0, r = 0, m = 0, hkv_m = 0;
};
PD_RANGE_FN RangeConsts range_consts(int64_t nnz, int ngroups, int Hkv) {
    return {(uint32_t)(nnz / ngroups), (uint32_t)(nnz % ngroups), div_multiplier((uint32_t)ngroups),
            div_multiplier((uint32_t)Hkv)};
}

// nnz g / ngroups (g <= ngroups). From 65536 ranges on r g may pass 32 bits.
PD_RANGE_FN uint32_t range_start(const RangeConsts& c, int64_t nnz, int ngroups, uint32_t g) {
    if (ngroups < 65536) return c.q * g + div_by(c.r * g, (uint32_t)ngroups, c.m);
    return (uint32_t)((uint64_t)nnz * g / (uint32_t)ngroups);
}

}  // namespace pdattn
