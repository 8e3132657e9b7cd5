// launch_rules.h -- rules of the host's dispatch that are arithmetic alone (host code, no HIP).
#pragma once

#include <algorithm>
#include <cstdint>

namespace pdattn {

// Sources per row that the device-range merge sizes its round trips for. A row has at most ngroups of
// them and ngroups / B + 2 on average, but one long sequence among short ones has nearly all, so never
// fewer than 16 per trip. One sequence of 30000 tokens and 31 of 200 (64 ranges) with 8 / 16 / 32 / 64
// per trip: 37.7 / 35.8 / 35.2 / 35.3 us, and 63 of 200 42.0 / 40.0 / 40.3 / 41.6; 32 ragged sequences of
// 200-6000 73.2 / 72.4 / 72.9 / 73.7.
inline int merge_ranges_sources(int ngroups, int B) { return std::min(ngroups, std::max(ngroups / B + 2, 16)); }

// The uniform split's launch: `chunks` (chunk, sequence) pairs of Hkv kv heads as items of hp heads of one
// chunk, `per` items per workgroup, W workgroups. A workgroup holds at most seg_max items.
struct UniformSplit {
    int hp;
    int64_t items, per, W;
};
inline UniformSplit uniform_items(int64_t chunks, int Hkv, int hp, int64_t cus, int64_t seg_max) {
    const int64_t items = chunks * (Hkv / hp);
    const int64_t per = std::max<int64_t>(1, std::min((items + cus - 1) / cus, seg_max));
    return {hp, items, per, (items + per - 1) / per};
}
// One or two heads per item: two read 512 contiguous bytes of every token row, which streams faster, but
// make the items twice as long, so that the last round of workgroups may leave more of the chip idle. Two
// need items enough for every CU (8 x 8192 tokens in 4 chunks: 47.9 us with one head, 54.1 with two); then
// they are taken unless the longest workgroup grows by more than a quarter and fewer than three quarters of
// the CUs have one. Chunks of 1024 tokens, 8 kv heads, one / two heads: 65 sequences 49.3 / 54.4 us, 88
// 58.4 / 61.3, 96 65.8 / 65.1, 100 74.2 / 67.2; 200 of 300 tokens 45.4 / 43.6, 140 of 256 30.4 / 28.0; 17 of
// 1024 with 32 kv heads 51.1 / 53.3.
inline UniformSplit uniform_split(int64_t chunks, int Hkv, int64_t cus, int64_t seg_max) {
    const UniformSplit one = uniform_items(chunks, Hkv, 1, cus, seg_max);
    if (Hkv % 2 != 0 || one.items < 2 * cus) return one;
    const UniformSplit two = uniform_items(chunks, Hkv, 2, cus, seg_max);
    auto longest = [&](const UniformSplit& u) { return (u.W + cus - 1) / cus * u.per * u.hp; };
    return 4 * longest(two) <= 5 * longest(one) || 4 * two.W >= 3 * cus ? two : one;
}

// Whether a uniform-split workgroup at G <= 4 holds two 32-key blocks per wave in LDS (decode_body.h). A
// second block in flight pays where it is all there is to start with, but its q rows then go through LDS
// with every block. One / two, us: 8 x 8192 tokens 47.7 / 48.3, 1 x 32768 27.9 / 28.2, 33 of 66-333 13.3 /
// 13.9, 65 of 666-3333 with 4 kv heads 71.6 / 74.5; with one item of up to 32 pages per workgroup two are
// faster at G = 1 (32 kv heads: 2 of 66-333 7.04 / 6.76, 2 of 233-1166 9.55 / 9.34, 8 of 66-333 9.96 / 9.77)
// and within 0.3 either way at G = 4.
inline bool uniform_two_slots(int64_t per, int64_t pages_per_item) { return per == 1 && pages_per_item <= 32; }

// Whether a plan of two kv heads per workgroup at G <= 4 holds one block per wave instead. One is faster where
// a range holds a few blocks per wave, of several sequences; its q rows then come to registers once per
// segment, which very short segments wait for, the more heads the longer. So: at least 12 sequences, at most
// 64 pages per range, and at least 4 pages per sequence at G <= 2, 20 at G = 4. One / two, us: G = 4, 64 x 1024
// tokens 41.8 / 42.4, 20 of 300-1000 with 16 kv heads 25.0 / 25.8, but 64 of 7-224 15.8 / 15.5 and 64 of 11-67
// 15.8 / 15.2; G = 2, 32 of 300-1000 20.2 / 20.8, 128 of 7-224 19.8 / 20.4; G = 1, 37 of 18-432 with 16 kv heads
// 18.0 / 18.7 (18.0 with the vector-unit body), 32 of 7-224 with 32 19.2 / 20.3, but 200 of 11-67 41.4 / 40.8.
// Past 64 pages two are as fast or faster at G = 1 (128 of 16-512 with 32 kv heads, 131 pages, 95.2 / 94.5)
// and within 0.6% at G = 2 and 4; of fewer sequences some are faster with two (6 of 512-2560 13.7 / 13.4, 1 x
// 32768 26.8 / 26.2) and with one head per workgroup as many lose as gain (12 of 18-432, 16 kv heads, 12.1 /
// 11.7).
inline bool plan_one_slot(int64_t B, int64_t nnz, int64_t ngroups, int G) {
    return B >= 12 && nnz <= 64 * ngroups && nnz >= (G <= 2 ? 4 : 20) * B;
}

// Kv heads per workgroup of the device-range decode over `cus` CUs. Two heads stream faster but double the
// ranges, and so the partials of every long sequence; the lengths are not known here, only that a sequence
// attends at most per_seq pages. Two from 16 such pages per range on (about 8 real ones in a ragged batch,
// as in a plan), or with more sequences than ranges of one head; never for one sequence. One / two heads,
// us: 1 x 2048 tokens 9.0 / 9.7, 1 x 32768 28.3 / 28.8, 4 of 200-900 11.2 / 11.6, 8 of 94-988 12.4 / 12.6,
// with 32 kv heads 19.2 / 18.7, 32 of 200-6000 73.2 / 72.4, one of 30000 and 15 of 200 33.5 / 32.4.
inline int device_range_heads(int64_t B, int64_t per_seq, int Hkv, int64_t cus) {
    if (Hkv % 2 != 0 || B < 2) return 1;
    const int64_t ranges = std::max<int64_t>(1, cus / Hkv);
    return B * per_seq >= 16 * 2 * ranges || B > ranges ? 2 : 1;
}

}  // namespace pdattn
