// The dispatch rules of csrc/launch_rules.h and the range arithmetic of csrc/range_arith.h behind C
// functions, for tests/test_launch_rules.py and tests/test_range_arithmetic.py.
#include "../../cuda-kernel-lab_amd/csrc/launch_rules.h"
#include "../../cuda-kernel-lab_amd/csrc/range_arith.h"

extern "C" {

int rule_merge_ranges_sources(int ngroups, int B) { return pdattn::merge_ranges_sources(ngroups, B); }

// out: heads per item, items, items per workgroup, workgroups
void rule_uniform_split(int64_t chunks, int Hkv, int64_t cus, int64_t seg_max, int64_t* out) {
    const pdattn::UniformSplit u = pdattn::uniform_split(chunks, Hkv, cus, seg_max);
    out[0] = u.hp;
    out[1] = u.items;
    out[2] = u.per;
    out[3] = u.W;
}

bool rule_uniform_two_slots(int64_t per, int64_t pages) { return pdattn::uniform_two_slots(per, pages); }

bool rule_plan_one_slot(int64_t B, int64_t nnz, int64_t ngroups, int G) {
    return pdattn::plan_one_slot(B, nnz, ngroups, G);
}

int rule_device_range_heads(int64_t B, int64_t per_seq, int Hkv, int64_t cus) {
    return pdattn::device_range_heads(B, per_seq, Hkv, cus);
}

uint32_t rule_div(uint32_t x, uint32_t d) { return pdattn::div_by(x, d, pdattn::div_multiplier(d)); }
uint32_t rule_range_start(int64_t nnz, int ngroups, int Hkv, uint32_t g) {
    return pdattn::range_start(pdattn::range_consts(nnz, ngroups, Hkv), nnz, ngroups, g);
}
// w / Hkv as the kernel works it out
uint32_t rule_group_of(uint32_t w, int64_t nnz, int ngroups, int Hkv) {
    return pdattn::div_by(w, (uint32_t)Hkv, pdattn::range_consts(nnz, ngroups, Hkv).hkv_m);
}

}
