// The dispatch rules of csrc/launch_rules.h behind C functions, for tests/test_launch_rules.py.
#include "../../cuda-kernel-lab_amd/csrc/launch_rules.h"

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

int rule_device_range_heads(int64_t B, int64_t per_seq, int Hkv, int64_t cus) {
    return pdattn::device_range_heads(B, per_seq, Hkv, cus);
}

}
