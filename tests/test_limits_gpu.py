"""GPU parity at the plan path's limits, through the C ABI, against the fp64 oracle.

* A workgroup's page list at its maximum (2048 page ids staged in LDS), and a range that would
  exceed it (the planner doubles the number of ranges), for one kv head per workgroup and for two; and
  the shorter list of the fused cascade step's decode role (1024 page ids).
* Thousands of tiny sequences: ranges hold up to 24 segments (the descriptor block's limit) and
  the planner grows the grid past one workgroup per CU.
* The same batches through the reference-shaped uniform split.
"""
import numpy as np
import pytest

import oracle
import pdattn
from _checks import check_lse, check_out
from pdattn import inputs

pytestmark = pytest.mark.gpu


def _ref(bt):
    return oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, bt.Hq, bt.Hkv, threads=8)


@pytest.mark.parametrize("lens,wg,pages_per_range", [
    ([4096 * 16], 16, 2048),          # 2 ranges of exactly 2048 pages
    ([40000, 40000], 8, 1250),        # 5000 pages: 1 range -> 2 (2500) -> 4 (1250)
], ids=["range_at_2048_pages", "range_past_2048_doubles"])
def test_full_page_lists(lens, wg, pages_per_range):
    import _gpu
    print(f"[case] full page lists lens={lens} W={wg}", flush=True)
    bt = inputs.make_batch(lens, 32, 8, seed=61)
    ro, rl = _ref(bt)
    db = _gpu.DeviceBatch(bt)
    o, l, info = _gpu.run_plan(db, wg)
    assert info.chunk_pages == pages_per_range
    segs, _ = pdattn.Plan(bt.indptr, bt.last, bt.B, 32, 8, force_workgroups=wg).schedule()
    assert max(sum(s[3] for s in ss) for ss in segs) == pages_per_range
    check_out(o, ro, tag=f"full page lists W={info.workgroups}")
    check_lse(l, rl, tag=f"full page lists W={info.workgroups}")


def test_many_tiny_sequences():
    import _gpu
    rng = np.random.default_rng(62)
    lens = [int(x) for x in rng.integers(1, 49, size=2500)]
    lens[7] = 0
    print(f"[case] {len(lens)} tiny sequences", flush=True)
    bt = inputs.make_batch(lens, 32, 8, seed=63)
    ro, rl = _ref(bt)
    db = _gpu.DeviceBatch(bt)
    o, l, info = _gpu.run_plan(db)
    segs, _ = pdattn.Plan(bt.indptr, bt.last, bt.B, 32, 8).schedule()
    most = max(len(ss) for ss in segs)
    assert info.workgroups > pdattn.device_info().compute_units   # the grid grew
    assert 12 < most <= pdattn.SCHEDULE_SEGMENTS
    check_out(o, ro, tag=f"tiny sequences plan W={info.workgroups} segs<={most}")
    check_lse(l, rl, tag="tiny sequences plan")
    o, l, nc = _gpu.run_uniform(db)
    check_out(o, ro, tag=f"tiny sequences uniform chunks={nc}")
    check_lse(l, rl, tag="tiny sequences uniform")


def _repeated_pages(bt, n, seed):
    """The batch over a cache of n pages, its page table full of repeats (long ranges in little memory)."""
    rng = np.random.default_rng(seed)
    bt.indices = rng.integers(0, n, size=bt.indices.size).astype(np.int32)
    bt.num_pages = n
    bt.q = rng.standard_normal((bt.B, bt.Hq, 128)).astype(np.float16)
    bt.k = rng.standard_normal((n, 16, bt.Hkv, 128)).astype(np.float16)
    bt.v = rng.standard_normal((n, 16, bt.Hkv, 128)).astype(np.float16)
    return bt


@pytest.mark.parametrize("pages,ranges,longest", [(4 * 256, 4, 256), (4 * 256 + 1, 4, 257), (4 * 2048, 4, 2048),
                                                  (4 * 2048 + 1, 8, 1025)])
def test_full_page_lists_of_two_heads(pages, ranges, longest):
    """The default plan of 128 kv heads: 4 ranges, two heads per workgroup, up to one page list load per
    thread (256), past it, up to the whole list and past that (the ranges double)."""
    import torch
    import _gpu
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("cases sized for 256 CUs")
    print(f"[case] full page lists of two heads, {pages} pages", flush=True)
    lens = [16 * (pages - 30) - 5, 16 * 29 + 1]
    bt = _repeated_pages(inputs.make_batch(lens, 128, 128, seed=65, fill=False), 40, 65)
    assert int(bt.indptr[-1]) == pages
    ro, rl = _ref(bt)
    o, l, info = _gpu.run_plan(_gpu.DeviceBatch(bt))
    assert info.paired == 1 and info.workgroups == ranges * 128 and info.chunk_pages == longest
    segs, _ = pdattn.Plan(bt.indptr, bt.last, bt.B, 128, 128).schedule()
    assert max(sum(s[3] for s in ss) for ss in segs) == longest
    check_out(o, ro, tag=f"{pages} pages")
    check_lse(l, rl, tag=f"{pages} pages")


@pytest.mark.parametrize("Hq", [128, 1024], ids=["G1", "G8"])
@pytest.mark.parametrize("pages,launched", [(4 * 256 + 1, 256), (4 * 1024, 256), (4 * 1024 + 1, 512)])
def test_full_page_lists_of_a_cascade_suffix(pages, launched, Hq):
    """Suffix ranges of 257 and 1024 pages (the fused step's whole list) and past it."""
    import torch
    import _gpu
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("cases sized for 256 CUs")
    print(f"[case] cascade suffix of {pages} pages, Hq={Hq}", flush=True)
    bt = inputs.make_shared_prefix_batch(64, [16 * (pages - 100) - 3, 16 * 70, 16 * 30 - 15], Hq, 128, seed=66,
                                         fill=False)
    bt = _repeated_pages(bt, 40, 66)
    for b in range(bt.B):   # (four pages of their own for the prefix; the first private pages differ)
        bt.indices[bt.indptr[b]:bt.indptr[b] + 4] = np.arange(40, 44)
        bt.indices[bt.indptr[b] + 4] = b
    rng = np.random.default_rng(67)
    bt.num_pages = 44
    bt.k = np.concatenate([bt.k, rng.standard_normal((4, 16, 128, 128)).astype(np.float16)])
    bt.v = np.concatenate([bt.v, rng.standard_normal((4, 16, 128, 128)).astype(np.float16)])
    ro, rl = _ref(bt)
    o, l, info = _gpu.run_cascade(_gpu.DeviceBatch(bt), min_prefix=16)
    assert info.use == 1 and info.prefix_tokens == 64 and info.mode == pdattn.CASCADE_FUSED
    assert info.suffix_workgroups == launched
    check_out(o, ro, tag=f"suffix of {pages} pages")
    check_lse(l, rl, tag=f"suffix of {pages} pages")
