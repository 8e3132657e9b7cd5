"""The host's dispatch rules (csrc/launch_rules.h, compiled here with the host compiler) -- CPU only."""
import ctypes

import pytest


@pytest.fixture
def rules(host_rules):
    return host_rules


def test_merge_trips_fit_the_longest_row(rules):
    """A row's sources in at most four trips for up to 64 ranges, whatever the average; no trip sized past
    the number of ranges."""
    for ngroups in (1, 2, 8, 16, 32, 64):
        for B in (1, 2, 3, 8, 16, 32, 64, 128, 1023):
            n = rules.rule_merge_ranges_sources(ngroups, B)
            assert 1 <= n <= ngroups
            assert -(-ngroups // n) <= 4, (ngroups, B, n)
            assert n >= min(ngroups, ngroups // B + 2)


def _uniform(rules, chunks, Hkv, cus=256, seg_max=24):
    out = (ctypes.c_int64 * 4)()
    rules.rule_uniform_split(ctypes.c_int64(chunks), Hkv, ctypes.c_int64(cus), ctypes.c_int64(seg_max), out)
    return list(out)


def test_uniform_split_covers_the_items(rules):
    for Hkv in (1, 2, 3, 8, 16, 32):
        for chunks in list(range(1, 300)) + [1000, 4097, 100000]:
            for seg_max in (1, 7, 24):
                hp, items, per, W = _uniform(rules, chunks, Hkv, seg_max=seg_max)
                assert hp in (1, 2) and Hkv % hp == 0 and items * hp == chunks * Hkv
                assert 1 <= per <= seg_max and (W - 1) * per < items <= W * per


def test_two_heads_per_item_leave_no_more_of_the_chip_idle(rules):
    """Two heads where the longest workgroup is at most a quarter longer or three quarters of the CUs
    have one; never with fewer items than would keep every CU busy."""
    for Hkv in (2, 8, 32):
        for chunks in range(1, 1200):
            hp, items, per, W = _uniform(rules, chunks, Hkv)
            if hp == 1:
                continue
            assert items >= 256
            one = min(24, -(-chunks * Hkv // 256))
            assert W >= 192 or 2 * per <= 1.25 * one or W > 256, (Hkv, chunks)
    assert [_uniform(rules, n, 8)[0] for n in (32, 65, 88, 96, 100, 140, 200)] == [1, 1, 1, 2, 2, 2, 2]
    assert _uniform(rules, 17, 32)[0] == 1
    assert _uniform(rules, 64, 7)[0] == 1


def test_uniform_split_slots(rules):
    """Two blocks per wave only where a workgroup has one short item."""
    def two(per, pages):
        f = rules.rule_uniform_two_slots
        f.restype = ctypes.c_bool
        return f(ctypes.c_int64(per), ctypes.c_int64(pages))
    assert [two(1, n) for n in (2, 32, 33, 129, 2048)] == [True, True, False, False, False]
    assert not two(2, 2) and not two(24, 32)


def test_plan_slots(rules):
    """One block per wave for 12 and more sequences of 4 (G <= 2) or 20 pages and more each, up to 64 pages
    per range."""
    def one(B, nnz, ngroups, G):
        f = rules.rule_plan_one_slot
        f.restype = ctypes.c_bool
        return f(ctypes.c_int64(B), ctypes.c_int64(nnz), ctypes.c_int64(ngroups), G)
    for G, least in ((1, 4), (2, 4), (4, 20)):
        assert [one(B, 30 * B, 32, G) for B in (1, 11, 12, 60)] == [False, False, True, True]
        assert one(64, 64 * 64, 64, G) and not one(64, 64 * 64 + 1, 64, G)
        assert one(64, least * 64, 64, G) and not one(64, least * 64 - 1, 64, G)


def test_device_ranges_of_short_batches_keep_one_head(rules):
    """Two heads only where every range holds enough pages, or there are more sequences than ranges."""
    def heads(B, longest, Hkv, cus=256):
        return rules.rule_device_range_heads(ctypes.c_int64(B), ctypes.c_int64(longest // 16 + 2), Hkv,
                                             ctypes.c_int64(cus))
    assert [heads(1, n, 8) for n in (16, 2048, 32768, 200000)] == [1, 1, 1, 1]
    assert [heads(B, 988, 8) for B in (2, 4, 8, 17, 32)] == [1, 1, 1, 2, 2]
    assert heads(32, 6000, 8) == 2 and heads(33, 16, 8) == 2 and heads(32, 16, 8) == 1
    assert heads(8, 988, 32) == 2 and heads(64, 4096, 7) == 1
    assert heads(300, 16, 512) == 2   # more kv heads than CUs


def test_items_per_workgroup_of_the_parity_cases(rules):
    """What the uniform split's GPU parity cases say they cover (300 sequences, 256 CUs)."""
    assert [_uniform(rules, 300 * nc, 8)[:3:2] for nc in (1, 2, 3, 6)] == [[2, 5], [2, 10], [2, 15], [2, 24]]
    assert _uniform(rules, 300 * 4, 7)[:3:2] == [1, 24]
