"""The page ranges the decode kernel works out without a division (csrc/range_arith.h, compiled here with
the host compiler), compared with nnz * g // ngroups over small, large and random plans, on both sides of
the 65536 ranges where 32 bits stop being enough -- CPU only."""
import ctypes
import random


def test_quotients_are_exact(host_rules):
    rng = random.Random(5)
    div = host_rules.rule_div
    div.argtypes, div.restype = [ctypes.c_uint32] * 2, ctypes.c_uint32
    for d in list(range(1, 300)) + [rng.randrange(300, 1 << 20) for _ in range(300)] + [2 ** 31, 2 ** 32 - 1]:
        xs = [0, 1, d - 1, d, min(d + 1, 2 ** 32 - 1), 2 ** 32 - 1] + [rng.randrange(1 << 32) for _ in range(20)]
        for x in xs:
            assert div(x, d) == x // d, (x, d)


def test_ranges_are_exact(host_rules):
    rng = random.Random(6)
    start = host_rules.rule_range_start
    start.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_uint32]
    start.restype = ctypes.c_uint32
    group = host_rules.rule_group_of
    group.argtypes, group.restype = [ctypes.c_uint32, ctypes.c_int64, ctypes.c_int, ctypes.c_int], ctypes.c_uint32
    for _ in range(4000):
        ng = rng.choice([rng.randrange(1, 600), rng.randrange(1, 65536), 65535, 65536, rng.randrange(65536, 1 << 24)])
        nnz = rng.choice([rng.randrange(ng, ng + 5000), rng.randrange(ng, (1 << 31) - 1)])
        Hkv = rng.choice([1, 2, 3, 7, 8, 32, 128])
        for g in {0, 1, ng // 2, ng - 1, ng, rng.randrange(ng + 1)}:
            assert start(nnz, ng, Hkv, g) == nnz * g // ng, (nnz, ng, g)
        w = rng.randrange(min(ng * Hkv, 1 << 32))
        assert group(w, nnz, ng, Hkv) == w // Hkv
