"""The page ranges the decode kernel works out without a division (decode_body.h: dec_div, dec_range),
restated here and compared with nnz * g // NG over small, large and random plans -- CPU only."""
import random


def div(x, d, m):
    t = (x * m) >> 32
    return t + (1 if (t + 1) * d <= x else 0)


def test_quotients_are_exact():
    rng = random.Random(5)
    for d in list(range(1, 300)) + [rng.randrange(300, 1 << 20) for _ in range(300)]:
        m = 0xFFFFFFFF // d
        xs = [0, 1, d - 1, d, d + 1, 2 ** 32 - 1] + [rng.randrange(1 << 32) for _ in range(20)]
        for x in xs:
            assert div(x, d, m) == x // d, (x, d)


def test_ranges_are_exact():
    rng = random.Random(6)
    for _ in range(4000):
        ng = rng.choice([rng.randrange(1, 600), rng.randrange(1, 65536)])
        nnz = rng.choice([rng.randrange(ng, ng + 5000), rng.randrange(ng, 1 << 31)])
        q, r, m = nnz // ng, nnz % ng, 0xFFFFFFFF // ng
        for g in {0, 1, ng // 2, ng - 1, ng, rng.randrange(ng + 1)}:
            assert r * g < 1 << 32
            assert q * g + div(r * g, ng, m) == nnz * g // ng, (nnz, ng, g)
