"""The MFMA decode body at the sizes where it can go wrong, against the fp64 oracle: sequences around
one and two pages, around a wave's share (its 32-key blocks with one page or none of its own) and
around a workgroup's, for every group size and for one and two kv heads per workgroup, through the
plan path, the uniform split, its fp32 partials and the device-range drop-in, with NaN and Inf in
every cache slot that holds no key; infinite V values in keys that count, weights far below the largest.

The weights of the PV product are fp32 in three fp16 parts, so the fp32 partials are held to fp32's
own accuracy: n keys in fp32 sums give about 2^-24 sqrt(n) of the result, and four times that is
allowed.
"""
import numpy as np
import pytest

import oracle
from _checks import check_lse, check_out
from pdattn import inputs

pytestmark = pytest.mark.gpu

HEADS = [(8, 8), (16, 8), (32, 8), (64, 8), (3, 3), (24, 3), (2, 1), (16, 2)]
LENS = [1, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 0, 127, 128, 129, 255, 257, 513]


def _poison(bt):
    """NaN / Inf in every slot of K and V past a sequence's end."""
    for b in range(bt.B):
        pb, pe = int(bt.indptr[b]), int(bt.indptr[b + 1])
        if pe > pb and int(bt.last[b]) < 16:
            page, n = int(bt.indices[pe - 1]), int(bt.last[b])
            bt.k[page, n::2] = np.float16(np.nan)
            bt.v[page, n::2] = np.float16(np.inf)
            bt.k[page, n + 1::2] = np.float16(-np.inf)
            bt.v[page, n + 1::2] = np.float16(np.nan)


@pytest.mark.parametrize("Hq,Hkv", HEADS, ids=[f"{q}x{k}" for q, k in HEADS])
def test_block_edges(Hq, Hkv):
    import _gpu
    print(f"[case] block edges Hq={Hq} Hkv={Hkv}", flush=True)
    bt = inputs.make_batch(LENS, Hq, Hkv, seed=71)
    ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, threads=8)
    _poison(bt)
    db = _gpu.DeviceBatch(bt)
    for wg in (0, 5, Hkv, 16 * Hkv):
        o, l, info = _gpu.run_plan(db, wg)
        check_out(o, ro, tag=f"plan W={info.workgroups}")
        check_lse(l, rl, tag=f"plan W={info.workgroups}")
    for force in (1, 3):
        o, l, nc = _gpu.run_uniform(db, force)
        check_out(o, ro, tag=f"uniform {nc} chunks")
        check_lse(l, rl, tag=f"uniform {nc} chunks")
    o, l = _gpu.run_balanced(db)
    check_out(o, ro, tag="device ranges")
    check_lse(l, rl, tag="device ranges")


@pytest.mark.parametrize("Hq,Hkv", HEADS, ids=[f"{q}x{k}" for q, k in HEADS])
def test_partials_keep_fp32_accuracy(Hq, Hkv):
    """Unaligned starts and chunks (an edge block at both ends of a range)."""
    import _gpu
    print(f"[case] partials Hq={Hq} Hkv={Hkv}", flush=True)
    bt = inputs.make_batch([300, 77, 16, 450], Hq, Hkv, seed=72)
    nc, ct, kv_start = 4, 100, 23
    ro, rl = oracle.partials(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, nc, ct, kv_start)
    po, pl = _gpu.run_partials(_gpu.DeviceBatch(bt), nc, ct, kv_start)
    check_lse(pl, rl, tag="partial lse")
    assert np.linalg.norm(po - ro) <= 4 * 2.0 ** -24 * np.sqrt(ct) * np.linalg.norm(ro)


@pytest.mark.parametrize("Hq", [8, 16, 32, 64], ids=["G1", "G2", "G4", "G8"])
def test_paired_plans_with_one_and_two_blocks_per_wave(Hq):
    """Two kv heads per workgroup, block edges and poison: 36 short sequences (6 pages each: one LDS block per
    wave at G <= 2), 30 with long ones among them (26 pages each: one), 16 longer ones and 11 (two)."""
    import _gpu
    print(f"[case] paired plans Hq={Hq}", flush=True)
    long = [1000 - 13 * i for i in range(12)]
    for lens in (LENS * 2, LENS + long, [5000 - 77 * i for i in range(16)], [900 + i for i in range(11)]):
        bt = inputs.make_batch(lens, Hq, 8, seed=80)
        ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, 8, threads=8)
        _poison(bt)
        o, l, info = _gpu.run_plan(_gpu.DeviceBatch(bt))
        assert info.paired == 1
        check_out(o, ro, tag=f"{len(lens)} sequences")
        check_lse(l, rl, tag=f"{len(lens)} sequences")


@pytest.mark.parametrize("chunk_tokens", [495, 497, 512])
@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (32, 8), (64, 8)], ids=["G1", "G2", "G4", "G8"])
def test_uniform_partials_where_the_layout_changes(Hq, Hkv, chunk_tokens):
    """Items of 32 and 33 pages, and two items per workgroup (36 x 8): one and two LDS blocks per wave;
    unaligned starts."""
    import _gpu
    print(f"[case] uniform layouts Hq={Hq} Hkv={Hkv} chunk={chunk_tokens}", flush=True)
    for lens in ([1200, 33, 700], [int(x) for x in range(480, 552, 2)]):
        bt = inputs.make_batch(lens, Hq, Hkv, seed=79)
        nc = 2 if bt.B == 3 else 1
        ro, rl = oracle.partials(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, nc, chunk_tokens, 23)
        po, pl = _gpu.run_partials(_gpu.DeviceBatch(bt), nc, chunk_tokens, 23)
        check_lse(pl, rl, tag="partial lse")
        assert np.linalg.norm(po - ro) <= 4 * 2.0 ** -24 * np.sqrt(chunk_tokens) * np.linalg.norm(ro)


def test_infinite_values():
    """An infinite V makes its dim infinite in every head (its weight's low half must not turn it into
    NaN) and leaves the other dims alone."""
    import _gpu
    print("[case] infinite V values", flush=True)
    bt = inputs.make_batch([70, 5, 200], 32, 8, seed=73)
    bt.q *= np.float16(0.125)   # weights of the same order
    ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, 32, 8, threads=8)
    for b in range(bt.B):
        page = int(bt.indices[int(bt.indptr[b])])
        bt.v[page, 2, :, 17] = np.float16(np.inf)
        bt.v[page, 3, :, 90] = np.float16(-np.inf)
    o, l, _ = _gpu.run_plan(_gpu.DeviceBatch(bt))
    assert np.all(o[..., 17] == np.inf) and np.all(o[..., 90] == -np.inf)
    keep = [d for d in range(128) if d not in (17, 90)]
    check_out(o[..., keep], ro[..., keep], tag="other dims")
    check_lse(l, rl, tag="infinite V")


def _peaked(Hq, Hkv, gap, seed, lens=(300, 41, 513)):
    """Every sequence has one key (token 5) whose score is about `gap` above all the others', for every
    head, and whose V is 0 in dims 0-63: those dims are made of weights around exp(-gap) alone."""
    bt = inputs.make_batch(list(lens), Hq, Hkv, seed=seed)
    rng = np.random.default_rng(seed)
    u = rng.choice([-1.0, 1.0], 128)
    bt.q[:] = (4 * u + 0.1 * rng.standard_normal(bt.q.shape)).astype(np.float16)
    bt.k[:] = (0.005 * rng.standard_normal(bt.k.shape)).astype(np.float16)
    for b in range(bt.B):
        page = int(bt.indices[int(bt.indptr[b])])
        bt.k[page, 5] = (gap * np.sqrt(128.0) / (4 * 128) * u).astype(np.float16)
        bt.v[page, 5, :, :64] = 0
    return bt


@pytest.mark.parametrize("gap", [6, 12, 18, 24])
@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (32, 8), (64, 8)], ids=["G1", "G2", "G4", "G8"])
def test_small_weights_keep_fp32_accuracy(Hq, Hkv, gap):
    """Weights of 2^-9 to 2^-35 of the largest. The scores are fp32: a rounding of 2^-24 of a score up to
    gap + 1 (in base 2, 1.45 times that) moves a weight by as much, four of them on the way (the sum over
    dims, the scale, the maximum, the exponential); weights below 2^-27 also carry an error up to 2^-51,
    2^-16 of 2^-35."""
    import _gpu
    print(f"[case] small weights gap={gap} Hq={Hq} Hkv={Hkv}", flush=True)
    bt = _peaked(Hq, Hkv, gap, seed=74)
    nc, ct = 1, 528
    ro, rl = oracle.partials(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, nc, ct, 0)
    po, pl = _gpu.run_partials(_gpu.DeviceBatch(bt), nc, ct)
    check_lse(pl, rl, tag="partial lse")
    weight = np.exp(-gap)
    assert 0.1 * weight < np.abs(ro[..., :64]).max() < 600 * weight   # what the dims hold
    bound = 4 * 2.0 ** -24 * 1.45 * (gap + 1) + (2.0 ** -51 / weight if weight < 2.0 ** -27 else 0)
    err = np.linalg.norm(po[..., :64] - ro[..., :64]) / np.linalg.norm(ro[..., :64])
    print(f"    error {err:.2e}, bound {bound:.2e}", flush=True)
    assert err <= bound
    assert np.linalg.norm(po - ro) <= 4 * 2.0 ** -24 * np.sqrt(ct) * np.linalg.norm(ro)


@pytest.mark.parametrize("gap", [0, 12, 24])
@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (32, 8), (64, 8), (24, 3)], ids=["G1", "G2", "G4", "G8", "odd"])
def test_infinite_values_at_small_weights(Hq, Hkv, gap):
    """An infinite V is infinite whatever its key's weight (2^-35 and less of the largest here), on every
    path; the other dims are as they were."""
    import _gpu
    print(f"[case] infinite V gap={gap} Hq={Hq} Hkv={Hkv}", flush=True)
    bt = _peaked(Hq, Hkv, gap, seed=75)
    ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, threads=8)
    for b in range(bt.B):
        page = int(bt.indices[int(bt.indptr[b])])
        bt.v[page, 2, :, 17] = np.float16(np.inf)
        bt.v[page, 3, :, 90] = np.float16(-np.inf)
    db = _gpu.DeviceBatch(bt)
    keep = [d for d in range(128) if d not in (17, 90)]
    runs = {"plan": lambda: _gpu.run_plan(db)[:2], "uniform": lambda: _gpu.run_uniform(db, 3)[:2],
            "device ranges": lambda: _gpu.run_balanced(db)}
    for tag, f in runs.items():
        o, l = f()
        assert np.all(o[..., 17] == np.inf) and np.all(o[..., 90] == -np.inf), tag
        check_out(o[..., keep], ro[..., keep], tag=tag)
        check_lse(l, rl, tag=tag)


@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (64, 8)], ids=["G4", "G8"])
def test_infinite_values_in_a_cascade_suffix(Hq, Hkv):
    import _gpu
    print(f"[case] infinite V in a suffix Hq={Hq} Hkv={Hkv}", flush=True)
    bt = inputs.make_shared_prefix_batch(256, [5, 40, 17], Hq, Hkv, seed=76)
    ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, threads=8)
    for b in range(bt.B):
        page = int(bt.indices[int(bt.indptr[b]) + 16])
        bt.v[page, 2, :, 17] = np.float16(np.inf)
        bt.v[page, 3, :, 90] = np.float16(-np.inf)
    o, l, info = _gpu.run_cascade(_gpu.DeviceBatch(bt), min_prefix=16)
    assert info.use == 1
    keep = [d for d in range(128) if d not in (17, 90)]
    assert np.all(o[..., 17] == np.inf) and np.all(o[..., 90] == -np.inf)
    check_out(o[..., keep], ro[..., keep], tag="other dims")
    check_lse(l, rl, tag="cascade")


@pytest.mark.parametrize("scale", [0.0, -0.3, -1e-3])
@pytest.mark.parametrize("Hq,Hkv", [(32, 8), (64, 8)], ids=["G4", "G8"])
def test_scale_signs(Hq, Hkv, scale):
    """The running maximum is taken over the unscaled scores, q carrying a negative scale's sign; a scale
    of 0 weighs all keys alike; edge blocks and padding pages with poison in them."""
    import torch
    import _gpu
    import pdattn
    print(f"[case] scale {scale} Hq={Hq} Hkv={Hkv}", flush=True)
    bt = inputs.make_batch([1, 33, 0, 300, 77], Hq, Hkv, seed=77)
    ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, sm_scale=scale, threads=8)
    _poison(bt)
    db = _gpu.DeviceBatch(bt)
    plan = pdattn.Plan(bt.indptr, bt.last, bt.B, Hq, Hkv)
    ws = torch.empty(max(plan.workspace_bytes, 256), dtype=torch.uint8, device="cuda:0")
    plan.upload(ws, ws.numel())
    plan.run(db.q, db.k, db.v, db.indptr, db.indices, db.last, db.out, db.lse, ws, ws.numel(), sm_scale=scale)
    o, l = db.results()
    plan.close()
    check_out(o, ro, tag=f"scale {scale}")
    check_lse(l, rl, tag=f"scale {scale}")


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (32, 8), (64, 8)], ids=["G1", "G4", "G8"])
def test_huge_scores(Hq, Hkv):
    """Scores up to 10^10: one key has all the weight, and the lse is its score (no exponent is formed from
    a rounded product, which at this size would be off by thousands)."""
    import _gpu
    print(f"[case] huge scores Hq={Hq} Hkv={Hkv}", flush=True)
    bt = inputs.make_batch([17, 3, 40], Hq, Hkv, seed=78)
    bt.q *= np.float16(8192)
    bt.k *= np.float16(8192)
    assert np.isfinite(bt.q).all() and np.isfinite(bt.k).all()
    ro, rl = oracle.decode(bt.q, bt.k, bt.v, bt.indptr, bt.indices, bt.last, Hq, Hkv, threads=8)
    db = _gpu.DeviceBatch(bt)
    for tag, (o, l) in (("plan", _gpu.run_plan(db)[:2]), ("uniform", _gpu.run_uniform(db, 2)[:2]),
                        ("device ranges", _gpu.run_balanced(db))):
        check_out(o, ro, tag=tag)
        check_lse(l, rl, tag=tag)
