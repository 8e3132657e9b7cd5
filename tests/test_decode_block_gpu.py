"""The MFMA decode body at the sizes where it can go wrong, against the fp64 oracle: sequences around
one and two pages, around a wave's share (its 32-key blocks with one page or none of its own) and
around a workgroup's, for every group size and for one and two kv heads per workgroup, through the
plan path, the uniform split, its fp32 partials and the device-range drop-in, with NaN and Inf in
every cache slot that holds no key; infinite V values in keys that count.

The weights of the PV product are two fp16 halves (22 bits), so the fp32 partials are held to fp32's
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
