"""The log-sum-exp merge at the source counts where its kernels change (8, 16, 24, 32 sources in one
round trip, 64 per trip beyond), for few rows (one wave per workgroup) and many, against the fp64
merge: random partial states, some of them empty (lse = -inf, any bits in their rows), a row with
none. out is fp16 of an fp32 sum of n terms: half an ulp of values below 4 is 1e-3."""
import numpy as np
import pytest

from _checks import check_lse, check_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 64, 65])
@pytest.mark.parametrize("n", [1, 2, 8, 9, 16, 17, 24, 25, 32, 33, 64, 65, 200])
def test_merge_states(rows, n):
    import torch
    import pdattn
    print(f"[case] merge rows={rows} sources={n}", flush=True)
    rng = np.random.default_rng(1000 * rows + n)
    o = rng.standard_normal((rows, n, 128)).astype(np.float32)
    lse = (3.0 * rng.standard_normal((rows, n))).astype(np.float32)
    empty = rng.random((rows, n)) < 0.2
    empty[-1] = True
    lse[empty] = -np.inf
    ref_o, ref_l = np.zeros((rows, 128)), np.full(rows, -np.inf)
    for r in range(rows):
        keep = ~empty[r]
        if keep.any():
            m = lse[r][keep].max()
            w = np.exp(lse[r][keep].astype(np.float64) - m)
            ref_o[r] = (w[:, None] * o[r][keep].astype(np.float64)).sum(0) / w.sum()
            ref_l[r] = m + np.log(w.sum())
    o[empty] = np.nan
    d = torch.device("cuda:0")
    out = torch.full((rows, 128), 7.0, dtype=torch.float16, device=d)
    got = torch.full((rows,), 7.0, dtype=torch.float32, device=d)
    pdattn.merge_states(torch.from_numpy(o).to(d), torch.from_numpy(lse).to(d), out, got, rows, n)
    torch.cuda.synchronize()
    check_out(out.float().cpu().numpy(), ref_o, tag=f"{rows} rows, {n} sources")
    check_lse(got.cpu().numpy(), ref_l, tag=f"{rows} rows, {n} sources")
