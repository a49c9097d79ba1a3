"""The one-launch dispatch plan against the oracle around its edges (rounds of 64 picks, its largest pick count and the
first one past it), with windows, absent picks, one expert for all, and top-k below 8."""
import numpy as np
import pytest
import torch

import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,topk,lo,n,bm,bal,kind", [
    (1, 8, 0, 256, 128, True, "any"), (8, 8, 0, 256, 128, True, "any"), (127, 8, 40, 100, 16, False, "any"),
    (128, 8, 0, 256, 64, True, "any"), (129, 8, 0, 176, 128, True, "any"), (200, 3, 5, 7, 256, True, "any"),
    (300, 1, 0, 2, 16, True, "one"), (512, 8, 0, 256, 128, True, "any"), (513, 8, 0, 256, 128, True, "any"),
    (512, 8, 200, 56, 1, False, "any"), (100, 8, 0, 256, 128, True, "none"), (4096, 1, 3, 1, 256, True, "one")])
def test_dispatch_one(T, topk, lo, n, bm, bal, kind):
    from hecate_amd import tier
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(T + n)
    if kind == "one":
        sel = np.full((T, topk), lo, np.int64)
    else:
        sel = np.argsort(rng.random((T, 256)), axis=1)[:, :topk].astype(np.int64) + (10000 if kind == "none" else 0)
        sel[::5, 0] = -3
    rw = O.f32_to_f16(rng.random((T, topk)).astype(np.float32))
    pf = tier.PrefillBuffers(T, topk, lo, n, 256, dev, bm=bm)
    pf.run(torch.from_numpy(sel).to(dev), torch.from_numpy(rw.view(np.int16)).to(dev).view(torch.float16), bal)
    torch.cuda.synchronize()
    counts, tok, eid, wt, inv = O.dispatch(sel, rw, lo, n)
    npos, meta = len(tok), pf.meta.cpu().numpy()
    ref = O.pick_groups(counts, bm, bal)
    assert meta[0] == npos and meta[1] == len(ref) == meta[2]
    assert np.array_equal(pf.counts.cpu().numpy(), counts.astype(np.int32))
    assert np.array_equal(pf.tok[:npos].cpu().numpy(), tok)
    assert np.array_equal(pf.eid[:npos].cpu().numpy(), eid)
    assert np.array_equal(pf.wt[:npos].cpu().numpy().view(np.uint32), wt.view(np.uint32))
    assert np.array_equal(pf.inv.cpu().numpy(), inv)
    assert np.array_equal(pf.rbt[:meta[1]].cpu().numpy().reshape(-1, 4), np.asarray(ref).reshape(-1, 4))
