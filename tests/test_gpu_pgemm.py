"""The grouped expert GEMM at every pick-tile count and its edges: one expert with n picks (and a neighbour with 3), through
the device dispatch and moe4p.forward, against a torch fp32 reference on the same dequantised weights."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NS = (1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 144, 200, 256, 257)


@pytest.fixture(scope="module")
def lay():
    from hecate_amd import synth
    return synth.make_layer(0, torch.device("cuda:0"), resident=[3, 7], shared=False)


@pytest.mark.parametrize("ordered", (True, False))
@pytest.mark.parametrize("bm", (128, 256))
@pytest.mark.parametrize("n", NS)
def test_pick_counts(lay, n, bm, ordered):
    from hecate_amd import moe4p, synth, tier
    from torchref import moe_rows
    dev = lay.device
    T = n + 3
    x = synth.gen_x(50 + n, T, dev)
    sel = torch.zeros((T, 1), dtype=torch.int64, device=dev)
    sel[torch.arange(3, device=dev) * (T // 3)] = 1                       # the neighbour's picks, among the others
    rw = (0.25 + 0.5 * torch.rand((T, 1), generator=torch.Generator().manual_seed(n))).half().to(dev)
    pf = tier.PrefillBuffers(T, 1, 0, 2, 256, dev, bm=bm).run(sel, rw)
    y = torch.zeros((T, 6144), dtype=torch.float32, device=dev)
    gq, uq, dq, gs, us, ds = lay.bank.tables()
    moe4p.forward(x, pf.tok, pf.eid, pf.wt, pf.rbt, gq, uq, dq, gs, us, ds, *pf.scr, y,
                  inv=pf.inv if ordered else None, meta=pf.meta, topk=1, npos=T, nrb=pf.nrb_max)
    ref = moe_rows(lay, x, sel, rw, with_shared=False)
    # the act rows are rounded to f16: each of the 2048 terms of an output carries an independent error of at most 2^-11 of
    # it, so the output's error has a standard deviation of at most 2^-11 of the row's rms (the act row is heavy-tailed: a
    # few terms make most of it, so the bound of one rounding is taken, not its average); five of those for the largest of
    # ~10^6 outputs, and, ordered, the down row is rounded once more
    bound = 5 * 2.0 ** -11 * ref.square().mean(1, keepdim=True).sqrt() + (2.0 ** -11) * ref.abs()
    worst = ((y - ref).abs() / bound).max().item()
    assert worst <= 1.0, (n, bm, ordered, worst)
