"""The grouped expert GEMMs at every pick-tile count and their edges: one expert with n picks (and a neighbour with 3), through
the device dispatch and moe4p.forward or, on either side of its rule, moe4t.forward, against a torch fp32 reference on the
same dequantised weights; and the shared expert in the same launches at the edges of its token blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NS = (1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 144, 200, 256, 257)


@pytest.fixture(scope="module")
def lay():
    from hecate_amd import synth
    return synth.make_layer(0, torch.device("cuda:0"), resident=[3, 7])


def bound(ref):
    # the act rows are rounded to f16: each of the 2048 terms of an output carries an independent error of at most 2^-11 of
    # it, so the output's error has a standard deviation of at most 2^-11 of the row's rms (the act row is heavy-tailed: a
    # few terms make most of it, so the bound of one rounding is taken, not its average); five of those for the largest of
    # ~10^6 outputs, and, ordered, the down row is rounded once more
    return 5 * 2.0 ** -11 * ref.square().mean(1, keepdim=True).sqrt() + (2.0 ** -11) * ref.abs()


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
    worst = ((y - ref).abs() / bound(ref)).max().item()
    assert worst <= 1.0, (n, bm, ordered, worst)


@pytest.mark.parametrize("T", (1, 16, 17, 32, 33, 64, 65, 96, 97, 128, 129, 130, 256, 257, 300))
def test_shared_blocks(lay, T):
    from hecate_amd import moe4p, synth, tier
    from torchref import moe_rows
    dev = lay.device
    x = synth.gen_x(400 + T, T, dev)
    sel = torch.full((T, 1), 2, dtype=torch.int64, device=dev)            # outside the window, but for a few tokens
    sel[::5] = 0
    rw = torch.full((T, 1), 0.5, dtype=torch.float16, device=dev)
    pf = tier.PrefillBuffers(T, 1, 0, 2, 256, dev).run(sel, rw)
    out = torch.empty((T, 6144), dtype=torch.bfloat16, device=dev)
    y = torch.zeros((T, 6144), dtype=torch.float32, device=dev)
    gq, uq, dq, gs, us, ds = lay.bank.tables()
    a = (x, pf.tok, pf.eid, pf.wt, pf.rbt, gq, uq, dq, gs, us, ds, *pf.scr)
    kw = dict(inv=pf.inv, meta=pf.meta, topk=1, npos=T, nrb=pf.nrb_max, shared=lay.shared_rows())
    moe4p.forward(*a, y, **kw)
    moe4p.forward(*a, None, out_bf16=out, **kw)
    routed = moe_rows(lay, x, sel, rw, with_shared=False)
    ref = moe_rows(lay, x, sel, rw)
    worst = ((y - ref).abs() / (bound(ref - routed) + bound(routed).clamp_min(1e-30))).max().item()
    assert worst <= 1.0, (T, worst)
    assert torch.equal(out.view(torch.int16), y.bfloat16().view(torch.int16))


@pytest.mark.parametrize("n", NS)
def test_wide_tables(lay, n):
    """the down launch with three column blocks a workgroup (tables of 128 experts, 200 picks or more of room; from 257 tokens
    and 192 experts the shared expert's blocks too) against the one of few experts: the same sums in the same order, so the
    same bits, the shared expert's rows among them"""
    from hecate_amd import moe4p, synth, tier
    dev = lay.device
    T = n + 3
    x = synth.gen_x(800 + n, T, dev)
    sel = torch.zeros((T, 1), dtype=torch.int64, device=dev)
    sel[torch.arange(3, device=dev) * (T // 3)] = 1
    rw = torch.full((T, 1), 0.5, dtype=torch.float16, device=dev)
    for shared in (None, lay.shared_rows()):
        ys = []
        for room, experts in ((T, 2), (max(T, 200), 128), (max(T, 200), 192)):
            pf = tier.PrefillBuffers(room, 1, 0, experts, 256, dev).run(sel, rw)
            y = torch.zeros((T, 6144), dtype=torch.float32, device=dev)
            moe4p.forward(x, pf.tok, pf.eid, pf.wt, pf.rbt, *[t.repeat(experts // 2) for t in lay.bank.tables()], *pf.scr, y,
                          inv=pf.inv[:T], meta=pf.meta, topk=1, npos=pf.F, nrb=pf.nrb_max, shared=shared)
            ys.append(y)
        for y in ys[1:]:
            assert bool(y.any()) and torch.equal(ys[0].view(torch.int32), y.view(torch.int32)), (n, shared is None)


def test_shared_apart(lay):
    """past 3584 tokens the shared expert runs in launches of its own: its rows of the first 3584 tokens against the ones of
    the grouped launches, the same sums in the same order, so the same bits"""
    from hecate_amd import moe4p, synth, tier
    dev = lay.device
    x = synth.gen_x(61, 3587, dev)
    sel = torch.full((3587, 1), 2, dtype=torch.int64, device=dev)         # outside the window, but for a few tokens
    sel[::9] = 0
    rw = torch.full((3587, 1), 0.5, dtype=torch.float16, device=dev)
    ys = []
    for T in (3584, 3587):
        pf = tier.PrefillBuffers(T, 1, 0, 2, 256, dev).run(sel[:T], rw[:T])
        y = torch.zeros((T, 6144), dtype=torch.float32, device=dev)
        moe4p.forward(x[:T], pf.tok, pf.eid, pf.wt, pf.rbt, *lay.bank.tables(), *pf.scr, y, inv=pf.inv, meta=pf.meta, topk=1,
                      npos=T, nrb=pf.nrb_max, shared=lay.shared_rows())
        ys.append(y)
    assert bool(ys[1].abs().amax(1).all()) and torch.equal(ys[0].view(torch.int32), ys[1][:3584].view(torch.int32))


@pytest.mark.parametrize("ordered", (True, False))
@pytest.mark.parametrize("room", (264, 265))
@pytest.mark.parametrize("n", NS[:-2] + (239, 240, 241, 255, 256))
def test_moe4t_pick_counts(lay, n, room, ordered):
    """moe4t.forward on both of its kernels: 132 picks an expert is the last bound on the picks (264 for 2 experts) that
    takes the tile-count GEMM, and one more takes the one of 16 tiles a pass, which cuts no block of up to 256"""
    from hecate_amd import moe4t, synth, tier
    from torchref import moe_rows
    dev = lay.device
    T = n + 3
    x = synth.gen_x(500 + n, T, dev)
    sel = torch.zeros((T, 1), dtype=torch.int64, device=dev)
    sel[torch.arange(3, device=dev) * (T // 3)] = 1
    rw = (0.25 + 0.5 * torch.rand((T, 1), generator=torch.Generator().manual_seed(n))).half().to(dev)
    pf = tier.PrefillBuffers(room, 1, 0, 2, 256, dev, bm=256, long=True).run(sel, rw)
    y = torch.zeros((T, 6144), dtype=torch.float32, device=dev)
    moe4t.forward(x, pf.tok, pf.eid, pf.wt, pf.rbt, *lay.bank.tables(), *pf.scr, y, meta=pf.meta, npos=room, nrb=pf.nrb_max,
                  inv=pf.inv[:T] if ordered else None, topk=1)
    assert int(pf.meta[1].item()) == 2
    ref = moe_rows(lay, x, sel, rw, with_shared=False)
    worst = ((y - ref).abs() / bound(ref)).max().item()
    assert worst <= 1.0, (n, room, ordered, worst)


@pytest.mark.parametrize("ordered", (True, False))
def test_moe4t_skewed_blocks(lay, ordered):
    """the 16-tile GEMM on an uneven plan: one expert cut into blocks of 205, one of 40 picks, tokens with both, one or none"""
    from hecate_amd import moe4t, synth, tier
    from torchref import moe_rows
    dev = lay.device
    T = 900
    x = synth.gen_x(77, T, dev)
    sel = torch.full((T, 2), 9, dtype=torch.int64, device=dev)             # outside the window
    sel[:820, 0] = 0                                                      # 820 picks: 4 blocks of 205
    sel[800:840, 1] = 1
    rw = (0.25 + 0.5 * torch.rand((T, 2), generator=torch.Generator().manual_seed(4))).half().to(dev)
    pf = tier.PrefillBuffers(T, 2, 0, 2, 256, dev, bm=256, long=True).run(sel, rw)
    assert pf.rbt[:int(pf.meta[1].item()), 2].tolist() == [205] * 4 + [40]
    y = torch.zeros((T, 6144), dtype=torch.float32, device=dev)
    moe4t.forward(x, pf.tok, pf.eid, pf.wt, pf.rbt, *lay.bank.tables(), *pf.scr, y, meta=pf.meta, npos=pf.F, nrb=pf.nrb_max,
                  inv=pf.inv if ordered else None, topk=2)
    parts = [moe_rows(lay, x, sel[:, k:k + 1], rw[:, k:k + 1], with_shared=False) for k in range(2)]
    ref, lim = parts[0] + parts[1], bound(parts[0]) + bound(parts[1])      # (each pick's row has its own roundings)
    none = ref.abs().amax(1) == 0
    assert int(none.sum()) == 60 and not bool(y[none].any())
    worst = ((y - ref).abs()[~none] / lim[~none]).max().item()
    assert worst <= 1.0, worst
