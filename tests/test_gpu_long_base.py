"""The long prefill's combine over a partial that is only read (moe4t.forward with base in out's place) and the shared
expert's rows written instead of added: bit for bit the forms that add into a zeroed fp32 partial and re-zero it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
H = 6144


@pytest.fixture(scope="module")
def lay():
    from hecate_amd import synth
    return synth.make_layer(0, torch.device("cuda:0"), resident=[3, 7])


@pytest.mark.parametrize("picks", (True, False))
@pytest.mark.parametrize("T", (1, 127, 129, 700))
def test_base_rows(lay, T, picks):
    from hecate_amd import _lib, moe4t, synth, tier
    dev = lay.device
    x = synth.gen_x(900 + T, T, dev).half()
    sel = torch.full((T, 2), 2, dtype=torch.int64, device=dev)           # outside the window
    if picks:
        sel[:, 0] = torch.arange(T, device=dev) % 3                      # experts 0 and 1, and every third token neither
    rw = torch.full((T, 2), 0.5, dtype=torch.float16, device=dev)
    pf = tier.PrefillBuffers(T, 2, 0, 2, 256, dev, bm=256, long=True).run(sel, rw)
    gq, uq, dq, gs, us, ds = lay.bank.tables()
    a = (x, pf.tok, pf.eid, pf.wt, pf.rbt, gq, uq, dq, gs, us, ds, *pf.scr)
    kw = dict(meta=pf.meta, npos=pf.F, nrb=pf.nrb_max, inv=pf.inv, topk=2)
    y = torch.zeros((T, H), device=dev)
    moe4t.shared(x, *lay.shared_rows(), pf.shw, y)
    sh = torch.full((T, H), float("nan"), device=dev)
    moe4t.shared(x, *lay.shared_rows(), pf.shw, sh, add=False)
    assert torch.equal(sh, y)
    o = [torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(4)]
    moe4t.forward(*a, None, out_bf16=o[0], base=sh, **kw)
    assert torch.equal(sh, y)                                            # the base is read only
    moe4t.forward(*a, y, out_bf16=o[1], **kw)
    moe4t.forward(*a, None, out_bf16=o[2], **kw)                         # no base
    moe4t.forward(*a, y, out_bf16=o[3], **kw)                            # (y zeroed by the call before)
    assert torch.equal(o[0].view(torch.int16), o[1].view(torch.int16))
    assert torch.equal(o[2].view(torch.int16), o[3].view(torch.int16))
    kw["npos"] = 0                                                       # no pick: the base alone
    moe4t.forward(*a, None, out_bf16=o[0], base=sh, **kw)
    assert torch.equal(o[0], sh.bfloat16())
    with pytest.raises(RuntimeError):
        moe4t.forward(*a, y, out_bf16=o[0], base=sh, **kw)
    with pytest.raises(RuntimeError):
        moe4t.forward(*a, None, **kw)
    assert _lib.lib().hmoe_moe4t_forward_base_bf16(*([None] * 5), 0, 0, 0, *([None] * 10), 0, None, 1, 0, None, 8, None,
                                                   None) != 0


@pytest.mark.parametrize("npos", (260, 600))
def test_many_row_blocks(lay, npos):
    """a plan's room for row blocks far past the plan (600,000, as blocks of one pick would need; the device's count says
    how many there are), on either grouped GEMM: the bits of the same call with the plan's own room"""
    from hecate_amd import moe4t, synth, tier
    dev = lay.device
    T = 130
    x = synth.gen_x(70, T, dev).half()
    sel = (torch.arange(2 * T, device=dev) % 3).view(T, 2)
    rw = torch.full((T, 2), 0.5, dtype=torch.float16, device=dev)
    pf = tier.PrefillBuffers(300, 2, 0, 2, 256, dev, bm=256, long=True).run(sel, rw)
    rbt = torch.zeros((600000, 4), dtype=torch.int32, device=dev)
    rbt[:pf.nrb_max] = pf.rbt
    ys = []
    for plan in (pf.rbt, rbt):
        y = torch.zeros((T, H), device=dev)
        moe4t.forward(x, pf.tok, pf.eid, pf.wt, plan, *lay.bank.tables(), *pf.scr, y, meta=pf.meta, npos=npos,
                      inv=pf.inv[:2 * T], topk=2)
        ys.append(y)
    assert bool(ys[0].any()) and torch.equal(ys[0], ys[1])


def test_base_without_picks(lay):
    """no pick reaches the tier: the base alone (or zeros), whatever the scratch's room, with neither tables nor act rows"""
    from hecate_amd import _lib
    dev = lay.device
    T = 33
    base = torch.randn((T, H), generator=torch.Generator().manual_seed(5)).to(dev)
    d = torch.full((1, H), float("nan"), dtype=torch.float16, device=dev)
    inv = torch.full((T * 8,), -1, dtype=torch.int32, device=dev)
    out = torch.empty((T, H), dtype=torch.bfloat16, device=dev)
    for b in (base, None):
        out.fill_(7)
        _lib.call("hmoe_moe4t_forward_base_bf16", *([None] * 5), 0, 0, 0, *([None] * 8), d.data_ptr(), _lib.ptr(b), 1, None, T,
                  _lib.XF_BF16, inv.data_ptr(), 8, out.data_ptr(), _lib.stream_of(dev))
        assert torch.equal(out, torch.zeros_like(out) if b is None else b.bfloat16())
