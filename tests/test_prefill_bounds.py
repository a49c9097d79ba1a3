"""The sizes a prefill chunk hands to its operators: the chunk's own, whatever chunk the layer's buffers were made for (the
operators choose their kernels by them)."""
import pytest
import torch

from hecate_amd import moe4p, moe4t, tier


def _layer(E=16, n=2):
    return tier.MoELayer(torch.zeros(E, 6144), torch.zeros(E), tier.ExpertBank(n, "cpu"), max_rows=16)


@pytest.mark.parametrize("long,first,then", [(False, 300, 17), (False, 40, 40), (True, 300, 21)])
def test_prefill_bounds(monkeypatch, long, first, then):
    monkeypatch.setattr(tier, "LONG_ROWS", 16 if long else 2048)
    lay, calls = _layer(), []
    for mod in (moe4p, moe4t):
        monkeypatch.setattr(mod, "forward", lambda *a, **k: calls.append(k))
    for T in (first, then):
        pf = lay._prefill_buffers(T)
        assert pf.T == first and pf.long == long
        lay.prefill_experts(pf.xh[:T], pf.y[:T])
        bm = 256 if long else 128
        assert calls[-1]["npos"] == T * 8 and calls[-1]["nrb"] == 2 + T * 8 // bm
        assert calls[-1]["inv"].numel() == T * 8
    assert len(calls) == 2


@pytest.mark.parametrize("form", ["short", "ordered", "ordered, no shared expert", "atomic"])
def test_prefill_fp32_buffers(monkeypatch, form):
    """a layer's prefill holds at most one fp32 [T, H] buffer, and none where no form of it needs one"""
    monkeypatch.setattr(tier, "LONG_ROWS", 2048 if form == "short" else 16)
    lay = _layer()
    lay.shared = None if "no shared" in form else (torch.zeros(2048 * 6144, dtype=torch.float16),) * 3
    lay.deterministic = form != "atomic"
    for mod, name in ((moe4p, "forward"), (moe4t, "forward"), (moe4t, "shared"), (tier.router, "router_fused"),
                      (tier.moe4, "finish_bf16"), (tier, "on_device"), (tier.PrefillBuffers, "run")):
        monkeypatch.setattr(mod, name, lambda *a, **k: None)
    lay.prefill(torch.zeros(40, 6144, dtype=torch.bfloat16))
    big = [k for k, v in vars(lay._pf).items() if torch.is_tensor(v) and v.dtype == torch.float32 and v.shape == (40, 6144)]
    assert len(big) == (0 if form in ("short", "ordered, no shared expert") else 1), big


@pytest.mark.gpu
def test_atomic_prefill_first_used_in_a_capture(dev):
    """the accumulator of the atomic form first asked for inside a capture belongs to the graph: an eager chunk before any
    replay, and every replay, still start from zeros"""
    from hecate_amd import synth
    lay = synth.make_layer(0, dev, resident=[3, 7], max_rows=16)
    x = synth.gen_x(32, 2100, dev)
    ref = lay.prefill(x).float()                                # ordered: no accumulator yet
    lay.deterministic = False
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = lay.prefill(x)
    tol = 2 ** -7 * ref.abs().max()                             # (one bf16 ulp of the largest: the adds' order is free)
    assert (lay.prefill(x).float() - ref).abs().max() <= tol
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert (out.float() - ref).abs().max() <= tol
        assert (lay.prefill(x).float() - ref).abs().max() <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("first,then", [(300, 17), (300, 40), (2300, 2100)])
def test_prefill_after_a_larger_chunk(dev, first, then):
    """a chunk after a larger one on the same layer: the bits of the same chunk on fresh buffers"""
    from hecate_amd import synth
    lay = synth.make_layer(0, dev, resident=[3, 7], max_rows=16)
    x = synth.gen_x(31, first, dev)
    fresh = lay.prefill(x[:then]).clone()
    lay._pf = None
    lay.prefill(x)
    assert lay._pf.T == first
    after = lay.prefill(x[:then])
    assert lay._pf.T == first and bool(fresh.any())
    assert torch.equal(after.view(torch.int16), fresh.view(torch.int16))
