"""The large router path's wave tiles at their edges (row counts around the rules' lines, experts and K that fill no tile):
logits, selection and weights bit-exact against the oracle's fixed order."""
import numpy as np
import pytest
import torch

import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,E,K,adv", [
    (17, 256, 6144, False), (32, 250, 6144, True), (33, 9, 6144, False), (96, 256, 6144, False), (97, 130, 6144, True),
    (320, 256, 6144, False), (321, 33, 6144, False), (768, 256, 6144, False), (769, 256, 6144, False),
    (50, 256, 256, True), (200, 70, 512, False), (400, 256, 1280, False),
    (128, 256, 512, True), (129, 256, 512, False), (256, 256, 512, False), (257, 250, 512, True), (512, 64, 512, False),
    (513, 64, 512, True), (500, 128, 512, False), (1536, 256, 512, False), (1537, 256, 512, True), (1536, 129, 512, False)])
def test_router_tiles(R, E, K, adv):
    from hecate_amd import router
    from test_gpu_parity import _adversarial, u16
    dev = torch.device("cuda:0")
    rng = np.random.default_rng(R + E + K)
    if adv:
        x, wg = _adversarial(rng, (R, K), False), _adversarial(rng, (E, K), True)
    else:
        x = (rng.standard_normal((R, K)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
        wg = (rng.standard_normal((E, K)) * 0.02).astype(np.float32)
    bias = (rng.standard_normal(E) * 0.001).astype(np.float32)
    lg_ref = np.asarray(O.router_logits(x, wg), np.float32)
    sel_ref, rw_ref = O.router_select(lg_ref, bias)
    xt = torch.from_numpy(x.view(np.int16)).to(dev).view(torch.bfloat16)
    logits, ctr = router.buffers(R, dev)
    sel = torch.empty((R, 8), dtype=torch.int64, device=dev)
    rw = torch.empty((R, 8), dtype=torch.float16, device=dev)
    xh = torch.empty((R, K), dtype=torch.float16, device=dev)
    router.router_fused(xt, torch.from_numpy(wg).to(dev), torch.from_numpy(bias).to(dev), logits, ctr, sel, rw, 8, 2.5, xh)
    torch.cuda.synchronize()
    seg = logits[:8 * R * 256].view(8, R, 256).cpu().numpy()[:, :, :E]
    tot = np.zeros((R, E), np.float32)
    for s in range(8):
        tot = (tot + seg[s]).astype(np.float32)
    assert np.array_equal(tot.view(np.uint32), lg_ref.view(np.uint32))
    assert np.array_equal(sel.cpu().numpy(), sel_ref)
    assert np.array_equal(u16(rw), rw_ref)
    assert torch.equal(xh, xt.half())
