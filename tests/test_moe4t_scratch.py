"""moe4t.forward's check of its scratch on the host: d holds the f16 copy of bf16 x, also where the tokens outnumber the
picks (a tier that few picks reach), so a shorter one is refused before any launch."""
import pytest
import torch

from hecate_amd import moe4t

H, I = 6144, 2048


@pytest.mark.parametrize("T,ps,dtype,d_rows,d_dtype,ok", [
    (9, 5, torch.bfloat16, 5, torch.float16, False), (9, 5, torch.bfloat16, 8, torch.float16, False),
    (9, 5, torch.bfloat16, 9, torch.float16, True), (9, 5, torch.bfloat16, 5, torch.float32, True),
    (9, 5, torch.float16, 5, torch.float16, True), (5, 9, torch.bfloat16, 9, torch.float16, True),
    (5, 9, torch.bfloat16, 8, torch.float16, False)])
def test_short_d_is_refused(monkeypatch, T, ps, dtype, d_rows, d_dtype, ok):
    calls = []
    monkeypatch.setattr(moe4t, "on_device", lambda *a: None)
    monkeypatch.setattr(moe4t, "stream_of", lambda *a: None)
    monkeypatch.setattr(moe4t, "call", lambda *a: calls.append(a[0]))
    i32 = lambda *s: torch.zeros(s, dtype=torch.int32)
    tab = torch.zeros(2, dtype=torch.int64)
    go = lambda: moe4t.forward(torch.zeros(T, H, dtype=dtype), i32(ps), i32(ps), torch.zeros(ps), i32(2, 4), *[tab] * 6, None,
                               torch.zeros(ps, I, dtype=torch.float16), torch.zeros(d_rows, H, dtype=d_dtype),
                               torch.zeros(T, H), npos=min(ps, 5), nrb=2)
    if ok:
        go()
        assert calls == ["hmoe_moe4t_forward"]
    else:
        with pytest.raises(RuntimeError, match="scratch"):
            go()
        assert not calls
