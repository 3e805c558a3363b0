"""The native form of the transformers attention call (the binding's hf()) against the Python route of
mi355_decode_attention, bit for bit over the layouts both take, and its refusals: every call it declines goes the Python
way, with the same result or error."""
import types

import pytest
import torch

from breeze_tts_2_flash_amd import gqa_decode_masked, hf_attention, kernels

pytestmark = pytest.mark.gpu

MODULE = types.SimpleNamespace(training=False)


def case(device, B=2, NH=16, NKV=8, D=128, S=300, q_len=1, dtype=torch.bfloat16, mask_dtype=torch.bfloat16, rows=None, extra=0):
    g = torch.Generator().manual_seed(B * S + NH)
    q = torch.randn(B, NH, q_len, D, generator=g).to(device, dtype)
    k, v = (torch.randn(B, NKV, S, D, generator=g).to(device, dtype) for _ in range(2))
    m = torch.zeros(rows or B, 1, q_len, S + extra, dtype=mask_dtype)
    m[-1, ..., :7] = torch.finfo(mask_dtype).min
    m[0, ..., 20:30] = -1.5
    return q, k, v, m.to(device)


def python_way(monkeypatch, *a, **kw):
    with monkeypatch.context() as mp:
        mp.setattr(hf_attention, "_native", None)
        return hf_attention.mi355_decode_attention(MODULE, *a, **kw)[0]


@pytest.mark.parametrize("kw", [{}, dict(D=64), dict(NH=8), dict(NH=64), dict(mask_dtype=torch.float32), dict(rows=1),
                                dict(extra=13), dict(B=1, S=1), dict(B=5, S=2049)])
@pytest.mark.parametrize("scaling", [0.07, None])
def test_native_equals_python(device, monkeypatch, kw, scaling):
    q, k, v, m = case(device, **kw)
    want = python_way(monkeypatch, q, k, v, m, scaling=scaling)
    assert hf_attention._native is None or hf_attention._native == kernels.eager().hf
    hf_attention.mi355_decode_attention(MODULE, q, k, v, m, scaling=scaling)  # binds the native form
    hits = hf_attention.calls["hip"]
    forms = [(q, k, v, m)]
    forms.append((q.transpose(1, 2).contiguous().transpose(1, 2), k, v, m))  # a projection's layout
    big = torch.zeros(k.size(0), k.size(1), k.size(2) + 40, k.size(3), dtype=k.dtype, device=device)
    kb, vb = big.clone(), big.clone()
    kb[:, :, :k.size(2)], vb[:, :, :k.size(2)] = k, v
    forms.append((q, kb[:, :, :k.size(2)], vb[:, :, :k.size(2)], m))         # a slice of a longer cache
    for f in forms:
        direct = kernels.eager().hf(*f, scaling)
        got = hf_attention.mi355_decode_attention(MODULE, *f, scaling=scaling)[0]
        torch.cuda.synchronize()
        assert direct is not None and got.shape == want.shape and got.is_contiguous()
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        assert torch.equal(direct.view(torch.int16), want.view(torch.int16))
    assert hf_attention.calls["hip"] == hits + len(forms)


def test_refusals_go_the_python_way(device, monkeypatch):
    q, k, v, m = case(device)
    hf_attention.mi355_decode_attention(MODULE, q, k, v, m)
    hf = kernels.eager().hf
    assert hf(q, k, v, m, None) is not None
    odd = [case(device, q_len=2), case(device, dtype=torch.float16), case(device, NH=24), case(device, D=32),
           (q, k, v.transpose(1, 2).contiguous().transpose(1, 2), m), (q, k, v, m.to(torch.float16)),
           (q, k, v, m[..., :200]), (q, k, v, m.expand(-1, -1, 3, -1)), tuple(t.cpu() for t in (q, k, v, m)),
           (q, k, v, None), (q, k, v, m[:, 0])]
    for f in odd:
        assert hf(*f, 0.1) is None
    # a mask of several query rows: the last one's, as before
    rows = m.expand(-1, -1, 3, -1).contiguous()
    rows[:, :, :2] = -1.0
    got = hf_attention.mi355_decode_attention(MODULE, q, k, v, rows)[0]
    want = gqa_decode_masked(q, k, v, m, 128 ** -0.5)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16).flatten(), want.view(torch.int16).flatten())
    # dropout in training, and shapes the kernel has no form for: eager attention
    before = hf_attention.calls["eager"]
    hf_attention.mi355_decode_attention(types.SimpleNamespace(training=True), q, k, v, m, dropout=0.5)
    hf_attention.mi355_decode_attention(MODULE, *case(device, NH=24))
    assert hf_attention.calls["eager"] == before + 2
    bad = m.expand(-1, 2, -1, -1)
    with pytest.raises(RuntimeError, match="mask must be"):
        hf_attention.mi355_decode_attention(MODULE, q, k, v, bad)


def test_new_stream_and_capture(device):
    q, k, v, m = case(device)
    want = hf_attention.mi355_decode_attention(MODULE, q, k, v, m)[0].clone()
    side = torch.cuda.Stream(device)
    side.wait_stream(torch.cuda.current_stream(device))
    with torch.cuda.stream(side):
        outs = [hf_attention.mi355_decode_attention(MODULE, q, k, v, m)[0] for _ in range(2)]
    torch.cuda.current_stream(device).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = hf_attention.mi355_decode_attention(MODULE, q, k, v, m)[0]
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured.view(torch.int16), want.view(torch.int16))
    for o in outs:
        assert torch.equal(o.view(torch.int16), want.view(torch.int16))
