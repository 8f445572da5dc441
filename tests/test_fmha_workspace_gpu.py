"""FMHA of 2561 and more query tokens needs nothing from earlier calls: no
shared buffer that a capture could not grow or that two streams would share."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(t, s, gpu, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v, gate = (torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)
                     for shape in ((t, 16, 256), (s, 2, 256), (s, 2, 256), (t, 8192)))
    return q, k, v, gate


@pytest.mark.parametrize("t,s", [(2561, 2561), (4096, 4096), (3072, 3400)])
def test_capture_without_an_eager_call(gpu, t, s, monkeypatch):
    from qwen36_attn import _lib, _tensors
    from qwen36_attn.full_attention import fmha_prefill, fmha_prefill_gated
    assert _lib.load(("qwen36_fmha_prefill",)).qwen36_fmha_prefill_workspace_bytes(t, s) > 0
    q, k, v, gate = _inputs(t, s, gpu, t + s)
    fmha_prefill_gated(*_inputs(64, 64, gpu, 1))   # set-up of another, small size
    monkeypatch.setattr(_tensors, "_SCRATCH", {})
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rows, gated = fmha_prefill(q, k, v), fmha_prefill_gated(q, k, v, gate)
    assert not _tensors._SCRATCH
    want = fmha_prefill(q, k, v), fmha_prefill_gated(q, k, v, gate)
    for _ in range(3):
        rows.zero_()
        gated.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(rows, want[0]) and torch.equal(gated, want[1])


def test_two_streams_at_once(gpu):
    from qwen36_attn.full_attention import fmha_prefill_gated
    calls = [_inputs(2700, 2700, gpu, i) for i in (1, 2)]
    want = [fmha_prefill_gated(*c) for c in calls]
    streams = [torch.cuda.Stream() for _ in calls]
    torch.cuda.synchronize()
    for _ in range(4):
        got = []
        for c, st in zip(calls, streams):
            with torch.cuda.stream(st):
                got.append(fmha_prefill_gated(*c))
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)
