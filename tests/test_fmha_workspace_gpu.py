"""FMHA split workspaces.  Up to 2560 query tokens one buffer that any call sized
serves all; from 2561 on a call needs nothing from earlier ones: no shared buffer
that a capture could not grow or that two streams would share."""
import pytest
import torch

ONE_SIZE = 66 * 3 * 2 * 256 * 258 * 4   # 66 tiles of 256 rows, 3 chunks, 2 KV heads


def test_one_size_up_to_2560_tokens():
    from qwen36_attn import _lib
    size = _lib.load(("qwen36_fmha_prefill_workspace_bytes",)).qwen36_fmha_prefill_workspace_bytes
    for t in [*range(1, 2561, 7), 360, 361, 672, 960, 961, 1344, 2048, 2111, 2112, 2113, 2560]:
        for prefix in (0, 1, 255, 256, 300, 1000, 4000, 24000, 65000):
            if t + prefix > 32:
                assert size(t, t + prefix) == ONE_SIZE
            else:                           # one chunk: tiles of 4 tokens
                assert size(t, t + prefix) == (t + 3) // 4 * 2 * 32 * 258 * 4
    for t, s in ((2561, 2561), (4096, 4096), (3072, 9000)):
        assert size(t, s) >= ONE_SIZE
    assert size(4097, 4097) == size(3073, 9000) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [64, 512, 2560])
def test_capture_after_a_call_of_another_geometry(gpu, warm, monkeypatch):
    from qwen36_attn import _tensors
    from qwen36_attn.full_attention import fmha_prefill_gated
    monkeypatch.setattr(_tensors, "_SCRATCH", {})
    fmha_prefill_gated(*_inputs(warm, warm, gpu, warm))
    torch.cuda.synchronize()
    for t, s in ((93, 24093), (2112, 2112), (2560, 4000)):
        print(f"capture T={t} S={s} after T={warm}", flush=True)
        args = _inputs(t, s, gpu, t + s)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = fmha_prefill_gated(*args)
        want = fmha_prefill_gated(*args)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)


def _inputs(t, s, gpu, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v, gate = (torch.randn(*shape, generator=g).to(torch.bfloat16).to(gpu)
                     for shape in ((t, 16, 256), (s, 2, 256), (s, 2, 256), (t, 8192)))
    return q, k, v, gate


@pytest.mark.gpu
@pytest.mark.parametrize("t,s", [(1, 32), (32, 32), (2561, 2561), (4096, 4096), (3072, 3400)])
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


@pytest.mark.gpu
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
