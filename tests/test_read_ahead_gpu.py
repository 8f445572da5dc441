"""The attention decode step told what the next launch streams: the workgroups that read it
ahead change nothing, whatever its size (a ragged last piece, one 16-byte row,
more pieces than workgroups), with one split workgroup per KV head, with the most
(128 beside 128 readers, 4096 rows) and where nothing is read ahead any more (4097
rows), and the hint never refuses a call."""
import pytest
import torch

from qwen36_attn import synthetic as syn

BF16 = torch.bfloat16
ELEMENTS = [8, 32768 + 24, 2048 * 4096, 16 << 20]


def test_read_ahead_hint_is_optional():
    from qwen36_attn._tensors import read_ahead
    dev = torch.device("cpu")
    x = torch.zeros(64, 8, dtype=BF16)
    assert read_ahead(x, dev) == (x.data_ptr(), 1024)
    for t in (None, x.t(), x[:0], x.view(-1)[4:], "o_proj", x.to("meta"),
              torch.empty((16 << 20) + 8, dtype=BF16)):
        assert read_ahead(t, dev) == (None, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("elements", ELEMENTS)
@pytest.mark.parametrize("rows,split", [(1, 0), (97, 0), (2051, 0), (2051, 1024), (4096, 0), (4096, 128),
                                        (4097, 0), (8193, 0)])
def test_attention_step_with_next_weight(gpu, rows, split, elements):
    from qwen36_attn.full_attention import decode_step
    g = syn.gen(rows)
    q, k, v = (syn.randn((1, n), g).to(gpu) for n in (8192, 512, 512))
    qw, kw = (syn.randn((256,), g, 0.1).to(gpu) for _ in range(2))
    kc, vc = (syn.randn((rows, 2, 256), g).to(gpu) for _ in range(2))
    kc2, vc2 = kc.clone(), vc.clone()
    w = syn.randn((elements,), syn.gen(1)).to(gpu)
    w0 = w.clone()
    print(f"decode step rows={rows} split={split} next={elements}", flush=True)
    got = decode_step(q, k, v, qw, kw, kc, vc, rows - 1, split_tokens=split, next_weight=w)
    want = decode_step(q, k, v, qw, kw, kc2, vc2, rows - 1, split_tokens=split)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.equal(kc, kc2) and torch.equal(vc, vc2)
    assert torch.equal(w, w0)


def test_next_weight_refusals():
    """C entries: bytes without an address, an address without bytes, more than
    the L2s hold, an address off 16 bytes."""
    from qwen36_attn import _lib
    L = _lib.load(("qwen36_decode_step_next",))
    for nxt in ((None, 16), (32, 0), (32, (32 << 20) + 1), (40, 16)):
        assert L.qwen36_decode_step_next(16, 16, 16, 16, 16, 16, 16, 0, 1, 1, 16, 16, 1 << 30, 0,
                                         *nxt, None) == 1
