"""Split sizes of short caches: edges of the block, of the split count's limit
and of the coarse rule, and workspaces."""
import pytest
import torch

from oracle.attention_bounds import Row


def test_workspace_serves_every_shorter_cache():
    from qwen36_attn import _lib
    size = _lib.load(("qwen36_decode_gqa_workspace_bytes",)).qwen36_decode_gqa_workspace_bytes
    per_split = 2 * 8 * 258 * 4
    assert {size(n, 0) for n in range(1, 8193)} == {64 * per_split}
    assert size(8193, 0) == 65 * per_split
    assert size(3000, 128) == 24 * per_split


@pytest.mark.gpu
@pytest.mark.parametrize("cache_end", [32, 33, 2048, 2049, 4097, 6144, 6145, 8192, 8193])
def test_default_split_matches_oracle(gpu, cache_end):
    from qwen36_attn import _lib
    from qwen36_attn.full_attention import decode_gqa
    g = torch.Generator().manual_seed(cache_end)
    q = torch.randn(16, 256, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(cache_end, 2, 256, generator=g).to(torch.bfloat16) for _ in range(2))
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    print(f"decode splits cache_end={cache_end}", flush=True)
    out = decode_gqa(qd, kd, vd, cache_end - 1, cache_end)
    # P enters the PV products as bf16, the output is rounded to bf16
    row = Row(q, k, v)
    bound = 2.0 ** -8 * row.ref.abs() + row.tol
    assert ((out.cpu().double().view(4096) - row.ref).abs() <= bound).all()
    if cache_end > 32:   # one block of the least split left out shows
        for block in (slice(0, 32), slice((cache_end - 1) // 32 * 32, cache_end)):
            assert ((row.without(block) - row.ref).abs() > 2 * bound).any(), block
    # a workspace with room for 128-token splits only is still accepted, and
    # gives what that split size gives
    lib = _lib.load(("qwen36_decode_gqa",))
    nb = min(64, (cache_end + 127) // 128) * 2 * 8 * 258 * 4
    if cache_end > 8192:
        return
    want = decode_gqa(qd, kd, vd, cache_end - 1, cache_end, split_tokens=128)
    ws, got = torch.empty(nb, dtype=torch.uint8, device=gpu), torch.empty_like(want)
    call = lambda n: lib.qwen36_decode_gqa(
        qd.data_ptr(), None, None, kd.data_ptr(), vd.data_ptr(), cache_end - 1, cache_end, cache_end,
        None, 0, got.data_ptr(), ws.data_ptr(), n, 0, torch.cuda.current_stream(gpu).cuda_stream)
    assert call(nb) == 0
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert call(nb - 1) == 1
