"""The decode's new K/V row, laid over the streamed block in LDS: positions at
the edges of a block, of the waves and of the rounds, with stale cache rows."""
import pytest
import torch

from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu

TOL = 2e-2   # bf16 output (P and the output rounded to bf16)


@pytest.mark.parametrize("position,cache_end", [
    (0, 1), (0, 40), (31, 32), (32, 33), (127, 128), (128, 129), (130, 700),
    (511, 512), (2050, 2051), (4095, 4096), (16384, 16385), (20000, 33000)])
def test_new_row_over_stale_cache(gpu, position, cache_end):
    from qwen36_attn.full_attention import decode_gqa
    g = torch.Generator().manual_seed(position + cache_end)
    q = torch.randn(16, 256, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(cache_end, 2, 256, generator=g).to(torch.bfloat16) for _ in range(2))
    kn, vn = k[position].clone(), v[position].clone()
    kd, vd = k.to(gpu), v.to(gpu)
    kd[position] = float("nan")   # whatever the row held is neither read nor used
    vd[position] = float("inf")
    out = decode_gqa(q.to(gpu), kd, vd, position, cache_end, kn.to(gpu), vn.to(gpu))
    torch.cuda.synchronize()
    assert torch.equal(kd[position].cpu(), kn) and torch.equal(vd[position].cpu(), vn)
    ref = O.decode_attention_f32(q, k, v, cache_end)
    assert (out.cpu().float() - ref.reshape(1, 4096).float()).abs().max().item() <= TOL


@pytest.mark.parametrize("cache_end,split_tokens", [
    (2000, 128), (2048, 128), (2049, 128), (4096, 128), (4097, 128), (8192, 128),
    (16384, 128), (16385, 128), (32768, 128)])
def test_combine_forms(gpu, cache_end, split_tokens):
    """16, 17, 32, 33, 64, 128, 129 and 256 splits: every form of the combine."""
    from qwen36_attn.full_attention import decode_gqa
    g = torch.Generator().manual_seed(cache_end)
    q = torch.randn(16, 256, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(cache_end, 2, 256, generator=g).to(torch.bfloat16) for _ in range(2))
    out = decode_gqa(q.to(gpu), k.to(gpu), v.to(gpu), cache_end - 1, cache_end,
                     split_tokens=split_tokens)
    ref = O.decode_attention_f32(q, k, v, cache_end)
    assert (out.cpu().float() - ref.reshape(1, 4096).float()).abs().max().item() <= TOL
