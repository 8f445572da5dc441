"""The decode's new K/V row, laid over the streamed block in LDS: positions at
the edges of a block, of the waves and of the rounds, with stale cache rows."""
import pytest
import torch

from oracle.attention_bounds import Row

pytestmark = pytest.mark.gpu


def _check(out, q, k, v, lost):
    """The output against 64 bits: P rounded to bf16 (Row), then the output (2^-8 of it at
    most).  Each of ``lost`` (a range of keys) left out would be seen."""
    row = Row(q, k, v)
    tol = row.tol + 2.0 ** -8 * row.ref.abs()
    assert ((out.cpu().double().view(4096) - row.ref).abs() <= tol).all()
    for keys in lost:
        if row.s > keys.stop - keys.start:
            assert ((row.without(keys) - row.ref).abs() > 2 * tol).any(), keys


@pytest.mark.parametrize("position,cache_end", [
    (0, 1), (0, 40), (31, 32), (32, 33), (127, 128), (128, 129), (130, 700),
    (511, 512), (2050, 2051), (4095, 4096), (16384, 16385), (20000, 33000)])
def test_new_row_over_stale_cache(gpu, position, cache_end):
    from qwen36_attn.full_attention import decode_gqa
    g = torch.Generator().manual_seed(position + cache_end)
    q = torch.randn(16, 256, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(cache_end, 2, 256, generator=g).to(torch.bfloat16) for _ in range(2))
    v[position] *= 16             # a row that is left out shows
    kn, vn = k[position].clone(), v[position].clone()
    kd, vd = k.to(gpu), v.to(gpu)
    kd[position] = float("nan")   # whatever the row held is neither read nor used
    vd[position] = float("inf")
    out = decode_gqa(q.to(gpu), kd, vd, position, cache_end, kn.to(gpu), vn.to(gpu))
    torch.cuda.synchronize()
    assert torch.equal(kd[position].cpu(), kn) and torch.equal(vd[position].cpu(), vn)
    _check(out, q, k, v, [slice(position, position + 1)])


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
    # blocks of 32 keys are dealt to the splits in turn
    nsplit = (cache_end + split_tokens - 1) // split_tokens
    blocks = torch.arange(cache_end) // 32
    _check(out, q, k, v, [])
    row = Row(q, k, v)
    for split in {0, 1, nsplit // 2, nsplit - 16, nsplit - 1} & set(range(nsplit)):
        assert row.sees(torch.nonzero(blocks % nsplit == split).flatten()), split
