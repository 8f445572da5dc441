"""FMHA over a long prefix: workgroups whose two halves share a tile's rows and
merge their halves of the chunk's keys in LDS.  Last chunks with an empty, a
one-key and a ragged second half, one-token last tiles, and rows that see none
of a half's keys, against the 64-bit softmax."""
import pytest
import torch

from oracle.attention_bounds import Row

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,s,scale", [
    (16, 88000, 1.0), (17, 83001, 1.0), (93, 40000, 1.0),   # 8 waves of rows
    (81, 18081, 1.0), (96, 15096, 1.0),          # a one-token (and an empty half), a full last tile
    (93, 24093, 1.0), (93, 24093, 12.0),         # large scores: halves of very different maxima
    (130, 11000, 1.0), (64, 22017, 1.0), (257, 5500, 1.0),
    (93, 15745, 1.0), (500, 2911, 1.0), (672, 2200, 1.0), (673, 2200, 1.0), (656, 2185, 1.0)])
def test_pair_merge_matches_oracle(gpu, t, s, scale):
    from qwen36_attn.full_attention import fmha_prefill
    g = torch.Generator().manual_seed(3 * t + s)
    q = (torch.randn(t, 16, 256, generator=g) * scale).to(torch.bfloat16)
    k = torch.randn(s, 2, 256, generator=g).to(torch.bfloat16)
    v = torch.randn(s, 2, 256, generator=g).to(torch.bfloat16)
    # the first and the last key (the one key of a one-key half) carry large values,
    # so a row without one of them is far off
    v[0] *= 8
    v[-1] *= 8
    print(f"pairs T={t} S={s} scale={scale}", flush=True)
    got = fmha_prefill(q.to(gpu), k.to(gpu), v.to(gpu)).cpu().double()
    assert torch.isfinite(got).all()
    for r in sorted({0, 1, 15, t // 3, t // 2, t - 17, t - 16, t - 2, t - 1} & set(range(t))):
        lim = s - t + r + 1
        row = Row(q[r], k[:lim], v[:lim])
        assert ((got[r] - row.ref).abs() <= row.tol).all(), r
        # (with large scores few keys weigh anything)
        if scale == 1.0:
            assert row.sees([0]) and row.sees(slice(lim - 32, lim)) and (r < t - 1 or row.sees([lim - 1]))
