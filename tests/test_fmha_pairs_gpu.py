"""FMHA over a long prefix: workgroups whose two halves share a tile's rows and
merge their halves of the chunk's keys in LDS.  Last chunks with an empty, a
one-key and a ragged second half, one-token last tiles, and rows that see none
of a half's keys, against the CPU oracle's SDPA."""
import pytest
import torch

from oracle import attention_oracle as O

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
    print(f"pairs T={t} S={s} scale={scale}", flush=True)
    got = fmha_prefill(q.to(gpu), k.to(gpu), v.to(gpu)).cpu()
    assert torch.isfinite(got).all()
    # fp32 rows against the fp32 oracle: only P is rounded to bf16, so o =
    # sum p_j v_j / sum p_j is off by at most 2^-9 max |v| (reached where one
    # key takes the whole row, as with large scores)
    tol = 2.0 ** -9 * v.float().abs().max().item() + 1e-4
    for r in sorted({0, 1, 15, t // 3, t // 2, t - 17, t - 16, t - 2, t - 1} & set(range(t))):
        lim = s - t + r + 1
        ref = O.prefill_attention(q[r:r + 1], k[:lim], v[:lim], position_start=lim - 1,
                                  out_dtype=torch.float32)
        assert (got[r:r + 1] - ref).abs().max().item() <= tol, r
