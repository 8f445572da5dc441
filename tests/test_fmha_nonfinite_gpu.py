"""FMHA with a NaN or an infinity among the keys: rows that see the key give
what the unsplit softmax gives, over every form that the key ranges take."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 5 * 2.0 ** -8 + 1e-4   # P rounded to bf16 (2^-8 of each at most), |v| below 5


@pytest.mark.parametrize("bad", [math.nan, math.inf])
@pytest.mark.parametrize("t,s,key", [
    (7, 7, 1), (20, 31, 15), (33, 33, 1), (24, 600, 300), (300, 300, 40), (900, 900, 700),     # square: 2, 3 and 4 chunks
    (2561, 2561, 100), (4096, 4096, 2100),            # split from 2561 tokens on
    (4097, 4097, 100),                                # unsplit
    (3000, 3400, 50), (40, 900, 450), (100, 1000, 3),
    (93, 24093, 12345), (93, 24093, 24050),           # halves that merge in LDS
    (8, 12000, 0), (3, 60003, 59000),                 # up to 128 chunks
])
def test_nonfinite_key(gpu, t, s, key, bad):
    from qwen36_attn.full_attention import fmha_prefill
    g = torch.Generator().manual_seed(t + s + key)
    q = torch.randn(t, 16, 256, generator=g).to(torch.bfloat16)
    k = torch.randn(s, 2, 256, generator=g).to(torch.bfloat16)
    v = torch.randn(s, 2, 256, generator=g).to(torch.bfloat16)
    qd, vd = q.to(gpu), v.to(gpu)
    clean = fmha_prefill(qd, k.to(gpu), vd).view(t, 16, 256).cpu()
    k[key, 1, 7] = bad
    print(f"nonfinite T={t} S={s} key={key} {bad}", flush=True)
    got = fmha_prefill(qd, k.to(gpu), vd).view(t, 16, 256).cpu()
    sees = torch.arange(t) + s - t >= key
    # the other KV head's rows are untouched; rows before the key may share a
    # wave with rows that see it, whose sums make the wave take new maxima, so
    # their P is rounded anew
    assert torch.equal(got[:, :8], clean[:, :8])
    assert ((got[~sees] - clean[~sees]).abs() <= 2 * TOL).all()
    got, qk = got[sees][:, 8:], q[sees][:, 8:, 7].float()
    if math.isnan(bad):
        assert got.isnan().all()
        return
    # a score of +inf makes the softmax NaN, one of -inf takes the key out
    assert got[qk > 0].isnan().all()
    rows = torch.nonzero(qk < 0)
    for r, h in rows[:: max(1, len(rows) // 12)].tolist():
        lim = s - t + int(torch.nonzero(sees)[r]) + 1
        keep = torch.arange(lim) != key
        x = q[sees][r, 8 + h].double()
        if keep.any():
            p = torch.softmax(k[:lim, 1].double()[keep] @ x / 16, 0)
            assert (got[r, h].double() - p @ v[:lim, 1].double()[keep]).abs().max() <= TOL, (r, h)
        else:
            assert got[r, h].isnan().all()
