"""GPU parity of the FMHA's head-packed tiles (8 query heads x 4, 8, 16 or 32
tokens a tile) and key-range splits at the edges of the tiles and of the
split rule, against the CPU oracle's SDPA."""
import pytest
import torch

from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu

# fp32 rows against the fp32 oracle: only P is rounded to bf16, by at most 2^-8 of
# each term p_j v_j, independently (their sum stays below max |v| ~ 5)
TOL = 5e-3
TOL_BF16 = 2e-2   # the gated rows' bf16 roundings


@pytest.mark.parametrize("t,s", [
    (8, 8), (9, 9), (33, 33),                    # one chunk (unsplit) and its first split
    (8, 12000), (9, 12000), (13, 7700),          # 2 waves, one and two tiles
    (26, 7692), (26, 7693), (93, 1593),          # 2 / 4 waves; 12 tiles of 2 waves
    (3, 60003), (64, 30064),                     # 128 chunks; 8 waves
    (32, 24032), (33, 24033), (93, 24093),       # full and one-token last tiles
    (360, 360), (361, 361), (960, 960), (961, 961), (1345, 1345), (2113, 2113),
    (4096, 4096), (4097, 4097),                  # last split and first unsplit length
    (3072, 3400), (3073, 3400),                  # the same over a prefix
    (1376, 2376), (1900, 2156), (1900, 2400),    # three chunks in place of two; two
])
def test_tile_and_split_edges(gpu, t, s):
    from qwen36_attn.full_attention import fmha_prefill, fmha_prefill_gated, output_gate
    g = torch.Generator().manual_seed(5 * t + s)
    q = torch.randn(t, 16, 256, generator=g).to(torch.bfloat16)
    k = torch.randn(s, 2, 256, generator=g).to(torch.bfloat16)
    v = torch.randn(s, 2, 256, generator=g).to(torch.bfloat16)
    gate = torch.randn(t, 9216, generator=g).to(torch.bfloat16)
    print(f"tiles T={t} S={s}", flush=True)
    qd, kd, vd, gd = q.to(gpu), k.to(gpu), v.to(gpu), gate.to(gpu)[:, :8192]
    got = fmha_prefill(qd, kd, vd)
    gated = fmha_prefill_gated(qd, kd, vd, gd)
    assert torch.equal(gated, output_gate(got, gd))
    got, gated = got.cpu(), gated.cpu()
    assert torch.isfinite(got).all()
    rows = {0, 7, 8, 15, 16, 31, 32, t // 3, t // 2, 2 * t // 3, t - 33, t - 32, t - 9, t - 1}
    for r in sorted(x for x in rows if 0 <= x < t):
        lim = s - t + r + 1
        ref = O.prefill_attention(q[r:r + 1], k[:lim], v[:lim], position_start=lim - 1,
                                  out_dtype=torch.float32)
        assert (got[r:r + 1] - ref).abs().max().item() <= TOL, r
        gref = O.output_gate(ref.to(torch.bfloat16), O.split_q_gate(gate[r:r + 1, :8192])[1])
        assert (gated[r:r + 1].float() - gref.float()).abs().max().item() <= TOL_BF16, r


@pytest.mark.parametrize("t,s", [(5, 5), (700, 700), (2050, 2050), (40, 5000)])
def test_provider_unsplit_tiles(gpu, t, s):
    """Unsplit launches of the provider ABI (a stream that does not own the
    split scratch): 2-, 4- and 8-wave tiles give the split result's rows
    within P's rounding."""
    from qwen36_attn import _lib
    from qwen36_attn.full_attention import fmha_prefill
    lib = _lib.load(("qrt_ck_fmha_bf16_launch_ex",))
    assert lib.qrt_ck_fmha_prepare(64) == 0
    g = torch.Generator().manual_seed(t)
    q, k, v = (torch.randn(n, h, 256, generator=g).to(torch.bfloat16).to(gpu)
               for n, h in ((t, 16), (s, 2), (s, 2)))
    # the current stream claims the scratch; another stream runs unsplit
    outs = [torch.empty(t, 4096, device=gpu) for _ in range(2)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for out, st in zip(outs, (torch.cuda.current_stream(), side)):
        assert lib.qrt_ck_fmha_bf16_launch_ex(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                              out.data_ptr(), t, s, st.cuda_stream) == 0
    torch.cuda.synchronize()
    ref = fmha_prefill(q, k, v)
    for out in outs:
        assert (out - ref).abs().max().item() <= 2 * TOL


def test_long_split_without_workspace_runs_unsplit(gpu):
    """2561 tokens and more split only if the caller gives the workspace; up
    to 2560 a missing one is refused."""
    from qwen36_attn import _lib
    from qwen36_attn.full_attention import fmha_prefill
    lib = _lib.load(("qwen36_fmha_prefill",))
    t = 2561
    assert lib.qwen36_fmha_prefill_workspace_bytes(t, t) > 0
    g = torch.Generator().manual_seed(t)
    q, k, v = (torch.randn(t, h, 256, generator=g).to(torch.bfloat16).to(gpu) for h in (16, 2, 2))
    out = torch.empty(t, 4096, device=gpu)
    st = torch.cuda.current_stream().cuda_stream
    args = (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr())
    assert lib.qwen36_fmha_prefill(*args, 2560, 2560, None, 0, st) == 1
    assert lib.qwen36_fmha_prefill(*args, t, t, None, 0, st) == 0
    assert (out - fmha_prefill(q, k, v)).abs().max().item() <= 2 * TOL


@pytest.mark.parametrize("t,s", [
    (1, 1), (3, 3), (4, 4), (5, 5), (1, 32), (29, 32), (32, 32),       # one chunk
    (1, 33), (33, 33), (48, 48), (49, 49), (5, 60), (17, 200),         # square
    (1, 257), (4, 320), (8, 1024), (9, 512), (24, 700), (45, 1000), (48, 1024),   # chunks of 32, 64 keys
    (48, 1025), (49, 1024)])                                           # 2 waves
def test_few_rows(gpu, t, s):
    """Tiles of one wave (4 tokens) and the one chunk of up to 32 keys: rows against
    64 bits, the gated rows' bits against the gate applied to the plain ones, and the
    optional workspace of one chunk."""
    from oracle.attention_bounds import Row
    from qwen36_attn import _lib
    from qwen36_attn.full_attention import fmha_prefill, fmha_prefill_gated, output_gate
    g = torch.Generator().manual_seed(1000 * t + s)
    q, k, v = (torch.randn(n, h, 256, generator=g).to(torch.bfloat16) for n, h in ((t, 16), (s, 2), (s, 2)))
    qg = torch.randn(t, 8192, generator=g).to(torch.bfloat16).to(gpu)
    qd, kd, vd = q.to(gpu), k.to(gpu), v.to(gpu)
    print(f"few rows T={t} S={s}", flush=True)
    rows, gated = fmha_prefill(qd, kd, vd), fmha_prefill_gated(qd, kd, vd, qg)
    for r in sorted({0, 3, 4, t // 2, t - 1} & set(range(t))):
        row = Row(q[r], k[:s - t + r + 1], v[:s - t + r + 1])
        assert ((rows[r].cpu().double() - row.ref).abs() <= row.tol).all(), r
    assert torch.equal(gated, output_gate(rows, qg))
    lib = _lib.load(("qwen36_fmha_prefill", "qwen36_fmha_prefill_gated"))
    st = torch.cuda.current_stream().cuda_stream
    out, out16 = torch.empty_like(rows), torch.empty_like(gated)
    plain = lib.qwen36_fmha_prefill(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(),
                                    t, s, None, 0, st)
    fused = lib.qwen36_fmha_prefill_gated(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), qg.data_ptr(),
                                          8192, out16.data_ptr(), t, s, None, 0, st)
    torch.cuda.synchronize()
    assert plain == fused == (0 if s <= 32 else 1)
    if s <= 32:
        assert torch.equal(out, rows) and torch.equal(out16, gated)
