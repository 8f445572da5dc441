"""GPU parity of the MoE block's streaming expert GEMMs (short prompts) at the
edges of their 64-row tiles and of the dispatch, against the CPU oracle."""
import pytest
import torch

from oracle import attention_oracle as O
from qwen36_attn import synthetic as syn

pytestmark = pytest.mark.gpu

TOL = 2e-2   # the block's output tolerance (bf16 roundings of each expert's rows)


@pytest.mark.parametrize("n_experts,tokens", [
    (8, 32), (8, 33), (8, 64),   # every expert has every token: one full tile
    (8, 65),                     # the first two-tile groups (64 and 1 rows)
    (8, 129), (8, 193),          # three and four tiles: 64-row tiles and a one-row rest
    (12, 70),                    # uneven groups around one tile
    (256, 2), (256, 16),         # few experts, one row each
    (64, 64), (64, 65),          # one and two column blocks per down workgroup
    (256, 17), (32, 512), (32, 513),   # alignment in two launches; router forms
    (256, 63), (252, 66),        # router rows and tokens past the tiles' ends
])
def test_stream_tile_edges(gpu, n_experts, tokens):
    from qwen36_attn.moe import MoEBlock
    g = syn.gen(900 + n_experts + tokens)
    w = syn.moe_weights(g, n_experts=n_experts)
    inp = syn.randn((tokens, 2048), g, 0.5)
    attn = syn.randn((tokens, 2048), g, 0.5)
    block = MoEBlock({k: v.to(gpu) for k, v in w.items()})
    print(f"moe stream E={n_experts} T={tokens}", flush=True)
    out, ids, rw, _, _ = block.prefill(inp.to(gpu), attn.to(gpu), debug=True)
    torch.cuda.synchronize()
    ref = O.moe_block(inp, attn, w, forced_ids=ids.cpu(), grouped=True)
    assert torch.isfinite(out).all()
    assert (out.cpu().float() - ref.float()).abs().max().item() <= TOL


def test_stream_one_expert_holds_most_rows(gpu):
    """A group of many tiles beside groups of none: identical tokens select
    the same eight experts, 300 rows each."""
    from qwen36_attn.moe import MoEBlock
    g = syn.gen(950)
    w = syn.moe_weights(g, n_experts=64)
    row = syn.randn((1, 2048), g, 0.5)
    inp, attn = row.repeat(300, 1).contiguous(), torch.zeros(300, 2048, dtype=torch.bfloat16)
    block = MoEBlock({k: v.to(gpu) for k, v in w.items()})
    out, ids, _, _, _ = block.prefill(inp.to(gpu), attn.to(gpu), debug=True)
    torch.cuda.synchronize()
    assert (ids == ids[:1]).all()
    assert torch.equal(out, out[:1].expand_as(out))   # every row is computed alike
    ref = O.moe_block(inp[:1], attn[:1], w, forced_ids=ids[:1].cpu(), grouped=True)
    assert (out[:1].cpu().float() - ref.float()).abs().max().item() <= TOL


@pytest.mark.parametrize("n_experts,tokens,copies", [
    (8, 2050, 1),      # every group has every token: nine tiles of 228 rows
    (64, 2300, 1),     # about 290 rows a group: two even tiles, ragged blocks
    (256, 6145, 1),    # two column blocks per down workgroup
    (64, 2304, 2304),  # identical tokens: eight groups of 9 tiles, the rest empty
])
def test_long_prompt_tiles_sampled_rows(gpu, n_experts, tokens, copies):
    """The 256-row tiles of long prompts: sampled rows against the oracle."""
    from qwen36_attn.moe import MoEBlock
    g = syn.gen(960 + n_experts + tokens)
    w = syn.moe_weights(g, n_experts=n_experts)
    inp = syn.randn((tokens // copies, 2048), g, 0.5).repeat(copies, 1).contiguous()
    attn = syn.randn((tokens // copies, 2048), g, 0.5).repeat(copies, 1).contiguous()
    block = MoEBlock({k: v.to(gpu) for k, v in w.items()})
    print(f"moe tiles E={n_experts} T={tokens}", flush=True)
    out, ids, _, _, _ = block.prefill(inp.to(gpu), attn.to(gpu), debug=True)
    torch.cuda.synchronize()
    out, ids = out.cpu(), ids.cpu()
    assert torch.isfinite(out.float()).all()
    if copies > 1:
        assert torch.equal(out, out[:1].expand_as(out))
    rows = torch.cat([torch.tensor([0, tokens - 1]),
                      torch.randperm(tokens, generator=syn.gen(961))[:24]])
    ref = O.moe_block(inp[rows], attn[rows], w, forced_ids=ids[rows], grouped=True)
    assert (out[rows].float() - ref.float()).abs().max().item() <= TOL


def _gate_pairs(n):
    """n (gate, up) values: every finite, normal bf16 gate whose SiLU is well inside
    bf16's range with up = 1, the rest random products."""
    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    act = torch.nn.functional.silu(g.double())
    g = g[g.isfinite() & (act.abs() > 2.0 ** -100) & (act.abs() < 2.0 ** 100)]
    rest, rng = n - len(g), syn.gen(971)
    more = torch.randn(rest, generator=rng) * 2.0 ** torch.randint(-8, 6, (rest,), generator=rng)
    more = more.clamp(-80, 80)   # (e^-g overflows 32 bits from 88.7 on)
    ups = torch.randn(rest, generator=rng) * 2.0 ** torch.randint(-6, 6, (rest,), generator=rng)
    u = torch.cat([torch.ones(len(g)), ups]).to(torch.bfloat16)
    return torch.cat([g, more.to(torch.bfloat16)]), u


@pytest.mark.parametrize("copies", [1, 25])   # 88 tokens (streaming kernels), 2200 (256-row tiles)
def test_silu_product_bits_every_gate(gpu, copies):
    """The experts' activation has the exact form's bits: fast SiLU with the exact
    fallback (prefill) against the one-token decode (exact SiLU).  Hidden column 0 is 1
    in every token's normalised row and the only one that the experts read, so a gate
    or up value is its weight; token i's column 1 + i selects its eight experts with
    weights of 1/8; and down passes an expert's 512 activations to columns of the output
    where the residual is 0 and no other expert writes: out = act / 8, exactly."""
    from qwen36_attn.moe import MoEBlock
    bf = torch.bfloat16
    gates, ups = _gate_pairs(240 * 512)
    # gates and products that are not finite or past the fast form's range, an expert each
    special = [(float("inf"), 1.0), (float("-inf"), 1.0), (float("nan"), 1.0), (60.5, 3.3e38),
               (-60.5, 2.0 ** 100), (88.0, -3.3e38), (3.0e38, 2.0), (2.0, float("nan"))]
    w = {"post_attention_layernorm": torch.full((2048,), -31 / 32, dtype=bf, device=gpu),
         "router": torch.zeros(256, 2048, dtype=bf), "shared_gate": torch.zeros(1, 2048, dtype=bf),
         "expert_gate_up": torch.zeros(256, 1024, 2048, dtype=bf, device=gpu),
         "expert_down": torch.zeros(256, 2048, 512, dtype=bf, device=gpu),
         "shared_gate_proj": torch.zeros(512, 2048, dtype=bf),
         "shared_up_proj": torch.zeros(512, 2048, dtype=bf),
         "shared_down_proj": torch.zeros(2048, 512, dtype=bf)}
    w["expert_gate_up"][:240, :512, 0] = gates.view(240, 512).to(gpu)
    w["expert_gate_up"][:240, 512:, 0] = ups.view(240, 512).to(gpu)
    j = torch.arange(512, device=gpu)
    for e in range(240):
        w["expert_down"][e, 512 + 512 * (e % 3) + j, j] = 1
    inp = torch.zeros(88, 2048, dtype=bf)
    inp[:, 0] = 64
    for t in range(88):
        inp[t, 1 + t] = 64      # rms 2, scaled by 1/32: the normalised row holds 1, 1 and zeros
        mine = [3 * t, 3 * t + 1, 3 * t + 2] if t < 80 else [160 + t]
        w["router"][mine + [*range(248, 256)][:8 - len(mine)], 1 + t] = 4
    for i, (gate, up) in enumerate(special):
        w["expert_gate_up"][240 + i, 100, 0] = gate
        w["expert_gate_up"][240 + i, 612, 0] = up
        w["expert_down"][240 + i, 512 + 100, 100] = 1
    block = MoEBlock({k: v.to(gpu) for k, v in w.items()})
    x = inp.repeat(copies, 1).contiguous().to(gpu)
    print(f"moe silu T={len(x)}", flush=True)
    out, _, rw, _, _ = block.prefill(x, torch.zeros_like(x), debug=True)
    assert (rw == 0.125).all()
    dec = torch.cat([block.decode(x[t:t + 1], torch.zeros_like(x[:1])) for t in range(88)])
    for rep in out.view(copies, 88, 2048):
        assert torch.equal(rep.nan_to_num(nan=7.0), dec.nan_to_num(nan=7.0))
    # ... and the activation is what shows: one rounding to bf16 of the 64-bit product
    # (the fp32 exponential and product move it over a midpoint once in some thousands)
    act = (dec[:80, 512:].double() * 8).cpu().reshape(-1)
    want = torch.nn.functional.silu(gates.double()) * ups.double()
    assert ((act - want).abs() <= 2.0 ** -8 * 1.001 * want.abs()).all()
    assert (act == want.to(bf).double()).double().mean() > 0.999
    shown = dec[80:, 612].float().cpu()
    assert shown[0] == float("inf") and shown[[1, 2, 7]].isnan().all()
    assert shown[3] == float("inf") and shown[5] == float("-inf") and shown[6] == float("inf")
    assert -1 < shown[4] * 8 / (60.5 * 2.0 ** 100 * 2.0 ** -87.28) < -0.9
