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
    (8, 129), (8, 193),          # three and four tiles, dealt evenly
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


def test_silu_product_bits_every_gate(gpu):
    """The experts' activation keeps the exact form's bits: prefill rows (fast
    SiLU with the exact fallback) and the one-token decode (exact SiLU) of the
    same tokens agree to the last bit wherever both accumulate alike; here one
    weight column is live, so every product is a single exact term."""
    from qwen36_attn.moe import MoEBlock
    g = syn.gen(970)
    w = syn.moe_weights(g, n_experts=8)
    # expert rows read hidden column 0 only; down passes column 0 of act through
    for name in ("expert_gate_up", "shared_gate_proj", "shared_up_proj"):
        w[name][..., 1:] = 0
    for name in ("expert_down", "shared_down_proj"):
        w[name][..., 1:] = 0
    inp = syn.randn((256, 2048), g, 2.0)
    attn = torch.zeros(256, 2048, dtype=torch.bfloat16)
    block = MoEBlock({k: v.to(gpu) for k, v in w.items()})
    out, ids, _, logits, _ = block.prefill(inp.to(gpu), attn.to(gpu), debug=True)
    same = 0
    for t in range(256):
        d, dids, _, dlogits = block.decode(inp[t:t + 1].to(gpu), attn[t:t + 1].to(gpu), debug=True)
        if torch.equal(dids, ids[t]) and torch.equal(dlogits, logits[t]):
            same += 1
            assert torch.equal(d[0], out[t]), t
    assert same >= 64
