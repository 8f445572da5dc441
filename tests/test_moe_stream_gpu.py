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
