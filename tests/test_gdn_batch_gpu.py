"""GPU parity of the batched vLLM-orientation update over sequence counts, row
strides and slot orders, against the CPU oracle."""
import pytest
import torch

from oracle import attention_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,pad", [(1, 0), (3, 8), (17, 24), (64, 0)])
def test_packed_decode_slots_and_strides(gpu, n, pad):
    from qwen36_attn.gated_deltanet import fused_recurrent_gated_delta_rule_packed_decode
    g = torch.Generator().manual_seed(40 + n)
    rows = torch.randn(n, 8192 + pad, generator=g).to(torch.bfloat16)
    a, b = (torch.randn(n, 32, generator=g).to(torch.bfloat16) for _ in range(2))
    a_log, dt = torch.randn(32, generator=g), torch.randn(32, generator=g)
    pool = torch.randn(n + 2, 32, 128, 128, generator=g) * 0.1
    index = torch.randperm(n + 2, generator=g)[:n].int()
    if n > 2:
        index[1] = -1   # a padding sequence
    dev = pool.to(gpu)
    out, _ = fused_recurrent_gated_delta_rule_packed_decode(
        rows.to(gpu)[:, :8192], a.to(gpu), b.to(gpu), a_log.to(gpu), dt.to(gpu), 128 ** -0.5,
        dev, ssm_state_indices=index.to(gpu))
    torch.cuda.synchronize()
    want = pool.clone()
    for i in range(n):
        sl = int(index[i])
        if sl < 0:
            continue
        q, k, v = rows[i, :2048], rows[i, 2048:4096], rows[i, 4096:8192]
        o, s = O.fused_sigmoid_gating_delta_rule_update(
            a_log, a[i:i + 1], b[i:i + 1], dt, q.reshape(1, 1, 16, 128), k.reshape(1, 1, 16, 128),
            v.reshape(1, 1, 32, 128), pool[sl:sl + 1].clone(), use_qk_l2norm_in_kernel=True)
        want[sl] = s[0]
        assert (out[i].cpu().float() - o.reshape(1, 32, 128).float()).abs().max().item() <= 2e-2
    # fp32 state: sums of 128 terms, a few ulps each
    assert (dev.cpu() - want).norm().item() <= 1e-5 * want.norm().item()
