"""Sums of the parts of the compacted dK/dV kernels: few units with many slots each (their slots are spread over threads and added up
through LDS, 1, 2, 4 or 8 chains side by side), and many units with few.  Against the fp32 eager restatement with the tolerances of
the gradients, and bit-equal on a second run: the sums have a fixed order (but for dBias that atomics add up)."""
import pytest
import torch

from oracle import eager
from _util import assert_grad_close, make_inputs, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,Hb,kept,causal,dtype", [
    (1, 100, 300, 2, 2, 64, 2, 200, False, torch.bfloat16),    # 1 or 2 slots a unit: one chain
    (1, 250, 250, 2, 2, 64, 0, 130, True, torch.float16),      # up to 4 slots, a last block of two keys, no bias
    (1, 250, 333, 4, 2, 128, 4, 333, False, torch.bfloat16),   # 8 slots; a bias row per query head
    (1, 320, 320, 8, 1, 128, 1, 200, True, torch.bfloat16),    # up to 40 slots: eight chains
    (2, 700, 700, 4, 1, 96, 1, 257, True, torch.float16),      # head dim below the instantiation's: 12 chunks of columns
    (2, 513, 513, 12, 2, 64, 12, 129, True, torch.bfloat16),   # slots of several local heads
    (2, 300, 300, 4, 2, 200, 2, 150, True, torch.bfloat16),    # two halves of a workgroup share the items
    (1, 1030, 1030, 8, 2, 256, 1, 500, False, torch.float16),  # one bias row for all kv heads: atomics
    (16, 130, 700, 2, 1, 128, 1, 640, False, torch.bfloat16),  # 80 units: whole 16-column items without LDS
    (16, 200, 640, 8, 2, 64, 2, 600, True, torch.float16),     # 160 units with a dBias of several heads to fold
])
def test_part_sums(B, Lq, Lk, H, Hk, D, Hb, kept, causal, dtype):
    from flash_sparse_attn import flash_sparse_attn_func

    print("sums", B, Lq, Lk, H, Hk, D, Hb, kept, causal, dtype, flush=True)
    set_compact("2")
    q, k, v, mask, bias = make_inputs(B, Lq, Lk, H, Hk, D, (B, Hb, 1, Lk) if Hb else None, (B, Hk, 1, Lk), kept, seed=Lq + D, dtype=dtype)
    q, k, v, mask = [t.to(DEV) for t in (q, k, v, mask)]
    leaves = [t.requires_grad_(True) for t in (q, k, v)] + ([bias.to(DEV).requires_grad_(True)] if Hb else [])
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    ref = eager.attention_forward_backward(q.detach(), k.detach(), v.detach(), mask, leaves[3].detach() if Hb else None, None, causal, dout)

    def grads():
        out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3] if Hb else None, None, causal)
        return torch.autograd.grad(out, leaves, dout)

    first, again = grads(), grads()
    for got, want, name in zip(first, ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got, want, name)
    for x, y in list(zip(first, again))[:3 if Hb == 1 and Hk > 1 else 4]:
        assert torch.equal(x, y)
