"""Sums of the parts of the compacted dK/dV kernels, both ways: a thread per sum, or several chains side by side (their slots are spread over
threads and added up through LDS, 1, 2, 4 or 8 chains).  Which way a case goes and how many parts its units have is read from the plan that the
device made.  Against the fp32 eager restatement with the tolerances of the gradients, and bit-equal on a second run: the sums have
a fixed order (but for dBias that atomics add up)."""
import pytest
import torch

from oracle import eager
from _util import assert_grad_close, make_inputs, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


def plan_in(ws, pairs, units):
    """The dK/dV plan in a backward's workspace: (query head groups, segments, summed by chains).  It lies at a multiple of 256 bytes:
    the number of units, ..., the lists' place, no overflow, ..., the units' prefix over the pairs."""
    words = ws[:ws.numel() // 256 * 256].view(torch.int32).reshape(-1, 64).cpu()
    at = (words[:, 0] == units) & (words[:, 5] == 8 + pairs + 1) & (words[:, 6] == 0) & (words[:, 8] == 0) & (words[:, 9] == units // pairs)
    found = words[at]
    assert found.shape[0] == 1
    return int(found[0, 1]), int(found[0, 2]), int(found[0, 7])


# parts: (groups of query heads, segments) of a unit at most; a unit that few queries see has fewer segments
@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,Hb,kept,causal,parts,chains,dtype", [
    # a thread per sum
    (1, 100, 300, 2, 2, 64, 2, 200, False, (1, 2), 0, torch.bfloat16),
    (1, 250, 250, 2, 2, 64, 0, 130, True, (1, 4), 0, torch.float16),      # a last block of two keys, no bias
    (1, 250, 333, 4, 2, 128, 4, 333, False, (2, 4), 0, torch.bfloat16),   # a bias row per query head
    (2, 300, 300, 4, 2, 200, 2, 150, True, (2, 5), 0, torch.bfloat16),    # two halves of a workgroup share the items
    (1, 1030, 1030, 8, 2, 256, 1, 500, False, (4, 9), 0, torch.float16),  # one bias row for all kv heads: atomics
    (16, 130, 700, 2, 1, 128, 1, 640, False, (2, 3), 0, torch.bfloat16),  # 80 units
    (16, 200, 640, 8, 2, 64, 2, 600, True, (4, 1), 0, torch.float16),     # 160 units
    (8, 800, 800, 12, 2, 64, 2, 630, True, (6, 3), 0, torch.float16),     # a dBias column of 18, 12 or 6 terms
    (16, 300, 300, 12, 2, 200, 2, 290, True, (6, 2), 0, torch.bfloat16),  # ... of 12 or 6, by halves of a workgroup
    (32, 300, 300, 12, 2, 64, 2, 290, True, (3, 1), 0, torch.bfloat16),   # several heads in a part: 6 terms
    (24, 200, 200, 32, 2, 64, 2, 200, False, (8, 1), 0, torch.float16),   # ... 16 terms
    (8, 400, 400, 12, 2, 128, 12, 400, False, (6, 1), 0, torch.bfloat16),
    # several chains: up to 8
    (1, 600, 600, 1, 1, 64, 1, 128, True, (1, 10), 1, torch.bfloat16),
    (1, 1030, 1030, 2, 1, 64, 1, 257, True, (2, 9), 1, torch.bfloat16),   # units of 18, fewer and 2 slots: 8 to 1 chains
    (1, 320, 320, 8, 1, 128, 1, 200, True, (8, 5), 1, torch.bfloat16),
    (2, 700, 700, 4, 1, 96, 1, 257, True, (4, 11), 1, torch.float16),     # head dim below the instantiation's: 12 chunks of columns
    (2, 513, 513, 12, 2, 64, 12, 129, True, (6, 9), 1, torch.bfloat16),   # a bias row per query head
    (1, 1030, 1030, 8, 1, 256, 1, 200, True, (8, 6), 1, torch.float16),   # two halves of a workgroup share the items
    (1, 1030, 1030, 8, 2, 256, 1, 128, False, (4, 9), 1, torch.float16),  # ... one bias row for all kv heads: atomics
    (2, 1030, 1030, 4, 2, 64, 0, 129, False, (2, 9), 1, torch.float16),   # no bias
    (8, 513, 513, 12, 2, 64, 2, 513, True, (6, 3), 1, torch.float16),     # many units
    (1, 500, 500, 32, 1, 64, 1, 200, True, (32, 8), 1, torch.float16),    # 256 slots
])
def test_part_sums(B, Lq, Lk, H, Hk, D, Hb, kept, causal, parts, chains, dtype, monkeypatch):
    from flash_sparse_attn import _cabi, flash_sparse_attn_func, flash_sparse_attn_interface as interface

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

    made, scratch = [], interface._scratch_with_room  # (the Python path's calls, whose workspaces can be looked into)
    monkeypatch.setattr(interface, "_scratch_with_room", lambda *a: made.append(scratch(*a).zero_()) or made[-1])
    monkeypatch.setattr(_cabi, "host", _cabi._NoHost)
    for x, y in list(zip(first, grads()))[:3 if Hb == 1 and Hk > 1 else 4]:
        assert torch.equal(x, y)
    assert plan_in(made[-1], B * Hk, B * Hk * -(-kept // 128)) == (*parts, chains)


# (not one key: P is 1 there and dP - D zero but for its rounding, 2^-8 of terms that cancel, so no relative bound holds for dQ and dK)
@pytest.mark.parametrize("kept", [2, 32, 33, 64, 65, 96, 97, 160, 161, 256])
@pytest.mark.parametrize("Lq,H,D,Hb,causal", [(33, 1, 128, 1, False), (1030, 2, 128, 2, True), (300, 8, 96, 8, True)])
def test_waves_behind_the_last_kept_key(kept, Lq, H, D, Hb, causal):
    """Last blocks of one to four waves with keys, in one step and in several, whole and in parts (whose sums of dropped columns nobody
    writes: the second run's scratch holds what the first left, and a NaN there must not show)."""
    print("waves", kept, Lq, H, D, Hb, causal, flush=True)
    from flash_sparse_attn import flash_sparse_attn_func

    set_compact("2")
    q, k, v, mask, bias = make_inputs(1, Lq, 300, H, 1, D, (1, Hb, 1, 300), (1, 1, 1, 300), kept, seed=kept, dtype=torch.bfloat16)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v, bias)]
    mask, dout = mask.to(DEV), torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(DEV)
    ref = eager.attention_forward_backward(*[t.detach() for t in leaves[:3]], mask, leaves[3].detach(), None, causal, dout)
    runs = []
    for _ in range(2):
        out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3], None, causal)
        runs.append(torch.autograd.grad(out, leaves, dout))
        torch.empty(1 << 22, device=DEV).fill_(float("nan"))  # (what the next call's scratch may be made of)
    for got, want, name in zip(runs[0], ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got, want, name)
    assert all(torch.equal(x, y) for x, y in zip(*runs))
