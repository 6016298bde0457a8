"""Head dims 65 to 96: kernels that leave the last quarter of a 128-wide tile out.  The same call with zeros appended to head dim 104 goes
through the kernels that do not, and what they add are products with zeros: the same bits, in every form of the keys, at tiles and parts
that end anywhere.  The scale is given, so it does not depend on the padding."""
import pytest
import torch

from flash_sparse_attn import flash_sparse_attn_func, flash_sparse_attn_varlen_func
from _util import set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(call, tensors, dout):
    """Outputs and gradients of call(q, k, v, ...) as it is, and with q, k, v and dout padded (and cut back)."""
    d = dout.shape[-1]
    runs = []
    for width in (d, 104):
        def padded(t):
            return torch.nn.functional.pad(t, (0, width - d)).contiguous()

        leaves = [(padded(t) if i < 3 else t.clone()).requires_grad_(True) for i, t in enumerate(tensors)]
        out = call(*leaves)
        grads = torch.autograd.grad(out, leaves, padded(dout))
        runs.append([out[..., :d]] + [g[..., :d] if i < 3 else g for i, g in enumerate(grads)])
        if width > d:
            assert all(not t[..., d:].any() for t in (out,) + grads[:3])
    for i, (a, b) in enumerate(zip(*runs)):
        assert torch.equal(a, b), ("out", "dq", "dk", "dv", "dbias")[i]


def _normal(g, dtype, *shape):
    return torch.randn(*shape, generator=g).to(dtype).to(DEV)


@pytest.mark.parametrize("d,dtype", [(72, torch.bfloat16), (88, torch.float16), (96, torch.bfloat16)])
@pytest.mark.parametrize("B,Lq,Lk,H,Hk,kept,compact,causal", [
    (2, 300, 777, 4, 2, 200, "2", True),    # compacted, few row blocks
    (1, 2300, 2300, 8, 4, 700, "2", True),  # ... and more of them than CUs hold in one group
    (1, 150, 260, 6, 1, 129, "2", False),   # a last block of one key
    (2, 129, 513, 4, 4, 300, "0", True),    # masked, not compacted: parts of key blocks
    (1, 1100, 400, 16, 8, 200, "0", False),
    (1, 1300, 1300, 2, 1, 0, "0", True),    # no mask, no bias: two key groups
    (2, 2050, 2050, 16, 16, 0, "0", True),  # ... one
])
def test_column_form(B, Lq, Lk, H, Hk, kept, compact, causal, d, dtype):
    print("column", B, Lq, Lk, H, Hk, kept, compact, causal, d, dtype, flush=True)
    g = torch.Generator().manual_seed(Lq + d)
    tensors = [_normal(g, dtype, B, Lq, H, d), _normal(g, dtype, B, Lk, Hk, d), _normal(g, dtype, B, Lk, Hk, d)]
    dout, mask = _normal(g, dtype, B, Lq, H, d), None
    if kept:
        scores = _normal(g, dtype, B, Hk, 1, Lk)
        mask = torch.zeros(scores.shape, dtype=torch.bool, device=DEV).scatter_(-1, scores.float().topk(kept, -1).indices, True)
        tensors.append(scores)
    set_compact(compact)
    try:
        _both(lambda q, k, v, bias=None: flash_sparse_attn_func(q, k, v, mask, bias, 0.11, causal), tensors, dout)
    finally:
        set_compact("auto")


@pytest.mark.parametrize("lens,H,Hk,d,causal", [
    ([1025, 33, 1, 257], 4, 2, 72, True),
    ([700, 2100, 64, 1], 16, 16, 96, True),
    ([130, 1500], 2, 1, 80, False),
])
def test_ragged(lens, H, Hk, d, causal):
    print("ragged", lens, H, Hk, d, causal, flush=True)
    g = torch.Generator().manual_seed(d)
    n, cu = sum(lens), torch.tensor([0] + lens, dtype=torch.int32).cumsum(0, dtype=torch.int32).to(DEV)
    tensors = [_normal(g, torch.bfloat16, n, h, d) for h in (H, Hk, Hk)]
    _both(lambda q, k, v: flash_sparse_attn_varlen_func(q, k, v, cu, cu, max(lens), max(lens), softmax_scale=0.11, is_causal=causal), tensors,
          _normal(g, torch.bfloat16, n, H, d))
