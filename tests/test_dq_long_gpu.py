"""dQ of the column form where whole stretches of keys are dropped: tiles are skipped by a bitmap, which covers 2^20 keys.
A hundred keys and more are kept: with a few, P is near 1 and dP about sqrt(D), whose rounding to 8 bits alone -- D^.5 2^-9 P --
reaches the absolute 5e-2 that the helper grants elements near zero."""
import pytest
import torch

from oracle import eager
from _util import assert_grad_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("Lq,Lk,H,Hk,D,causal,keep", [
    (200, 1300, 2, 1, 256, False, [(700, 805), (1290, 1300)]),
    (300, 1300, 2, 2, 256, True, [(0, 101), (1031, 1064)]),
    (129, 2081, 2, 1, 128, False, [(7, 139), (2080, 2081)]),
    (3, (1 << 19) + 96, 1, 1, 256, False, [(5, 70), ((1 << 19) - 1, (1 << 19) + 40)]),
    (3, (1 << 20) - 31, 1, 1, 128, False, [(31, 133), ((1 << 19) + 33, (1 << 19) + 134), ((1 << 20) - 131, (1 << 20) - 31)]),
    (3, 1 << 20, 2, 1, 64, False, [(100, 230), ((1 << 20) - 1, 1 << 20)]),
])
def test_dropped_stretches(Lq, Lk, H, Hk, D, causal, keep):
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    print("stretches", Lq, Lk, H, Hk, D, causal, flush=True)
    _cabi.set_compact_mode(_cabi.COMPACT_NEVER)
    g = torch.Generator(device=DEV).manual_seed(Lq + D)
    q, dout = [torch.randn(1, Lq, H, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2)]
    k, v = [torch.randn(1, Lk, Hk, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2)]
    bias = torch.randn(1, Hk, 1, Lk, generator=g, device=DEV).to(torch.bfloat16)
    kept = torch.cat([torch.arange(a, b, device=DEV) for a, b in keep])
    mask = torch.zeros(1, Hk, 1, Lk, dtype=torch.bool, device=DEV)
    mask[..., kept] = True
    leaves = [t.requires_grad_(True) for t in (q, k, v, bias)]
    grads = torch.autograd.grad(flash_sparse_attn_func(*leaves[:3], mask, leaves[3], None, causal), leaves, dout)
    if Lk < 4096:
        ref = eager.attention_forward_backward(*[t.detach() for t in leaves[:3]], mask, bias.detach(), None, causal, dout)[1:]
        for got, want, name in zip(grads, ref, ("dq", "dk", "dv", "dbias")):
            assert_grad_close(got, want, name)
        return
    # the kept keys alone
    ref = eager.attention_forward_backward(q.detach(), k.detach()[:, kept], v.detach()[:, kept], mask[..., kept], bias.detach()[..., kept], None, False, dout)[1:]
    for got, want, name in zip((grads[0], grads[1][:, kept], grads[2][:, kept], grads[3][..., kept]), ref, ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got, want, name)
    dropped = ~mask[0, 0, 0]
    assert not grads[1][:, dropped].any() and not grads[2][:, dropped].any() and not grads[3][..., dropped].any()
