"""dK / dV / dBias with a mask or bias row per query at head dims up to 64, rows of whole 16-key pieces: row and key counts that end
inside a step, a wave or a workgroup, waves without keys, key blocks above the diagonal (cleared by other workgroups), segments, one
to many heads per bias row, masks as bytes and as bits -- against the C oracle."""
import pytest
import torch

from oracle import c_oracle
from _util import assert_grad_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,hm,hb,rows,causal,bits", [
    (1, 70, 144, 4, 2, 64, 2, 2, 70, True, False),     # heads share the bias rows
    (1, 70, 144, 4, 2, 64, 2, 2, 70, False, True),
    (2, 33, 272, 2, 2, 64, 2, 2, 33, False, False),    # a last key block of one wave, half full
    (1, 300, 16, 4, 1, 40, 1, 1, 300, True, False),    # rows without visible keys
    (1, 513, 128, 4, 4, 64, 0, 4, 513, True, False),   # no mask; one row in the last step
    (1, 160, 640, 2, 2, 64, 2, 2, 160, True, True),
    (1, 700, 704, 4, 2, 64, 4, 4, 700, True, False),   # a bias row per query head of a group
    (2, 700, 704, 6, 3, 64, 3, 3, 700, True, True),
    (1, 200, 192, 4, 2, 64, 2, 2, 1, True, False),     # a bias value per key: column sums
    (1, 200, 192, 4, 2, 64, 4, 4, 1, False, False),
    (2, 129, 80, 2, 2, 64, 1, 0, 0, True, False),
    (1, 31, 48, 2, 1, 8, 1, 1, 31, False, False),
    (1, 1100, 1104, 2, 2, 64, 2, 2, 1100, True, False),
])
def test_against_oracle(B, Lq, Lk, H, Hk, d, hm, hb, rows, causal, bits, dtype):
    from flash_sparse_attn import flash_sparse_attn_func
    from flash_sparse_attn.utils.mask import mask_bits_of, topk_mask

    print("dkdv", B, Lq, Lk, H, Hk, d, hm, hb, rows, causal, bits, dtype, flush=True)
    g = torch.Generator().manual_seed(Lq * 1000 + Lk)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    q, k, v, dout = r(B, Lq, H, d), r(B, Lk, Hk, d), r(B, Lk, Hk, d), r(B, Lq, H, d)
    bias = r(B, hb, rows, Lk) if hb else None
    if bits:
        mask_dev = topk_mask(r(B, hm, Lq, Lk).to(DEV), None, Lk // 2, torch.finfo(dtype).min)
        assert mask_bits_of(mask_dev) is not None
        mask = mask_dev.cpu()
    else:
        mask = torch.rand(B, hm, Lq, Lk, generator=g) < 0.5 if hm else None
        mask_dev = None if mask is None else mask.to(DEV)
    ref = c_oracle.backward(q, k, v, dout, mask, bias, d ** -0.5, causal)
    runs = []
    for _ in range(2):
        leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)] + ([bias.to(DEV).requires_grad_(True)] if hb else [])
        out = flash_sparse_attn_func(*leaves[:3], mask_dev, leaves[3] if hb else None, None, causal)
        torch.full((64 << 20,), float("nan"), device=DEV)  # (what the gradients' memory may hold before)
        runs.append(torch.autograd.grad(out, leaves, dout.to(DEV)))
    for got, again, want, name in zip(*runs, ref, ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got.cpu(), want, name)
        assert torch.equal(got, again), name


def test_dbias_of_more_than_4_gib():
    """Rows above the diagonal are cleared wherever they lie: L = 46400, the first pieces of the last rows lie beyond 2^32 bytes."""
    from flash_sparse_attn import flash_sparse_attn_func

    L, D = 46400, 64
    g = torch.Generator(device=DEV).manual_seed(46)
    q, k, v, dout = [torch.randn(1, L, 1, D, generator=g, device=DEV).bfloat16() for _ in range(4)]
    bias = torch.empty(1, 1, L, L, dtype=torch.bfloat16, device=DEV)
    for r in range(0, L, 6400):
        bias[0, 0, r:r + 6400] = torch.randn(min(6400, L - r), L, generator=g, device=DEV)
    leaves = [k.requires_grad_(True), bias.requires_grad_(True)]
    out = flash_sparse_attn_func(q, k, v, None, bias, None, True)
    torch.full((L, L), float("nan"), dtype=torch.bfloat16, device=DEV)  # (what the gradient's memory may hold before)
    dbias = torch.autograd.grad(out, leaves, dout)[1][0, 0]
    k = k.detach()
    for r in range(0, L, 6400):
        rows = dbias[r:r + 6400]
        assert torch.isfinite(rows).all() and not torch.triu(rows, r + 1).any()
    rows = torch.tensor([0, 1, 31, 32, 200, 20000, L - 65, L - 17, L - 16, L - 1], device=DEV)
    s = q[0, rows, 0].float() @ k[0, :, 0].float().T * D ** -0.5 + bias.detach()[0, 0, rows].float()
    p = s.masked_fill(torch.arange(L, device=DEV)[None] > rows[:, None], float("-inf")).softmax(-1)
    dp = dout[0, rows, 0].float() @ v[0, :, 0].float().T
    assert_grad_close(dbias[rows], p * (dp - (p * dp).sum(-1, keepdim=True)), "dbias")
