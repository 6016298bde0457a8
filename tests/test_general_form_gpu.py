"""Masks and biases with a row per query at the edges of the general kernels' tiles (run with `-m gpu`): head dims on both
sides of 64 and 128, key counts that end inside an 8-key chunk, a 32-key wave, a 128-key workgroup; query counts that end
inside a step and make one or many segments; biases and masks with one head, a head per kv head, a head per query head, or
none -- against the C oracle, forward and all gradients, and two runs bit for bit the same where nothing is atomic."""
import pytest
import torch

from oracle import c_oracle
from _util import assert_grad_close, assert_out_close

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # B, Lq, Lk, H, Hk, d, mask heads, bias heads, bias rows, causal
    (1, 70, 130, 4, 2, 128, 2, 2, 70, True),     # group sum, fused tile shared by the group
    (1, 70, 130, 4, 2, 128, 4, 2, 70, False),    # group sum, a mask per query head
    (2, 64, 128, 2, 2, 128, 1, 2, 64, True),     # whole tiles, no group
    (1, 33, 257, 8, 2, 96, 2, 8, 33, False),     # a head dim in between, bias per query head
    (1, 300, 9, 4, 1, 128, 1, 1, 300, False),    # one key block, two query segments
    (1, 513, 129, 2, 1, 128, 0, 1, 513, True),   # no mask
    (1, 200, 190, 4, 2, 128, 2, 2, 1, True),     # bias row shared by the queries: column sums over segments
    (1, 200, 190, 4, 2, 72, 4, 4, 1, False),
    (2, 100, 100, 4, 2, 128, 1, 1, 100, True),   # dBias shared by kv heads: fp32 atomics
    (1, 129, 70, 2, 2, 128, 2, 0, 0, True),      # no bias; rows without visible keys
    (1, 5, 7, 2, 1, 128, 1, 1, 5, False),        # rows shorter than a chunk
    (1, 131, 203, 4, 2, 64, 2, 2, 131, True),
    (2, 257, 77, 4, 4, 40, 1, 4, 257, False),
    (1, 131, 203, 2, 1, 256, 1, 1, 131, True),
    (1, 90, 61, 2, 2, 200, 2, 2, 1, False),
    (1, 2100, 40, 2, 1, 128, 1, 1, 2100, True),  # the most query segments, of unequal length; rows without visible keys
]


def _padded(t):
    """The same values as a view whose rows start at 16-byte boundaries; what lies behind a row is garbage."""
    n = t.shape[-1]
    big = torch.full((*t.shape[:-1], (n + 31) // 16 * 16), True if t.dtype == torch.bool else float("nan"), dtype=t.dtype, device=t.device)
    big[..., :n] = t
    return big[..., :n]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_general_form_vs_oracle(case, dtype):
    from flash_sparse_attn import flash_sparse_attn_func

    B, Lq, Lk, H, Hk, d, hm, hb, rows, causal = case
    g = torch.Generator().manual_seed(Lq * 1000 + Lk)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    q, k, v, dout = r(B, Lq, H, d), r(B, Lk, Hk, d), r(B, Lk, Hk, d), r(B, Lq, H, d)
    mask = torch.rand(B, hm, Lq, Lk, generator=g) < 0.5 if hm else None
    bias = r(B if (hb, Hk) != (1, 2) else 1, hb, rows, Lk) if hb else None
    if mask is None and rows == 1:
        pytest.skip("not the general form")
    ro, _ = c_oracle.forward(q, k, v, mask, bias, d ** -0.5, causal)
    ref = c_oracle.backward(q, k, v, dout, mask, bias, d ** -0.5, causal)
    runs = []
    for shape in (lambda t: t, _padded):
        leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)]
        bd = None if bias is None else shape(bias.to(DEV)).requires_grad_(True)
        out = flash_sparse_attn_func(*leaves, None if mask is None else shape(mask.to(DEV)), bd, None, causal)
        runs.append((out,) + torch.autograd.grad(out, leaves + ([bd] if bd is not None else []), dout.to(DEV)))
    assert_out_close(runs[0][0].cpu(), ro)
    for got, want, name in zip(runs[0][1:], ref, ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got.cpu(), want, name)
    atomics = bias is not None and ((bias.shape[0] == 1 and B > 1) or (hb == 1 and Hk > 1))
    for i, (a, b) in enumerate(zip(*runs)):  # odd rows and padded rows: other kernels, the same arithmetic
        if not (atomics and i == 4):
            assert torch.equal(a, b), ("out", "dq", "dk", "dv", "dbias")[i]


def _off_by_one(t):
    """The same values as a view whose rows start an element behind 16-byte boundaries, a row apart like whole chunks."""
    big = torch.full((*t.shape[:-1], t.shape[-1] + 16), True if t.dtype == torch.bool else float("nan"), dtype=t.dtype, device=t.device)
    big[..., 1:t.shape[-1] + 1] = t
    return big[..., 1:t.shape[-1] + 1]


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,hm,hb,rows,causal,one_batch", [
    (1, 70, 136, 8, 2, 128, 2, 2, 70, True, False),    # four heads of a group to a workgroup
    (2, 300, 264, 4, 1, 96, 1, 0, 0, False, False),    # ... no bias
    (1, 129, 200, 4, 2, 128, 2, 2, 129, True, False),  # two heads
    (1, 65, 128, 6, 3, 128, 3, 3, 1, False, False),    # ... a bias value per key
    (1, 131, 200, 4, 4, 64, 4, 4, 131, True, False),   # head dims up to 64, rows of half a piece: dK/dV with tiles through registers
    (1, 300, 72, 4, 2, 64, 2, 2, 300, False, False),
    (1, 150, 264, 4, 1, 40, 1, 1, 1, True, False),
    (2, 90, 136, 4, 2, 64, 2, 2, 90, True, True),      # one bias for the batch: dBias by fp32 atomics
    (2, 90, 136, 8, 2, 128, 2, 2, 90, False, True),
])
def test_rows_of_whole_chunks_at_any_address(B, Lq, Lk, H, Hk, d, hm, hb, rows, causal, one_batch):
    """Aligned rows of whole 8-key chunks have kernels of their own: the same results as rows that start anywhere."""
    from flash_sparse_attn import flash_sparse_attn_func

    print("chunks", B, Lq, Lk, H, Hk, d, hm, hb, rows, causal, one_batch, flush=True)
    g = torch.Generator().manual_seed(Lq * 1000 + Lk)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, k, v, dout = r(B, Lq, H, d), r(B, Lk, Hk, d), r(B, Lk, Hk, d), r(B, Lq, H, d)
    mask = torch.rand(B, hm, Lq, Lk, generator=g) < 0.5
    bias = r(1 if one_batch else B, hb, rows, Lk) if hb else None
    ref = (c_oracle.forward(q, k, v, mask, bias, d ** -0.5, causal)[0],) + tuple(c_oracle.backward(q, k, v, dout, mask, bias, d ** -0.5, causal))
    runs = []
    for shape in (lambda t: t, _off_by_one):
        leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)] + ([shape(bias.to(DEV)).requires_grad_(True)] if hb else [])
        out = flash_sparse_attn_func(*leaves[:3], shape(mask.to(DEV)), leaves[3] if hb else None, None, causal)
        runs.append((out,) + torch.autograd.grad(out, leaves, dout.to(DEV)))
    assert_out_close(runs[0][0].cpu(), ref[0])
    for got, want, name in zip(runs[0][1:], ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got.cpu(), want, name)
    for a, b, name in zip(*runs, ("out", "dq", "dk", "dv", "dbias")):
        assert (one_batch and name == "dbias") or torch.equal(a, b), name


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("causal", [False, True])
def test_last_rows_end_with_their_memory(d, causal):
    """Mask rows of 10 MiB in all, which the allocator has from the device as a piece of that size: the last chunk of the last row ends where
    the memory does.  The same results as rows with room behind them."""
    from flash_sparse_attn import flash_sparse_attn_func

    print("last rows", d, causal, flush=True)
    H, Lq, Lk = 16, 32768, 20
    g = torch.Generator(DEV).manual_seed(d)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV, dtype=torch.bfloat16)
    q, k, v, dout = r(1, Lq, H, d), r(1, Lk, H, d), r(1, Lk, H, d), r(1, Lq, H, d)
    keep = torch.rand(1, H, Lq, Lk, generator=g, device=DEV) < 0.5
    torch.cuda.empty_cache()
    mask, bias = keep.clone(), r(1, H, Lq, Lk)
    assert mask.numel() % (2 << 20) == 0
    runs = []
    for shape in (lambda t: t, _padded):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v, shape(bias))]
        out = flash_sparse_attn_func(*leaves[:3], shape(mask), leaves[3], None, causal)
        runs.append((out.detach(),) + torch.autograd.grad(out, leaves, dout))
    assert not runs[0][0].isnan().any()
    for a, b, name in zip(*runs, ("out", "dq", "dk", "dv", "dbias")):
        assert torch.equal(a, b), name
