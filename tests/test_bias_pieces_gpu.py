"""Bias producer forward: pieces of 128 columns, requested one ahead of the one that is worked on.  Waves with no, one, an odd and an
even number of pieces, a short last piece, short and batch-crossing token tiles, contiguous and gapped heads (the same bits).  Against
the closed form in 64 bits; the result is rounded to its 16-bit type once."""
import pytest
import torch
import torch.nn.functional as F

from flash_sparse_attn.utils.bias import dynamic_mask_bias
from _util import rel_err

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,Hk,d,dtype", [
    (1, 31, 1, 16, torch.bfloat16),      # one step in wave 0, nothing in the others
    (2, 45, 2, 72, torch.float16),       # a piece, a step, nothing, nothing
    (1, 33, 4, 128, torch.bfloat16),     # one piece each
    (3, 50, 5, 112, torch.bfloat16),     # 2, 2, a short one, none
    (1, 64, 8, 192, torch.float16),      # 3
    (2, 40, 8, 256, torch.bfloat16),     # 4
    (1, 70, 20, 256, torch.bfloat16),    # 10
    (2, 65600, 3, 112, torch.bfloat16),  # a wave has all columns: 2 and a short one
])
def test_pieces(B, L, Hk, d, dtype):
    print("pieces", B, L, Hk, d, dtype, flush=True)
    g = torch.Generator().manual_seed(L + d)
    v = torch.randn(B, L, Hk, d, generator=g).to(dtype).to(DEV)
    w = (torch.randn(Hk, Hk * d, generator=g) / (Hk * d) ** 0.5).to(dtype).to(DEV)
    a = torch.linspace(0.5, 1.5, Hk).to(dtype).to(DEV)
    ref = (a.double() * F.softplus(v.double().reshape(B, L, -1) @ w.double().t())).transpose(-1, -2).unsqueeze(-2)
    gaps = torch.full((B, L, Hk, d + 16), float("nan"), dtype=dtype, device=DEV)  # (what lies between the heads is not read)
    gaps[..., :d] = v
    with torch.no_grad():
        bias, strided = dynamic_mask_bias(v, w, a), dynamic_mask_bias(gaps[..., :d], w, a)
    torch.cuda.synchronize()
    assert rel_err(bias, ref) <= 2.0 ** -8
    assert torch.equal(bias, strided)


@pytest.mark.parametrize("Hk,d,fit", [(8, 64, 512), (8, 128, 256), (4, 256, 256), (9, 64, 256), (16, 48, 256), (16, 256, 256), (32, 64, 256), (1, 16, 512)])
def test_no_more_runs_than_the_device_holds_at_a_time(Hk, d, fit):
    from flash_sparse_attn import _cabi

    a = _cabi.DynBiasArgs()
    a.batch, a.num_heads_k, a.head_dim = 1, Hk, d
    stride = -(-(Hk * Hk * d + 2 * Hk) // 4) * 4 * 4
    for L in (1, 32 * fit - 1, 32 * fit, 32 * fit + 1, 9000, 16385, 20000, 33000, 65537, 131072, 1 << 20):
        a.seqlen_k = L
        runs, rest = divmod(_cabi.lib.fdma_dyn_bias_bwd_workspace_bytes(a), stride)
        assert rest == 0 and -(-L // 32) >= runs > 0 and runs <= fit and (runs > fit * 3 // 4 or L <= 64 * fit)


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,Hk,d", [
    (1, 16385, 1, 16),   # runs of 40 tokens, the last of 25
    (2, 8990, 3, 48),    # a run across the batch entries
    (1, 36900, 9, 64),   # 152 tokens: two passes of 64 and one of 24
    (1, 8193, 8, 128),   # 40 tokens, the last of 33
    (3, 3500, 17, 64),   # 48 tokens, across the batch entries
])
def test_gradients_of_long_runs(B, L, Hk, d):
    """The backward's runs of tokens are whole eights, not whole passes.  Sums over the tokens in fp32, results rounded to 16 bits once."""
    print("runs", B, L, Hk, d, flush=True)
    g = torch.Generator().manual_seed(L)
    v = torch.randn(B, L, Hk, d, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(Hk, Hk * d, generator=g) / (Hk * d) ** 0.5).to(torch.bfloat16).to(DEV)
    a = torch.linspace(0.5, 1.5, Hk).to(torch.bfloat16).to(DEV)
    dbias = torch.randn(B, Hk, 1, L, generator=g).to(torch.bfloat16).to(DEV)
    leaves = [t.requires_grad_(True) for t in (v, w, a)]
    got = torch.autograd.grad(dynamic_mask_bias(*leaves), leaves, dbias)
    v64, w64, a64 = wide = [t.detach().double().requires_grad_(True) for t in leaves]
    ref = (a64 * F.softplus(v64.reshape(B, L, -1) @ w64.t())).transpose(-1, -2).unsqueeze(-2)
    for x, y in zip(got, torch.autograd.grad(ref, wide, dbias.double())):
        assert rel_err(x, y) <= 2.0 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,Hk,d,dtype", [
    (1, 33, 8, 96, torch.bfloat16),     # two groups of 512 columns, the second short; a run of one token
    (2, 45, 16, 72, torch.float16),     # two of 1024, a run across the batch entries
    (1, 70, 20, 256, torch.bfloat16),   # ten of 512
    (1, 64, 32, 40, torch.bfloat16),    # every head of a wave's lanes
    (1, 4100, 16, 128, torch.float16),  # too many runs for the groups side by side
    (3, 1, 1, 16, torch.bfloat16),
])
def test_gradients_of_column_groups(B, L, Hk, d, dtype):
    """The backward's groups of columns run side by side where there are few runs of tokens; the per-head sums are taken once.  Two calls
    give the same bits; sums over the tokens in fp32, results rounded to 16 bits once."""
    print("groups", B, L, Hk, d, dtype, flush=True)
    g = torch.Generator().manual_seed(L + Hk)
    v = torch.randn(B, L, Hk, d, generator=g).to(dtype).to(DEV)
    w = (torch.randn(Hk, Hk * d, generator=g) / (Hk * d) ** 0.5).to(dtype).to(DEV)
    a = torch.linspace(0.5, 1.5, Hk).to(dtype).to(DEV)
    dbias = torch.randn(B, Hk, 1, L, generator=g).to(dtype).to(DEV)
    leaves = [t.requires_grad_(True) for t in (v, w, a)]
    got, again = [torch.autograd.grad(dynamic_mask_bias(*leaves), leaves, dbias) for _ in range(2)]
    v64, w64, a64 = wide = [t.detach().double().requires_grad_(True) for t in leaves]
    ref = (a64 * F.softplus(v64.reshape(B, L, -1) @ w64.t())).transpose(-1, -2).unsqueeze(-2)
    for x, y, z in zip(got, torch.autograd.grad(ref, wide, dbias.double()), again):
        assert rel_err(x, y) <= 2.0 ** -7 and torch.equal(x, z)


@pytest.mark.gpu
@pytest.mark.parametrize("B,L,Hk,d,dtype", [
    (1, 15, 8, 16, torch.bfloat16),      # a short tile, a full range of columns
    (1, 17, 9, 16, torch.float16),       # a tile and a token; a range and half a block of columns; rows of up to sixteen heads
    (2, 64, 1, 64, torch.bfloat16),      # a tile for every wave, half a range
    (1, 129, 17, 16, torch.float16),     # a run of one token; more than sixteen heads; two whole ranges and a short one
    (40, 3, 3, 80, torch.bfloat16),      # tiles that cross several batch entries
    (1, 16400, 8, 128, torch.bfloat16),  # four ranges to a workgroup
    (1, 9300, 16, 80, torch.float16),    # ten ranges: four, four and two
    (1, 4200, 32, 72, torch.bfloat16),   # 18 of eight, eight and two
])
def test_gradients_of_column_ranges(B, L, Hk, d, dtype):
    """The backward's products, tiles of 16 tokens by ranges of 128 columns.  Sums over the tokens in fp32, results rounded to 16 bits once."""
    print("ranges", B, L, Hk, d, dtype, flush=True)
    g = torch.Generator().manual_seed(L + Hk + d)
    v = torch.randn(B, L, Hk, d, generator=g).to(dtype).to(DEV)
    w = (torch.randn(Hk, Hk * d, generator=g) / (Hk * d) ** 0.5).to(dtype).to(DEV)
    a, pb = torch.linspace(0.5, 1.5, Hk).to(dtype).to(DEV), torch.linspace(-1, 1, Hk).to(dtype).to(DEV)
    dbias = torch.randn(B, Hk, 1, L, generator=g).to(dtype).to(DEV)
    leaves = [t.requires_grad_(True) for t in (v, w, a, pb)]
    got = torch.autograd.grad(dynamic_mask_bias(*leaves), leaves, dbias)
    wide = [t.detach().double().requires_grad_(True) for t in leaves]
    v64, w64, a64, pb64 = wide
    ref = (a64 * F.softplus(v64.reshape(B, L, -1) @ w64.t() + pb64)).transpose(-1, -2).unsqueeze(-2)
    for x, y in zip(got, torch.autograd.grad(ref, wide, dbias.double())):
        assert rel_err(x, y) <= 2.0 ** -7
