"""Masks and biases that all queries share are taken at any address and row stride (run with `-m gpu`): the same values in
rows of an odd length and in padded, 16-byte aligned rows give the same results bit for bit; and decode from the mask
builder's list of kept keys against the C oracle.  K and V rows that lie on each other (stride 0): there is one row of memory, and nothing
behind it is read in the place of an absent mask or bias."""
import pytest
import torch

from oracle import c_oracle
from _util import assert_out_close, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _padded(t):
    """The same values as a view whose rows start at 16-byte boundaries; what lies behind a row is garbage."""
    n = t.shape[-1]
    fill = True if t.dtype == torch.bool else float("nan")
    big = torch.full((*t.shape[:-1], (n + 31) // 16 * 16), fill, dtype=t.dtype, device=t.device)
    big[..., :n] = t
    return big[..., :n]


def _case(B, Lq, Lk, H, Hk, d, keep, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    mask = torch.rand(B, Hk, 1, Lk, generator=g) < keep
    return r(B, Lq, H, d), r(B, Lk, Hk, d), r(B, Lk, Hk, d), mask, r(B, Hk, 1, Lk), r(B, Lq, H, d)


@pytest.mark.parametrize("mode", ["0", "2"])  # tile skipping, compaction
@pytest.mark.parametrize("Lq,Lk", [(1, 1), (1, 15), (1, 17), (1, 4097), (1, 20001), (40, 7), (33, 65), (130, 515), (64, 4099)])
def test_rows_of_any_length_and_address(Lq, Lk, mode):
    from flash_sparse_attn import flash_sparse_attn_func

    set_compact(mode)
    q, k, v, mask, bias, dout = [t.to(DEV) for t in _case(2, Lq, Lk, 4, 2, 64, 0.5, torch.bfloat16)]
    res = []
    for shape in (lambda t: t, _padded):
        leaves = [t.clone().requires_grad_(True) for t in (q, k, v)] + [shape(bias).requires_grad_(True)]
        out = flash_sparse_attn_func(*leaves[:3], shape(mask), leaves[3], None, Lq > 1)
        res.append([out] + (list(torch.autograd.grad(out, leaves, dout)) if Lq > 1 else []))
    assert not res[0][0].isnan().any()
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,Lk,H,Hk,d,window", [(1, 2049, 8, 2, 128, 512), (3, 5000, 4, 4, 64, 5000), (2, 300, 16, 2, 256, 7),
                                                (1, 9001, 4, 1, 96, 2048), (2, 70, 2, 2, 128, 0), (1, 40000, 8, 2, 128, 9000)])
@pytest.mark.parametrize("bias_heads", ["kv", "query"])
def test_decode_from_the_list_of_kept_keys(B, Lk, H, Hk, d, window, bias_heads):
    from flash_sparse_attn import flash_sparse_attn_func
    from flash_sparse_attn.utils.mask import create_mask, kept_keys_of

    q, k, v, _, bias, _ = _case(B, 1, Lk, H, Hk, d, 0.5, torch.bfloat16, seed=Lk)
    keep = create_mask(bias.to(DEV), None, B, 1, Lk, window, torch.finfo(torch.bfloat16).min)
    assert kept_keys_of(keep) is not None
    if bias_heads == "query":
        bias = torch.randn(B, H, 1, Lk, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    with torch.no_grad():
        out = flash_sparse_attn_func(q.to(DEV), k.to(DEV), v.to(DEV), keep, bias.to(DEV))
    ref, _ = c_oracle.forward(q, k, v, keep.cpu(), bias, d ** -0.5, False)
    assert_out_close(out.cpu(), ref)


@pytest.mark.parametrize("Lq,Lk,H,Hk,d", [(1, 3000, 8, 2, 128), (100, 3000, 4, 2, 64), (100, 3000, 4, 2, 128), (100, 3000, 4, 2, 256),
                                          (2100, 700, 32, 4, 64), (2100, 700, 32, 4, 128), (2100, 700, 32, 4, 256)])
@pytest.mark.parametrize("what", ["nothing", "mask", "bias"])
def test_one_row_of_keys_for_all(Lq, Lk, H, Hk, d, what):
    from flash_sparse_attn import flash_sparse_attn_func

    print("one row", Lq, Lk, H, Hk, d, what, flush=True)
    set_compact("0")
    q, k, v, mask, bias, dout = [t.to(DEV) for t in _case(1, Lq, Lk, H, Hk, d, 0.5, torch.bfloat16, seed=Lk)]
    mask, bias = mask if what == "mask" else None, bias if what == "bias" else None
    res = []
    for shape in (lambda t: t[:, :1].expand_as(t), lambda t: t[:, :1].expand_as(t).contiguous()):
        leaves = [t.detach().requires_grad_(True) for t in (q, shape(k), shape(v))]
        out = flash_sparse_attn_func(*leaves, mask, bias, None, Lq > 1)
        res.append((out.detach(),) + torch.autograd.grad(out, leaves, dout))
    assert leaves[1].stride(1) != 0 and not res[0][0].isnan().any()
    for a, b, name in zip(*res, ("out", "dq", "dk", "dv")):
        assert torch.equal(a, b), name
