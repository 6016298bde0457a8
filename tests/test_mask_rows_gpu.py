"""The keep-mask builder at the edges of its register form (run with `-m gpu`): row lengths around the chunk, the workgroup
sizes and the largest row, few and many rows, rows full of ties, against torch on the same rows; list and bit row against
the mask they belong to."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("L", [1, 7, 8, 9, 255, 2047, 2048, 2049, 4093, 4097, 8192, 8193, 16385, 40001, 65536, 65537])
@pytest.mark.parametrize("rows,heads,padded,ties", [(1, 3, True, False), (1, 2, False, True), (600, 2, False, True)])
def test_topk_rows(L, rows, heads, padded, ties):
    from flash_sparse_attn.utils.mask import create_mask, kept_keys_of, mask_bits_of

    if rows * L > 6e6:
        pytest.skip("as many rows at the shorter lengths")
    g = torch.Generator(device=DEV).manual_seed(L)
    dtype = torch.bfloat16 if ties else torch.float16
    bias = torch.randn(2, heads, rows, L, generator=g, device=DEV).to(dtype)
    if ties:
        # (+ 0: no negative zeros -- the builder orders them below zero where torch's sort calls them equal, and a tie's
        # choice is the builder's: utils/mask.py)
        bias = (bias * 2).round() / 2 + 0.0
    pad = torch.rand(2, L, generator=g, device=DEV) < 0.8 if padded else None
    window = max(1, L // 3)
    keep = create_mask(bias, pad, 2, rows, L, window, torch.finfo(dtype).min)
    # stable descending order: among equal values the lowest columns come first
    x = bias.float() if pad is None else bias.float().masked_fill(~pad[:, None, None, :], torch.finfo(dtype).min)
    order = torch.sort(x, dim=-1, descending=True, stable=True).indices[..., :window]
    want = torch.zeros_like(keep).scatter_(-1, order, True) & (x != torch.finfo(dtype).min)
    assert torch.equal(keep, want)
    if rows == 1:
        idx, cnt, count, _ = kept_keys_of(keep)
        m = keep.reshape(-1, L)
        assert torch.equal(count.long(), m.sum(-1)) and torch.equal(cnt[:, :L].long(), m.cumsum(-1))
        for i in range(m.shape[0]):
            assert torch.equal(idx[i, : count[i]].long(), m[i].nonzero().flatten())
    else:
        bits = mask_bits_of(keep)[..., : (L + 7) // 8]
        cols = torch.arange(L, device=DEV)
        assert torch.equal((bits[..., cols // 8] >> (cols % 8)) & 1, keep.to(torch.uint8))
