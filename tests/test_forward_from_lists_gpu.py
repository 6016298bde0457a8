"""Forward without a backward behind it, on handed-over lists of kept keys: the rows are read where they lie, without compacted copies.  The
same bits as the call that makes them (from the mask alone), at tiles that end anywhere; what dropped keys hold does not show."""
import pytest
import torch

from flash_sparse_attn import flash_sparse_attn_func
from flash_sparse_attn.utils import mask as M
from _util import rel_err, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("kept", [1, 31, 64, 65, 128, 129, 257, 500])
@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,mask_heads,bias_heads,causal,dtype", [
    (2, 300, 500, 4, 2, 128, 2, 2, True, torch.bfloat16),
    (1, 500, 500, 6, 2, 104, 1, 6, False, torch.float16),   # one mask row for all, a bias row per query head
    (3, 200, 501, 2, 1, 96, 1, 1, True, torch.bfloat16),    # rows of an odd length
    (1, 515, 515, 8, 8, 64, 8, 8, True, torch.float16),
    (2, 130, 700, 2, 2, 40, 2, 0, False, torch.bfloat16),   # no bias
    (1, 1900, 1900, 16, 8, 128, 8, 8, True, torch.bfloat16),  # 480 blocks of 64 rows: copies go to another kernel, see below
    (1, 1500, 1500, 16, 8, 72, 8, 8, True, torch.float16),
    (2, 1500, 1500, 16, 8, 64, 8, 8, True, torch.bfloat16),
    (5, 512, 512, 8, 4, 256, 4, 4, True, torch.bfloat16),   # 128-row blocks
    (4, 700, 500, 8, 2, 200, 2, 1, True, torch.float16),    # ... rows that see nothing
])
def test_same_bits(B, Lq, Lk, H, Hk, d, mask_heads, bias_heads, causal, dtype, kept):
    print("lists", B, Lq, Lk, H, Hk, d, mask_heads, bias_heads, causal, dtype, kept, flush=True)
    g = torch.Generator().manual_seed(Lq + d + kept)
    q, k, v = [torch.randn(B, n, h, d, generator=g).to(dtype).to(DEV) for n, h in ((Lq, H), (Lk, Hk), (Lk, Hk))]
    bias = torch.randn(B, bias_heads, 1, Lk, generator=g).to(dtype).to(DEV) if bias_heads else None
    scores = torch.randn(B, mask_heads, 1, Lk, generator=g).to(dtype).to(DEV)
    mask = M.topk_mask(scores, None, kept, torch.finfo(dtype).min)
    assert M.kept_keys_of(mask) is not None
    dropped = ~mask.expand(B, Hk, 1, Lk).transpose(1, 3).reshape(B, Lk, Hk, 1)
    k, v = k.masked_fill(dropped, float("nan")), v.masked_fill(dropped, float("inf"))
    set_compact("2")
    try:
        with torch.no_grad():
            copied = flash_sparse_attn_func(q, k, v, mask.clone(), bias, None, causal)
            torch.cuda.synchronize()
            before = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            direct = flash_sparse_attn_func(q, k, v, mask, bias, None, causal)
            peak = torch.cuda.max_memory_allocated() - before
    finally:
        set_compact("auto")
    assert torch.isfinite(direct.float()).all()
    if B * H * -(-Lq // 64) <= 256 or d > 128:
        assert torch.equal(direct, copied)
    else:  # (another order of summation: P rounded to 16 bits against another reference point, both results rounded once)
        assert rel_err(direct, copied) <= 2.0 * torch.finfo(dtype).eps
    # the output and the row statistics, in blocks of 512 bytes, and a mask or bias brought to whole chunks; no copies of K and V
    assert peak < direct.numel() * 2 + B * H * Lq * 4 + 4 * 1024 + (mask.numel() + (bias.numel() if bias_heads else 0)) * 8
