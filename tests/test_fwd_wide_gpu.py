"""The forward with key groups by direct loads (fdma_fwd_wide.hip): head dims above 128, and below on small grids.  Sizes at the edges of its row blocks (64 / 128 rows) and tiles (128 / 64 keys), key groups without a
kept key, scores that climb from tile to tile (the reference point moves in every one), empty rows."""
import pytest
import torch

from oracle import eager
from _util import assert_out_close, make_inputs, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(q, k, v, mask, bias, causal):
    from flash_sparse_attn import flash_sparse_attn_func

    q, k, v, mask, bias = [t if t is None else t.to(DEV) for t in (q, k, v, mask, bias)]
    out, lse, _ = flash_sparse_attn_func(q, k, v, mask, bias, None, causal, return_attn_probs=True)
    ro, rl = eager.attention_forward(q, k, v, mask, bias, None, causal)
    assert_out_close(out, ro)
    assert torch.equal(torch.isinf(lse), torch.isinf(rl))
    fin = torch.isfinite(rl)
    # the scaled Q is rounded to 16 bits: 2^-9 (bf16) of a score's terms, whose sum over d has a standard deviation of one
    assert (lse[fin] - rl[fin]).abs().max().item() <= 3e-2 * max(1.0, rl[fin].abs().max().item() / 8)


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,causal,dtype", [
    (1, 64, 129, 2, 1, 128, True, torch.bfloat16),
    (1, 65, 257, 4, 2, 128, False, torch.float16),
    (2, 63, 383, 4, 4, 72, True, torch.bfloat16),
    (1, 127, 130, 2, 1, 128, True, torch.float16),
    (1, 3, 1000, 8, 2, 104, True, torch.bfloat16),
    (1, 300, 140, 2, 2, 128, True, torch.bfloat16),     # rows without a key
    (1, 4100, 4100, 2, 1, 128, True, torch.bfloat16),
    (1, 64, 129, 2, 1, 64, True, torch.bfloat16),
    (1, 65, 257, 4, 2, 64, False, torch.float16),
    (3, 127, 128, 2, 2, 40, True, torch.bfloat16),
    (1, 2, 5000, 8, 2, 64, True, torch.float16),
    (1, 300, 140, 2, 2, 64, True, torch.bfloat16),      # rows without a key
    (1, 1, 64, 2, 1, 256, False, torch.bfloat16),
    (1, 128, 65, 2, 1, 256, True, torch.float16),
    (2, 129, 127, 4, 2, 136, True, torch.bfloat16),
    (1, 33, 63, 2, 2, 200, False, torch.bfloat16),
    (1, 700, 450, 2, 1, 256, True, torch.float16),
    (1, 65, 257, 2, 1, 256, False, torch.bfloat16),
    (1, 700, 450, 30, 15, 256, True, torch.float16),    # above head dim 128: more 64-row blocks than CUs, 128-row ones
    (2, 129, 127, 60, 20, 136, True, torch.bfloat16),
    (4, 65, 65, 36, 9, 200, False, torch.bfloat16),
])
@pytest.mark.parametrize("mode", ["0", "2"])
def test_edges(B, Lq, Lk, H, Hk, D, causal, dtype, mode):
    print(B, Lq, Lk, H, Hk, D, causal, dtype, mode, flush=True)
    set_compact(mode)
    q, k, v, mask, bias = make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, Hk, 1, Lk), max(1, Lk // 2), seed=Lq + Lk, dtype=dtype)
    _check(q, k, v, mask, bias, causal)


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("mode", ["0", "2"])
def test_climbing_scores_and_empty_groups(D, mode):
    set_compact(mode)
    B, Lq, Lk, H, Hk = 1, 100, 900, 2, 1
    q, k, v, mask, _ = make_inputs(B, Lq, Lk, H, Hk, D, None, (B, Hk, 1, Lk), Lk, seed=3)
    bias = (torch.arange(Lk).float() * 0.25).view(1, 1, 1, Lk).to(torch.bfloat16)  # (32 keys: 8 in log units, 11 in exponents of two)
    mask[..., 32:96] = False    # whole key groups of a tile
    mask[..., 256:640] = False  # whole tiles
    _check(q, k, v, mask, bias, False)
    _check(q, k, v, mask, bias, True)
    mask[:] = False
    mask[..., 77] = True
    _check(q, k, v, mask, bias, False)


@pytest.mark.parametrize("lens,H,Hk,D", [
    ([1, 200, 64, 65, 300], 4, 2, 128),
    ([1, 200, 64, 65, 300], 4, 2, 64),
    ([2500, 1800], 8, 4, 64),
    ([1100, 300, 5, 790], 13, 13, 96),  # an entry of half of the rows: up to two blocks of 64 rows per CU (481 here) ...
    ([7, 1300, 40], 32, 8, 64),         # ... or three (736)
    ([1024, 1023], 14, 14, 128),        # (476)
])
def test_ragged(lens, H, Hk, D):
    from flash_sparse_attn import flash_sparse_attn_varlen_func

    g = torch.Generator().manual_seed(5)
    q = torch.randn(sum(lens), H, D, generator=g).to(torch.bfloat16).to(DEV)
    k, v = [torch.randn(sum(lens), Hk, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2)]
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    out = flash_sparse_attn_varlen_func(q, k, v, cu, cu, max(lens), max(lens), is_causal=True)
    at = 0
    for n in lens:
        s = slice(at, at + n)
        assert_out_close(out[s], eager.attention_forward(q[None, s], k[None, s], v[None, s], None, None, None, True)[0][0])
        at += n


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lens,H,Hk,D", [
    ([1, 200, 64, 65, 300], 4, 2, 136),    # 64-row blocks with one stage of K and V
    ([1, 200, 64, 65, 300], 4, 2, 256),
    ([129, 1, 700, 127, 900], 16, 8, 256),  # more of them than CUs: 128-row ones with two stages
])
def test_ragged_above_head_dim_128(lens, H, Hk, D, causal):
    from flash_sparse_attn import flash_sparse_attn_varlen_func

    print(lens, H, Hk, D, causal, flush=True)
    g = torch.Generator().manual_seed(6)
    q = torch.randn(sum(lens), H, D, generator=g).to(torch.bfloat16).to(DEV)
    k, v = [torch.randn(sum(lens), Hk, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2)]
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    out = flash_sparse_attn_varlen_func(q, k, v, cu, cu, max(lens), max(lens), is_causal=causal)
    at = 0
    for n in lens:
        s = slice(at, at + n)
        assert_out_close(out[s], eager.attention_forward(q[None, s], k[None, s], v[None, s], None, None, None, causal)[0][0])
        at += n


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,lists", [
    (2, 131, 300, 4, 2, 64, False),
    (1, 3, 300, 4, 2, 96, False),
    (2, 70, 300, 4, 2, 128, True),
    (1, 200, 300, 4, 2, 256, False),
    (5, 512, 512, 8, 4, 256, True),   # 128-row blocks
])
def test_query_rows_in_descending_order(B, Lq, Lk, H, Hk, D, lists):
    """A negative row stride of Q (plain C callers): the same bits as from rows in ascending order."""
    from flash_sparse_attn import _cabi
    from flash_sparse_attn.utils import mask as M

    print("descending", B, Lq, Lk, H, Hk, D, lists, flush=True)
    q, k, v, _, bias = [t if t is None else t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), seed=Lq + D)]
    mask = M.topk_mask(bias, None, Lk // 3, torch.finfo(q.dtype).min) if lists else None
    idx, cnt, count, ld = M.kept_keys_of(mask) if lists else (None,) * 4
    rows = [q, q.flip(1).contiguous()]
    results = []
    set_compact("2" if lists else "0")
    for i in range(2):
        out, lse = torch.full_like(q, float("nan")), torch.full((B, H, Lq), float("nan"), dtype=torch.float32, device=DEV)
        a = _cabi.FwdArgs()
        _cabi.fill_fwd(a, q, k, v, mask, bias, out, lse, D ** -0.5, True, 0.0, kept=(idx, cnt, count, ld) if lists else None)
        if lists:
            assert _cabi.lib.fdma_fwd_takes_lists(a)
        if i:
            a.q, a.q_strides[1] = rows[1].data_ptr() + (Lq - 1) * q.stride(1) * 2, -q.stride(1)
        assert _cabi.lib.fdma_fwd(a, _cabi.current_stream(q.device)) == 0, _cabi.last_error()
        torch.cuda.synchronize()
        results.append((out, lse))
    for x, y in zip(*results):
        assert torch.equal(x, y)
    assert torch.isfinite(results[0][0].float()).all()
