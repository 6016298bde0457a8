"""Splits of a single-token call: how many there are, and that their merge -- in the launch itself or in one of its own, up to 32
splits requested at a time, the workspace aligned for pairs of floats or not -- gives the same bits and the eager restatement's result."""
import pytest
import torch

from oracle import eager
from _util import assert_out_close, make_inputs

DEV = "cuda"


@pytest.mark.parametrize("pairs", [(1, 1), (1, 2), (1, 8), (2, 16), (8, 8), (64, 16)])
def test_no_split_is_empty(pairs):
    from flash_sparse_attn import _cabi

    B, Hk = pairs
    a = _cabi.FwdArgs()
    for Lk in [1, 255, 256, 257, 384, 385, 512, 513, 4093, 8191, 8193, 32768, 32769, 50001, 65536, 131071, 1 << 20]:
        a.batch, a.seqlen_q, a.seqlen_k, a.num_heads, a.num_heads_k, a.head_dim = B, 1, Lk, Hk, Hk, 64
        n, rest = divmod(_cabi.lib.fdma_fwd_workspace_bytes(a), (64 + 1) * 4 * B * Hk)
        assert rest == 0 and n != 1 and n <= 128
        if n == 0:  # one split: no partial results
            assert Lk <= 384 or B * Hk >= 256
            continue
        span = (-(-Lk // n) + 255) // 256 * 256
        assert (n - 1) * span < Lk <= n * span


@pytest.mark.parametrize("Lk", [32769, 40960, 50001, 65535, 65536, 65537, 131071, 131072])
def test_spans_of_long_caches(Lk):
    """One pair's splits beyond 32768 keys span 1280 keys whatever the length is a multiple of."""
    from flash_sparse_attn import _cabi

    a = _cabi.FwdArgs()
    a.batch, a.seqlen_q, a.seqlen_k, a.num_heads, a.num_heads_k, a.head_dim = 1, 1, Lk, 2, 1, 64
    a.mask = 256  # (there is one; sizes alone are looked at)
    assert _cabi.lib.fdma_fwd_workspace_bytes(a) == -(-Lk // 1280) * (64 + 1) * 4 * 2


@pytest.mark.parametrize("B,H,Hk,Lk,masked,unmasked", [
    (1, 4, 1, 32768, 32, 32),
    (1, 4, 1, 33001, 26, 43),   # spans of 768
    (1, 64, 2, 50001, 40, 49),  # 1024
    (2, 32, 1, 65536, 52, 64),
    (1, 4, 1, 65537, 52, 52),   # 1280
    (1, 4, 1, 131072, 103, 103),
    (1, 65, 1, 33001, 26, 26),  # many query heads: no more partial results than with a mask
    (3, 3, 1, 33001, 26, 26),   # three pairs
])
def test_splits_without_a_mask(B, H, Hk, Lk, masked, unmasked):
    """A call without a mask keeps every key: few pairs take shorter spans.  The counters do not depend on it."""
    from flash_sparse_attn import _cabi

    a = _cabi.FwdArgs()
    a.batch, a.seqlen_q, a.seqlen_k, a.num_heads, a.num_heads_k, a.head_dim = B, 1, Lk, H, Hk, 256
    counters = _cabi.lib.fdma_fwd_counter_bytes(a)
    assert _cabi.lib.fdma_fwd_workspace_bytes(a) == unmasked * (256 + 1) * 4 * B * H
    a.mask = 256
    assert _cabi.lib.fdma_fwd_workspace_bytes(a) == masked * (256 + 1) * 4 * B * H and _cabi.lib.fdma_fwd_counter_bytes(a) == counters


@pytest.mark.parametrize("B,Lk,Hk,D,splits", [
    (5, 20096, 8, 256, 6),    # 240 workgroups of the 256 that run at once above head dim 128
    (11, 41381, 16, 256, 1),
    (10, 9000, 8, 128, 3),
    (9, 1595, 16, 96, 1),
    (10, 16384, 8, 128, 3),   # 240 are enough ...
    (11, 16384, 8, 128, 5),   # ... 176 are not: two to a CU
    (11, 16383, 8, 128, 2),
    (8, 65536, 8, 128, 8),    # two to a CU, spans of 8192
    (8, 65535, 8, 128, 4),
    (12, 61888, 16, 64, 4),   # three
    (11, 8192, 8, 64, 5),
    (13, 28627, 8, 64, 4),    # two splits of 104 pairs to 127 would be one workgroup to most CUs, which hold three at d = 64
    (127, 8192, 1, 64, 4),
    (127, 8191, 1, 64, 2),
    (16, 28627, 8, 64, 2),    # (128 pairs: one to every CU)
    (13, 28627, 8, 72, 2),
    (300, 65536, 1, 128, 1),
    (2, 4093, 64, 256, 2),
])
def test_workgroups_that_run_at_once(B, Lk, Hk, D, splits):
    from flash_sparse_attn import _cabi

    a = _cabi.FwdArgs()
    a.batch, a.seqlen_q, a.seqlen_k, a.num_heads, a.num_heads_k, a.head_dim = B, 1, Lk, Hk, Hk, D
    a.mask = 256  # (there is one; sizes alone are looked at)
    assert _cabi.lib.fdma_fwd_workspace_bytes(a) == (splits * (D + 1) * 4 * B * Hk if splits > 1 else 0)
    assert (_cabi.lib.fdma_fwd_counter_bytes(a) > 0) == (splits > 1)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lk,H,Hk,D,kept,splits,dtype", [
    (1, 384, 2, 1, 128, 384, 1, torch.bfloat16),     # the longest call of one split
    (1, 385, 2, 1, 64, 200, 2, torch.float16),       # the shortest of two
    (3, 2049, 6, 2, 72, 700, 9, torch.bfloat16),     # a second group; three of four waves merge, a last pair inside the row
    (1, 33793, 3, 1, 136, 2500, 27, torch.float16),  # a second round of elements of 8
    (1, 8191, 4, 4, 8, 100, 32, torch.bfloat16),     # one request whole; most splits without a kept key in some rows
    (1, 41000, 3, 1, 136, 2500, 33, torch.float16),  # a second request of one split, in both rounds of elements
    (1, 66000, 2, 1, 256, 1500, 52, torch.bfloat16),
    (1, 81920, 2, 1, 256, 1500, 64, torch.bfloat16),  # the last lane of the first weights
    (1, 81921, 2, 1, 72, 900, 65, torch.float16),    # the first of the second
    (1, 131000, 1, 1, 64, 5, 103, torch.float16),    # nearly all of them empty
    (1, 163840, 1, 1, 64, 4000, 128, torch.bfloat16),  # as many as there are
])
def test_merge_of_splits(B, Lk, H, Hk, D, kept, splits, dtype):
    from flash_sparse_attn import _cabi
    from flash_sparse_attn.flash_sparse_attn_interface import _pad_key_dim

    print("splits", B, Lk, H, Hk, D, kept, dtype, flush=True)
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, 1, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, Hk, 1, Lk), kept, seed=Lk + D, dtype=dtype)]
    ref, ref_lse = eager.attention_forward(q, k, v, mask, bias, None, False)
    mask, bias = _pad_key_dim(mask, Lk, 16), _pad_key_dim(bias, Lk, 8)

    def call(offset, merged):
        out, lse = torch.full_like(q, float("nan")), torch.full((B, H, 1), float("nan"), dtype=torch.float32, device=DEV)
        a = _cabi.FwdArgs()
        _cabi.fill_fwd(a, q, k, v, mask, bias, out, lse, D ** -0.5, False, 0.0)
        need, counted = _cabi.lib.fdma_fwd_workspace_bytes(a), _cabi.lib.fdma_fwd_counter_bytes(a)
        assert need == (splits * (D + 1) * 4 * B * H if splits > 1 else 0)
        ws = torch.empty(need + 16, dtype=torch.uint8, device=DEV)
        counters = torch.zeros(counted // 4 + 1, dtype=torch.int32, device=DEV)
        a.workspace, a.workspace_bytes = ws.data_ptr() + offset, need
        if merged:
            a.counters, a.counters_bytes = counters.data_ptr(), counted
        assert _cabi.lib.fdma_fwd(a, _cabi.current_stream(q.device)) == 0, _cabi.last_error()
        torch.cuda.synchronize()
        assert int(counters.abs().max()) == 0
        return out, lse

    out, lse = call(0, True)
    assert_out_close(out, ref)
    assert torch.allclose(lse, ref_lse.reshape(lse.shape), atol=2e-3, rtol=1e-3)
    for offset, merged in ((0, False), (4, True), (4, False)):
        again, lse_again = call(offset, merged)
        assert torch.equal(again, out) and torch.equal(lse_again, lse)


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_without_a_mask_behind_a_call_with_one(native, monkeypatch):
    """Each of the two has splits and a workspace of its own: the same keys in another order of sums."""
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    print("no mask", native, flush=True)
    if not native:
        monkeypatch.setattr(_cabi, "host", _cabi._NoHost)
    q, k, v, _, bias = [t.to(DEV) for t in make_inputs(1, 1, 33003, 32, 1, 256, (1, 1, 1, 33003), (1, 1, 1, 33003), 64, seed=5, dtype=torch.float16)]
    ref, _ = eager.attention_forward(q, k, v, None, bias, None, False)
    for mask in (torch.ones(1, 1, 1, 33003, dtype=torch.bool, device=DEV), None):
        assert_out_close(flash_sparse_attn_func(q, k, v, mask, bias, is_causal=False), ref)
