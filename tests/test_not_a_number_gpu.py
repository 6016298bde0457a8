"""Inputs that are no numbers (run with `-m gpu`): a NaN in a key or a query reaches every output row that sees it, and no other.

The kernels sum probabilities without a maximum, leave keys out by weights of zero and put partial results together by the
logarithms of their sums: in each of these a NaN could get lost.  Rows and heads that see none are compared with the same call
on inputs without it (out max-abs <= 2e-2, gradients within 5e-2 of their scale, as everywhere)."""
import pytest
import torch

from _util import GRAD_RTOL, assert_out_close, make_inputs, rel_err, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _call(a, entry, q, size):
    from flash_sparse_attn import _cabi

    ws = torch.zeros(max(size, 1), dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = (ws.data_ptr(), size) if size else (None, 0)
    assert getattr(_cabi.lib, entry)(a, _cabi.current_stream(q.device)) == 0, _cabi.last_error()
    torch.cuda.synchronize()


@pytest.mark.parametrize("where", ["key", "query"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_shares_of_the_keys(where, dtype):
    """Keys cut into shares against the same call with whole keys (a workspace without room for the shares): a NaN in one
    share, and in all of them, is in the result."""
    from flash_sparse_attn import _cabi

    B, Lq, Lk, H, Hk, D = 1, 16, 8200, 8, 2, 128
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, Hk, 1, Lk), 3000, seed=1, dtype=dtype)]
    if where == "key":
        mask[0, 0, 0, 5000] = True
        k[0, 5000, 0, 7] = float("nan")
    else:
        q[0, 3, 5, 7] = float("nan")
    hit = torch.zeros(Lq, H, dtype=torch.bool, device=DEV)
    if where == "key":
        hit[:, :H // Hk] = True
    else:
        hit[3, 5] = True
    results = []
    for whole in (False, True):
        out, lse = torch.zeros_like(q), torch.zeros(B, H, Lq, device=DEV)
        a = _cabi.FwdArgs()
        _cabi.fill_fwd(a, q, k, v, mask, bias, out, lse, D ** -0.5, True, 0.0)
        a.compact_mode = _cabi.COMPACT_ALWAYS
        need = _cabi.lib.fdma_fwd_workspace_bytes(a)
        _call(a, "fdma_fwd", q, need - 4 if whole else need)
        results.append((out, lse))
    (out, lse), (out_w, lse_w) = results
    assert not torch.equal(out, out_w)  # (two routes)
    assert torch.equal(torch.isnan(out).all(-1)[0], hit) and torch.equal(torch.isnan(out).any(-1)[0], hit)
    assert torch.equal(torch.isnan(out_w), torch.isnan(out))
    assert_out_close(out[0][~hit], out_w[0][~hit])
    seen = ~hit.T
    assert torch.equal(torch.isfinite(lse[0]), torch.isfinite(lse_w[0])) and (lse[0][seen] - lse_w[0][seen]).abs().max() <= 1e-2


# route: rows of mask and bias per query or shared; compaction policy; Lq, Lk, H, Hk, D, kept keys
ROUTES = {
    "decode": ("column", "0", 1, 3000, 8, 2, 128, 700),
    "decode, every split": ("column", "0", 1, 9000, 8, 2, 64, 4000),
    "key groups": ("column", "0", 70, 700, 4, 2, 128, 300),
    "key groups, compacted": ("column", "2", 70, 700, 4, 2, 128, 300),
    "one group": ("column", "0", 200, 400, 4, 2, 256, 200),
    "compacted, many rows": ("column", "2", 2100, 300, 16, 2, 64, 150),
    "tile images": ("column", "2", 300, 700, 4, 2, 128, 300),
    "no mask": ("none", "0", 130, 200, 4, 2, 128, 0),
    "per query": ("query", "0", 150, 260, 4, 2, 64, 130),
    "per query, segments": ("query", "0", 500, 260, 4, 2, 128, 130),
    "per query, a row per head": ("query", "0", 150, 264, 2, 2, 64, 130),
}


@pytest.mark.parametrize("where", ["key", "query"])
@pytest.mark.parametrize("route", ROUTES)
def test_every_row_that_sees_it_and_no_other(route, where, request):
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    rows, mode, Lq, Lk, H, Hk, D, window = ROUTES[route]
    set_compact(mode)
    before = _cabi.stream_min_items(1 if route == "tile images" else 0)
    request.addfinalizer(lambda: _cabi.stream_min_items(before))
    shape = None if rows == "none" else (1, Hk, Lq if rows == "query" else 1, Lk)
    clean = [t.to(DEV) if t is not None else None for t in make_inputs(1, Lq, Lk, H, Hk, D, shape, shape, window, seed=Lq + Lk)]
    at = Lk // 2 + 3
    if clean[3] is not None:
        clean[3][..., at] = True  # (every row sees the key)
    hit = torch.zeros(Lq, H, dtype=torch.bool, device=DEV)
    bad = list(clean)
    if where == "key":
        bad[1] = clean[1].clone()
        bad[1][0, at, 0, 5] = float("nan")
        hit[:, :H // Hk] = True
    else:
        bad[0] = clean[0].clone()
        bad[0][0, Lq // 2, 0, 5] = float("nan")
        hit[Lq // 2, 0] = True
    dout = torch.randn(clean[0].shape, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16).to(DEV)
    results = []
    for q, k, v, mask, bias in (clean, bad):
        leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v, bias) if t is not None]
        out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3] if bias is not None else None, None, False)
        results.append((out.detach(),) + torch.autograd.grad(out, leaves, dout))
    (o, dq, dk, dv, *_), (bo, bdq, bdk, bdv, *_) = results
    for got in (bo, bdq):
        nan = torch.isnan(got[0])
        assert torch.equal(nan.any(-1), hit) and torch.equal(nan.all(-1), hit)
    assert_out_close(bo[0][~hit], o[0][~hit])
    assert rel_err(bdq[0][~hit], dq[0][~hit]) <= GRAD_RTOL
    assert torch.isnan(bdk[0, at, 0]).all()
    for good, got in ((dk, bdk), (dv, bdv)):  # (the other kv heads)
        assert rel_err(got[:, :, 1:], good[:, :, 1:]) <= GRAD_RTOL


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("route", [r for r in ROUTES if ROUTES[r][0] != "none"])
def test_bias_of_dropped_keys(route, value, request):
    """What the mask drops may have any bias: the results are those of a zero there, to the bit."""
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    rows, mode, Lq, Lk, H, Hk, D, window = ROUTES[route]
    set_compact(mode)
    before = _cabi.stream_min_items(1 if route == "tile images" else 0)
    request.addfinalizer(lambda: _cabi.stream_min_items(before))
    shape = (1, Hk, Lq if rows == "query" else 1, Lk)
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(1, Lq, Lk, H, Hk, D, shape, shape, window, seed=Lq + Lk)]
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(7)).to(torch.bfloat16).to(DEV)
    results = []
    for fill in (0.0, value):
        leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v, torch.where(mask, bias, fill))]
        out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3], None, Lq > 1)
        results.append((out.detach(),) + torch.autograd.grad(out, leaves, dout))
    for a, b, name in zip(*results, ("out", "dq", "dk", "dv", "dbias")):
        assert torch.equal(a, b), name
    assert not results[1][4][~mask].any()
