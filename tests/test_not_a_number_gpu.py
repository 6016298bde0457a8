"""Inputs that are no numbers (run with `-m gpu`): a NaN in a key or a query reaches every output row that sees it, and no other.

The kernels sum probabilities without a maximum, leave keys out by weights of zero and put partial results together by the
logarithms of their sums: in each of these a NaN could get lost.  Rows and heads that see none are compared with the same call
on inputs without it (out max-abs <= 2e-2, as everywhere)."""
import pytest
import torch

from _util import assert_out_close, make_inputs

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
