"""Forward on grids that do not fill the chip (run with `-m gpu`): two groups of waves take the key tiles of a workgroup's
rows in turn up to as many 128-row blocks as compute units, and a chunk of queries against a long cache is cut into shares of
its keys.  Against the C oracle or the fp32 eager restatement (oracle/eager.py); out max-abs <= 2e-2, LSE within 1e-2, as
everywhere."""
import pytest
import torch

from oracle import c_oracle, eager
from _util import assert_grad_close, assert_out_close, make_inputs, set_compact

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _policy():
    yield
    set_compact(None)


def _forward(q, k, v, mask, bias, causal):
    from flash_sparse_attn import flash_sparse_attn_func

    with torch.no_grad():
        out, lse, _ = flash_sparse_attn_func(q, k, v, mask, bias, None, causal, None, None, True)
    assert torch.equal(out, flash_sparse_attn_func(q, k, v, mask, bias, None, causal).detach())  # (the other host path)
    return out, lse


@pytest.mark.parametrize("mode", ["0", "2"])  # tile skipping, compacted keys
@pytest.mark.parametrize("Lq,Lk,H,Hk,D,window,dtype", [
    (63, 129, 2, 1, 64, 129, torch.bfloat16),    # rows end inside the only workgroup; three tiles: the last turn has one
    (64, 256, 2, 2, 128, 64, torch.float16),     # one tile of kept keys: nothing for the second group
    (65, 300, 4, 2, 128, 65, torch.bfloat16),    # a workgroup of one row, a second tile of one key
    (16, 2000, 8, 2, 128, 700, torch.bfloat16),  # a chunk against a long cache
    (200, 190, 2, 1, 96, 130, torch.bfloat16),   # more rows than keys: rows that see nothing
    (129, 515, 4, 4, 8, 300, torch.float16),     # the smallest head dim
])
@pytest.mark.parametrize("causal", [True, False])
def test_two_key_groups(Lq, Lk, H, Hk, D, window, dtype, causal, mode):
    set_compact(mode)
    q, k, v, mask, bias = make_inputs(2, Lq, Lk, H, Hk, D, (2, Hk, 1, Lk), (2, Hk, 1, Lk), window, seed=Lq + Lk, dtype=dtype)
    out, lse = _forward(*[t.to(DEV) for t in (q, k, v, mask, bias)], causal)
    ro, rl = c_oracle.forward(q, k, v, mask, bias, D ** -0.5, causal)
    assert_out_close(out.cpu(), ro)
    fin = torch.isfinite(rl)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and (lse.cpu()[fin] - rl[fin]).abs().max() <= 1e-2


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Lq,H", [(1025, 16), (2048, 16), (2049, 16)])  # 144, 256 and 272 blocks of 128 rows
def test_either_side_of_a_block_per_compute_unit(Lq, H, D):
    for mask_form in ("column", None):
        q, k, v, mask, bias = make_inputs(1, Lq, 1100, H, 4, D, (1, 4, 1, 1100), (1, 4, 1, 1100), 500, seed=Lq + H)
        if mask_form is None:
            mask = bias = None
        d = [t.to(DEV) if t is not None else None for t in (q, k, v, mask, bias)]
        out, lse = _forward(*d, True)
        assert_out_close(out, eager.attention_forward(*d, None, True)[0])


@pytest.mark.parametrize("mode", ["0", "2"])
@pytest.mark.parametrize("dtype,jump", [(torch.bfloat16, 60.0), (torch.float16, 40.0)])
def test_scores_that_climb_after_the_first_tiles(dtype, jump, mode):
    """Beyond the range of the reference point that the first tile of a group sets: both groups take the safe path."""
    set_compact(mode)
    q, k, v, mask, bias = make_inputs(1, 70, 640, 4, 2, 128, (1, 2, 1, 640), (1, 2, 1, 640), 400, seed=9, dtype=dtype)
    bias = bias.clone()
    bias[..., 330:] += jump
    out, _ = _forward(*[t.to(DEV) for t in (q, k, v, mask, bias)], False)
    ro, _ = c_oracle.forward(q, k, v, mask, bias, 128 ** -0.5, False)
    assert_out_close(out.cpu(), ro)


def _close(got, ref):
    (out, lse), (ro, rl) = got, ref
    assert_out_close(out.cpu(), ro)
    fin = torch.isfinite(rl)
    assert torch.equal(torch.isfinite(lse.cpu()), fin) and (lse.cpu()[fin] - rl[fin]).abs().max() <= 1e-2


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,window,dtype", [
    (1, 2, 3072, 2, 1, 64, 3072, torch.bfloat16),      # the fewest rows and keys that are cut (three shares), all kept
    (1, 16, 8200, 8, 2, 128, 3000, torch.bfloat16),    # eight shares of uneven numbers of tiles
    (2, 100, 9001, 4, 2, 96, 70, torch.float16),       # two tiles of kept keys for eight shares: most are empty
    (1, 300, 4099, 4, 4, 128, 1, torch.bfloat16),      # a single kept key: rows above it see none
    (2, 129, 3100, 4, 2, 8, 1500, torch.float16),      # the smallest head dim; a block of one row
])
@pytest.mark.parametrize("causal", [True, False])
def test_shares_of_the_keys(B, Lq, Lk, H, Hk, D, window, dtype, causal):
    set_compact("2")
    q, k, v, mask, bias = make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, Hk, 1, Lk), window, seed=Lq + Lk, dtype=dtype)
    mask[B - 1, Hk - 1] &= B == 1  # a kv head without kept keys
    _close(_forward(*[t.to(DEV) for t in (q, k, v, mask, bias)], causal), c_oracle.forward(q, k, v, mask, bias, D ** -0.5, causal))


def test_shares_with_a_mask_row_per_query_head_and_scores_that_climb_in_one_share():
    set_compact("2")
    q, k, v, mask, bias = make_inputs(1, 40, 4096, 4, 2, 64, (1, 4, 1, 4096), (1, 4, 1, 4096), 1500, seed=3)
    bias = bias.clone()
    bias[..., 1200:] += 40.0
    _close(_forward(*[t.to(DEV) for t in (q, k, v, mask, bias)], False), c_oracle.forward(q, k, v, mask, bias, 0.125, False))


def test_a_workspace_without_room_for_the_shares():
    """The call is made with whole keys; and the entry point that allocates nothing takes what it took without shares."""
    from flash_sparse_attn import _cabi

    B, Lq, Lk, H, Hk, D = 1, 512, 4096, 8, 2, 128
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, Hk, 1, Lk), 1000, seed=5)]
    ref, _ = eager.attention_forward(q, k, v, mask, bias, None, True)
    out, lse = torch.empty_like(q), torch.empty(B, H, Lq, device=DEV)
    a = _cabi.FwdArgs()
    _cabi.fill_fwd(a, q, k, v, mask, bias, out, lse, D ** -0.5, True, 0.0)
    need = _cabi.lib.fdma_fwd_workspace_bytes(a)
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    results = []
    for entry, size in (("fdma_fwd", need), ("fdma_fwd", need - 4), ("fdma_fwd_noalloc", 0)):
        out.fill_(float("nan"))
        a.workspace, a.workspace_bytes = (ws.data_ptr(), size) if size else (None, 0)
        assert getattr(_cabi.lib, entry)(a, _cabi.current_stream(q.device)) == 0, _cabi.last_error()
        torch.cuda.synchronize()
        assert_out_close(out, ref)
        results.append(out.clone())
    assert need > _cabi.NOALLOC_SCRATCH_BYTES and torch.equal(results[1], results[2])
    a.workspace, a.workspace_bytes = ws.data_ptr(), 1 << 16
    assert _cabi.lib.fdma_fwd(a, _cabi.current_stream(q.device)) == -3


@pytest.mark.parametrize("per_query_head", [False, True])
def test_no_room_for_the_copies_of_a_long_key_axis(per_query_head):
    """Few rows against many keys are compacted under the library's own rule; the entry point that allocates nothing, whose
    scratch does not hold the copies, skips tiles and still takes the call."""
    from flash_sparse_attn import _cabi

    B, Lq, Lk, H, Hk, D = 1, 64, 16384, 8, 4, 128
    heads = H if per_query_head else Hk
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, D, (B, heads, 1, Lk), (B, heads, 1, Lk), 1000, seed=6)]
    out, lse = torch.full_like(q, float("nan")), torch.empty(B, H, Lq, device=DEV)
    a = _cabi.FwdArgs()
    _cabi.fill_fwd(a, q, k, v, mask, bias, out, lse, D ** -0.5, True, 0.0)
    assert _cabi.lib.fdma_fwd_workspace_bytes(a) > _cabi.NOALLOC_SCRATCH_BYTES
    assert _cabi.lib.fdma_fwd_noalloc(a, _cabi.current_stream(q.device)) == 0, _cabi.last_error()
    torch.cuda.synchronize()
    assert_out_close(out, eager.attention_forward(q, k, v, mask, bias, None, True)[0])


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,window,dtype", [
    (1, 100, 4096, 16, 16, 128, 1024, torch.bfloat16),  # 2 groups of dQ workgroups, 128 that sum
    (1, 2, 3072, 2, 1, 64, 3072, torch.bfloat16),       # the fewest rows and keys at d <= 64, all kept
    (1, 2, 2048, 2, 1, 128, 900, torch.bfloat16),       # ... and above
    (2, 33, 5000, 4, 2, 96, 900, torch.float16),
    (16, 2, 8192, 8, 8, 64, 1500, torch.bfloat16),      # 128 pairs: more units of keys than there are parts to be made
    (4, 64, 3100, 8, 8, 64, 300, torch.bfloat16),
    (1, 129, 6200, 6, 3, 256, 700, torch.float16),      # two row blocks, one of a single row
    (1, 300, 3073, 32, 8, 64, 2, torch.bfloat16),       # two kept keys (with one, dQ is zero and has no scale to compare against)
])
@pytest.mark.parametrize("causal", [True, False])
def test_gradients_of_few_rows_against_many_keys(B, Lq, Lk, H, Hk, D, window, dtype, causal):
    """Under the library's own rule these are compacted; the partial dK / dV are many for few dQ workgroups."""
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, Hk, 1, Lk), window, seed=Lq + Lk, dtype=dtype)]
    a = _cabi.FwdArgs()
    _cabi.fill_fwd(a, q, k, v, mask, bias, q, torch.empty(B, H, Lq, device=DEV), D ** -0.5, causal, 0.0)
    assert _cabi.lib.fdma_fwd_workspace_bytes(a) > 0  # (compacted)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    ref = eager.attention_forward_backward(q, k, v, mask, bias, None, causal, dout)
    runs = []
    for _ in range(2):
        leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v, bias)]
        out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3], None, causal)
        runs.append((out.detach(),) + torch.autograd.grad(out, leaves, dout))
    assert_out_close(runs[0][0], ref[0])
    for got, want, name in zip(runs[0][1:], ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got, want, name)
    for x, y in zip(*runs):
        assert torch.equal(x, y)


def test_gradients_of_few_rows_with_a_mask_row_per_query_head():
    """The forward compacts per query head; the backward skips tiles, group members together."""
    from flash_sparse_attn import flash_sparse_attn_func

    B, Lq, Lk, H, Hk, D = 1, 60, 3100, 4, 2, 64
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, D, (B, Hk, 1, Lk), (B, H, 1, Lk), 700, seed=8)]
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(q.dtype).to(DEV)
    ref = eager.attention_forward_backward(q, k, v, mask, bias, None, True, dout)
    leaves = [t.detach().clone().requires_grad_(True) for t in (q, k, v, bias)]
    out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3], None, True)
    assert_out_close(out, ref[0])
    for got, want, name in zip(torch.autograd.grad(out, leaves, dout), ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got, want, name)
