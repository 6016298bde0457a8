"""dQ without mask and bias on few row blocks, whose key tiles two groups of waves take in turn: odd and even numbers of tiles, entries of
no tile, one tile and one key, rows that see nothing, head dims on both sides of 64, against the fp32 eager restatement; reruns bit for
bit the same."""
import pytest
import torch

from test_varlen_gpu import _cu, _make, _op, _reference
from _util import assert_grad_close, assert_out_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("lens_q,lens_k", [
    ([1025, 33, 1, 257], [1025, 33, 1, 257]),   # 33 tiles of 32; two; one; nine
    ([1, 130, 70], [1100, 0, 1057]),            # a single row, an entry without keys, rows far in front of their last key
    ([1300, 64, 31], [1088, 1, 2000]),          # rows that see nothing
])
@pytest.mark.parametrize("H,Hk,D", [(2, 1, 64), (3, 3, 40), (4, 2, 128), (2, 2, 72)])
@pytest.mark.parametrize("causal,dtype", [(True, torch.bfloat16), (False, torch.float16)])
def test_ragged(lens_q, lens_k, H, Hk, D, causal, dtype):
    print("groups", lens_q, lens_k, H, Hk, D, causal, flush=True)
    q, k, v, do = [t.to(DEV) for t in _make(lens_q, lens_k, H, Hk, D, dtype, seed=D)]
    ref = _reference(q, k, v, do, lens_q, lens_k, causal)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    runs = []
    for _ in range(2):
        out = _op()(*leaves, _cu(lens_q).to(DEV), _cu(lens_k).to(DEV), max(lens_q), max(lens_k), is_causal=causal)
        runs.append((out,) + torch.autograd.grad(out, leaves, do))
    assert_out_close(runs[0][0], ref[0])
    for got, want, name in zip(runs[0][1:], ref[2:], ("dq", "dk", "dv")):
        assert_grad_close(got, want, name)
    assert all(torch.equal(a, b) for a, b in zip(*runs))


@pytest.mark.parametrize("L,D", [(1055, 128), (1088, 64)])
def test_fixed_lengths(L, D):
    from flash_sparse_attn import flash_sparse_attn_func

    q, k, v, do = [t.to(DEV) for t in _make([L], [L], 2, 1, D, torch.bfloat16, seed=L)]
    ref = _reference(q, k, v, do, [L], [L], True)
    leaves = [t[None].requires_grad_(True) for t in (q, k, v)]
    out = flash_sparse_attn_func(*leaves, None, None, is_causal=True)
    for got, want, name in zip(torch.autograd.grad(out, leaves, do[None]), ref[2:], ("dq", "dk", "dv")):
        assert_grad_close(got[0], want, name)
