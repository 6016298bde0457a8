"""Few query rows of the general form, whose key tiles are cut into shares: at the edges of tiles, of shares and of the head
dims that a kernel serves, against the C oracle and against the same call with whole keys (the shares' results are fp32, so the two
differ by the last rounding to 16 bits and, where probabilities are rounded against another reference point, by that)."""
import pytest
import torch

from oracle import c_oracle
from _util import assert_grad_close, assert_out_close

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [
    # B, Lq, Lk, H, Hk, d, mask heads, bias heads, causal, dQ in shares too
    (1, 512, 512, 2, 1, 64, 1, 1, True, False),      # two shares; the first rows see no tile of the second
    (1, 70, 1537, 2, 1, 64, 1, 1, False, True),      # a last tile of one key, alone behind its pair
    (1, 40, 1600, 4, 1, 64, 1, 0, True, True),       # four heads to a workgroup, no bias
    (2, 33, 1543, 4, 2, 128, 2, 2, True, True),      # two heads to a workgroup, two key halves; odd rows
    (1, 130, 1600, 1, 1, 96, 0, 1, False, False),    # no mask; dQ is made from dS
    (1, 577, 577, 2, 1, 256, 1, 1, True, True),      # tiles of 32 keys
    (1, 65, 520, 2, 2, 136, 2, 1, False, True),
    (1, 1700, 1100, 1, 1, 128, 1, 1, True, False),   # rows without a key
    (2, 66, 1601, 8, 2, 96, 2, 1, True, True),       # four heads to a workgroup, two key halves; odd rows
    (1, 100, 1600, 8, 2, 128, 2, 0, False, True),
]


def _many_heads(B, Lq, Lk, H, Hk, d, bias_heads):
    g = torch.Generator().manual_seed(Lq + Lk + d)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    mask = (torch.rand(B, Hk, Lq, Lk, generator=g) < 0.3).to(DEV)
    mask[:, :, Lq // 2, Lk // 3:] = False  # (a row that keeps nothing of the last share)
    return r(B, Lq, H, d), r(B, Lk, Hk, d), r(B, Lk, Hk, d), r(B, Lq, H, d), mask, r(B, bias_heads, Lq, Lk) if bias_heads else None


def _not_a_number_everywhere():
    """Memory that the allocator hands out next holds NaN."""
    held = [torch.full((n << 18,), float("nan"), device=DEV) for n in (1, 4, 16, 64, 256) for _ in range(4)]
    torch.cuda.synchronize()
    del held


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x) for x in c))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_shares_vs_oracle_and_whole(case, dtype, monkeypatch):
    from flash_sparse_attn import _cabi, flash_sparse_attn_func
    from flash_sparse_attn import flash_sparse_attn_interface as interface

    print(case, dtype, flush=True)
    B, Lq, Lk, H, Hk, d, hm, hb, causal, dq_too = case
    g = torch.Generator().manual_seed(Lq + Lk)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    q, k, v, dout = r(B, Lq, H, d), r(B, Lk, Hk, d), r(B, Lk, Hk, d), r(B, Lq, H, d)
    mask = torch.rand(B, hm, Lq, Lk, generator=g) < 0.3 if hm else None
    if mask is not None:
        mask[:, :, : Lq // 2, Lk // 3:] = False  # whole shares without a kept key
        mask[:, :, 3] = False                     # and a row without any
    bias = r(B, hb, Lq, Lk) if hb else None
    ro, rl = c_oracle.forward(q, k, v, mask, bias, d ** -0.5, causal)
    ref = c_oracle.backward(q, k, v, dout, mask, bias, d ** -0.5, causal)
    leaves = [t.to(DEV).requires_grad_(True) for t in (q, k, v)] + ([bias.to(DEV).requires_grad_(True)] if hb else [])
    asked = {"fdma_fwd_optional_bytes": [], "fdma_bwd_optional_bytes": []}

    def run(probs=True):
        got = flash_sparse_attn_func(*leaves[:3], None if mask is None else mask.to(DEV), leaves[3] if hb else None, None, causal, return_attn_probs=probs)
        out, lse = got[:2] if probs else (got, None)
        return (out, lse) + torch.autograd.grad(out, leaves, dout.to(DEV))

    native = run(probs=False)  # (the native path declines calls that want the LSE)
    assert native[0].grad_fn.name() == "FlashDMAttnFuncBackward"
    monkeypatch.setattr(_cabi, "host", _cabi._NoHost)  # (the Python path makes the calls)
    for name, seen in asked.items():
        fn = getattr(_cabi.lib, name)
        monkeypatch.setattr(_cabi.lib, name, lambda a, fn=fn, seen=seen: seen.append(fn(a)) or seen[-1])
    shares = run()
    assert asked["fdma_fwd_optional_bytes"][0] > 0 and (asked["fdma_bwd_optional_bytes"][0] > 0) == dq_too
    assert not any(int(c.abs().max()) for _, c in interface._decode_scratch.values())  # (arrival counters are left zero)
    with monkeypatch.context() as m:
        m.setattr(_cabi.lib, "fdma_fwd_counter_bytes", lambda a: 0)
        apart = run()  # (added up by a launch of its own)
    assert torch.equal(apart[0], shares[0]) and torch.equal(apart[1], shares[1])
    for name in asked:
        monkeypatch.setattr(_cabi.lib, name, lambda a: 0)
    whole = run()
    assert_out_close(shares[0].cpu(), ro)
    finite = torch.isfinite(rl)
    got = shares[1].cpu()
    assert torch.equal(torch.isfinite(got), finite) and (got[finite] - rl[finite]).abs().max() < 1e-2
    for x, want, name in zip(shares[2:], ref, ("dq", "dk", "dv", "dbias")):
        assert_grad_close(x.cpu(), want, name)
    eps = torch.finfo(dtype).eps
    for i, (a, b, c) in enumerate(zip(shares, whole, native)):
        assert i == 1 or torch.equal(a, c), i
        if i == 1:
            ok = (a == b) | ((a - b).abs() <= 1e-5 * (1 + b.abs()))
        else:  # (a probability is rounded to eps / 2 of itself against either reference point; sums of many of them, and what LSE and O carry on)
            ok = (a.float() - b.float()).abs() <= eps * (2 * b.float().abs() + b.float().abs().max())
        assert ok.all(), i


LINE = [
    (16, 2, 1473, 32, 8, 96, 0),     # 512 blocks of 256 rows: whole keys, by the kernels that have no shares
    (16, 16, 4096, 32, 8, 128, 0),
    (16, 32, 1473, 32, 8, 128, 1),   # a bias that kv heads share: dQ is not made from dS
    (32, 33, 1473, 16, 4, 96, 0),
    (32, 32, 4096, 16, 4, 128, 1),
    (15, 32, 1537, 32, 8, 128, 0),   # 480: two shares, four heads to a workgroup
    (15, 16, 4096, 32, 8, 96, 1),
    (15, 30, 1539, 32, 8, 72, 0),    # ... rows of an odd length
    (2, 65, 1600, 8, 2, 128, 1),     # more shares; a row block of one row
]


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,bias_heads", LINE)
@pytest.mark.parametrize("native", [True, False])
def test_gradients_where_the_kernel_changes(B, Lq, Lk, H, Hk, d, bias_heads, native, monkeypatch):
    """Either side of the line at which kernels of 256 query rows take a call: the gradients do not hold what lay in the scratch before."""
    from oracle import eager
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    print("line", B, Lq, Lk, H, Hk, d, bias_heads, native, flush=True)
    q, k, v, dout, mask, bias = _many_heads(B, Lq, Lk, H, Hk, d, bias_heads)
    ref = eager.attention_forward_backward(q, k, v, mask, bias, None, True, dout)
    if not native:
        monkeypatch.setattr(_cabi, "host", _cabi._NoHost)
    leaves = [t.requires_grad_(True) for t in (q, k, v) + ((bias,) if bias_heads else ())]
    out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3] if bias_heads else None, None, True)
    _not_a_number_everywhere()
    grads = torch.autograd.grad(out, leaves, dout)
    for x, want, name in zip(grads, ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(x, want, name)


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,bias_heads", LINE + [(16, 32, 705, 32, 8, 128, 0), (15, 32, 769, 32, 8, 128, 1)])
def test_forward_where_the_kernel_changes(B, Lq, Lk, H, Hk, d, bias_heads, monkeypatch):
    """... nor does the forward, with arrival counters or without."""
    from oracle import eager
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    print("line, forward", B, Lq, Lk, H, Hk, d, bias_heads, flush=True)
    q, k, v, _, mask, bias = _many_heads(B, Lq, Lk, H, Hk, d, bias_heads)
    ref, ref_lse = eager.attention_forward(q, k, v, mask, bias, None, True)

    def call():
        _not_a_number_everywhere()
        with torch.no_grad():
            return flash_sparse_attn_func(q, k, v, mask, bias, None, True, return_attn_probs=True)[:2]

    runs = [call()]
    for name in ("fdma_fwd_counter_bytes", "fdma_fwd_optional_bytes"):  # (added up by a launch of its own; whole keys)
        monkeypatch.setattr(_cabi.lib, name, lambda a: 0)
        runs.append(call())
    for out, lse in runs:
        assert_out_close(out, ref)
        assert torch.allclose(lse, ref_lse.reshape(lse.shape), atol=2e-3, rtol=1e-3)


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,kept", [
    (1, 70, 5003, 4, 2, 128, 3000),   # four shares; a row block of six rows
    (2, 16, 8200, 2, 1, 64, 8200),    # eight
    (1, 130, 4100, 3, 3, 72, 900),    # offered four, one taken: the result is written whole
    (1, 64, 6000, 2, 1, 96, 1100),    # two of five
])
def test_few_rows_against_many_keys(B, Lq, Lk, H, Hk, d, kept, monkeypatch):
    """The column form's shares: added up by the last workgroup of a row block or by a launch, the same bits."""
    from oracle import eager
    from _util import make_inputs
    from flash_sparse_attn import _cabi, flash_sparse_attn_func
    from flash_sparse_attn import flash_sparse_attn_interface as interface

    print("few rows", B, Lq, Lk, H, Hk, d, kept, flush=True)
    q, k, v, mask, bias = [t.to(DEV) for t in make_inputs(B, Lq, Lk, H, Hk, d, (B, Hk, 1, Lk), (B, Hk, 1, Lk), kept, seed=Lk)]
    ref, ref_lse = eager.attention_forward(q, k, v, mask, bias, None, True)
    call = lambda: flash_sparse_attn_func(q, k, v, mask, bias, None, True, return_attn_probs=True)[:2]
    with torch.no_grad():
        native = flash_sparse_attn_func(q, k, v, mask, bias, None, True)
        monkeypatch.setattr(_cabi, "host", _cabi._NoHost)
        asked = []
        fn = _cabi.lib.fdma_fwd_counter_bytes
        monkeypatch.setattr(_cabi.lib, "fdma_fwd_counter_bytes", lambda a: asked.append(fn(a)) or asked[-1])
        out, lse = call()
        assert asked[0] > 0 and not any(int(c.abs().max()) for _, c in interface._decode_scratch.values())
        monkeypatch.setattr(_cabi.lib, "fdma_fwd_counter_bytes", lambda a: 0)
        apart, lse_apart = call()
    assert torch.equal(out, native) and torch.equal(out, apart) and torch.equal(lse, lse_apart)
    assert_out_close(out, ref)
    assert torch.allclose(lse, ref_lse.reshape(lse.shape), atol=2e-3, rtol=1e-3)
