"""dK / dV of key blocks that are cut into parts (the column form on the original key axis, and ragged batches): few heads and
short rows, at the edges of blocks, heads and parts.  Against the fp32 eager restatement, with and without the room for parts (the
sums of a part are fp32, so the two differ by the last rounding to 16 bits alone)."""
import pytest
import torch

from oracle import eager
from _util import assert_grad_close, make_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _whole(monkeypatch, grads):
    """grads() once with the room for parts -- which the call asks for -- and once without."""
    from flash_sparse_attn import _cabi

    asked = []

    def counted(fn):
        return lambda a: asked.append(fn(a)) or asked[-1]

    monkeypatch.setattr(_cabi, "host", _cabi._NoHost)  # (the Python path makes the calls)
    for name in ("fdma_bwd_optional_bytes", "fdma_varlen_bwd_optional_bytes"):
        monkeypatch.setattr(_cabi.lib, name, counted(getattr(_cabi.lib, name)))
    again = grads()
    assert len(asked) == 1 and asked[0] > 0
    for name in ("fdma_bwd_optional_bytes", "fdma_varlen_bwd_optional_bytes"):
        monkeypatch.setattr(_cabi.lib, name, lambda a: 0)
    return again, grads()


def _close(parts, whole, names):
    for a, b, name in zip(parts, whole, names):
        # one unit in the last place of the 16-bit results where sums of another order fall on the other side of a tie,
        # and of what cancels the rounding of fp32 sums (2^-24 of the terms, a few hundred of them at most)
        eps = torch.finfo(a.dtype).eps
        err = (a.float() - b.float()).abs()
        assert (err <= eps * b.float().abs() + 2e-5 * b.float().abs().max()).all(), name


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,Hb,causal,dtype", [
    (1, 672, 672, 16, 4, 128, 4, True, torch.bfloat16),
    (1, 563, 563, 8, 2, 128, 8, True, torch.float16),     # a bias column per query head: parts end inside a head's steps
    (2, 500, 1100, 4, 1, 128, 1, False, torch.bfloat16),
    (2, 300, 300, 12, 4, 96, 1, True, torch.bfloat16),     # one bias row for all kv heads: added up by atomics
    (1, 1100, 513, 6, 2, 64, 2, True, torch.bfloat16),    # rows without a key, a last block of one key
    (1, 129, 900, 12, 1, 64, 12, False, torch.float16),
    (1, 417, 417, 3, 1, 128, 0, True, torch.bfloat16),    # no bias; 14 steps of 32 rows, one row in the last
    (1, 1, 640, 24, 1, 128, 1, True, torch.bfloat16),     # a step per head
    (2, 256, 256, 12, 4, 256, 4, True, torch.bfloat16),
    (1, 700, 260, 4, 2, 200, 2, False, torch.float16),
])
def test_column_form(B, Lq, Lk, H, Hk, D, Hb, causal, dtype, monkeypatch):
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    print("column", B, Lq, Lk, H, Hk, D, Hb, causal, dtype, flush=True)
    _cabi.set_compact_mode(_cabi.COMPACT_NEVER)
    q, k, v, mask, bias = make_inputs(B, Lq, Lk, H, Hk, D, (B, Hb, 1, Lk) if Hb else None, (B, Hk, 1, Lk), Lk * 2 // 3, seed=Lq + D, dtype=dtype)
    q, k, v, mask = [t.to(DEV) for t in (q, k, v, mask)]
    leaves = [t.requires_grad_(True) for t in (q, k, v)] + ([bias.to(DEV).requires_grad_(True)] if Hb else [])
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    ref = eager.attention_forward_backward(q.detach(), k.detach(), v.detach(), mask, leaves[3].detach() if Hb else None, None, causal, dout)

    def grads():
        out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3] if Hb else None, None, causal)
        return torch.autograd.grad(out, leaves, dout)

    names = ("dq", "dk", "dv", "dbias")
    parts = grads()
    for got, want, name in zip(parts, ref[1:], names):
        assert_grad_close(got, want, name)
    again, whole = _whole(monkeypatch, grads)
    if Hb != 1 or Hk == 1:  # (atomics add in any order)
        for x, y in zip(parts, again):
            assert torch.equal(x, y)
    _close(parts, whole, names)


@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,causal,dtype", [
    ([300, 1, 700, 128, 45], None, 4, 1, 128, True, torch.bfloat16),
    ([1000, 2], None, 8, 4, 64, True, torch.float16),
    ([0, 513, 64], [100, 700, 0], 6, 3, 96, False, torch.bfloat16),
    ([257, 500, 1], [900, 129, 128], 4, 2, 128, True, torch.float16),
    ([300, 1, 700, 33], None, 4, 1, 256, True, torch.bfloat16),
    ([129, 500], [260, 90], 4, 2, 136, False, torch.float16),
    ([40] * 70 + [900], None, 2, 1, 128, True, torch.bfloat16),   # more entries than a wave has lanes
    ([300, 1, 1500, 33], None, 64, 16, 64, True, torch.float16),     # two and three lists of units per XCD
    ([33, 1500, 1, 300], [300, 1100, 129, 60], 48, 12, 128, False, torch.bfloat16),
])
def test_ragged(lens_q, lens_k, H, Hk, D, causal, dtype, monkeypatch):
    from flash_sparse_attn import flash_sparse_attn_varlen_func

    lens_k = lens_q if lens_k is None else lens_k
    print("ragged", lens_q[:6], lens_k[:6], H, Hk, D, causal, dtype, flush=True)
    g = torch.Generator().manual_seed(len(lens_q) + D)
    q = torch.randn(sum(lens_q), H, D, generator=g).to(dtype).to(DEV).requires_grad_(True)
    k, v = [torch.randn(sum(lens_k), Hk, D, generator=g).to(dtype).to(DEV).requires_grad_(True) for _ in range(2)]
    dout = torch.randn(q.shape, generator=g).to(dtype).to(DEV)
    cu = [torch.tensor([0] + lens, device=DEV).cumsum(0).int() for lens in (lens_q, lens_k)]

    def grads():
        out = flash_sparse_attn_varlen_func(q, k, v, cu[0], cu[1], max(lens_q), max(lens_k), is_causal=causal)
        return torch.autograd.grad(out, (q, k, v), dout)

    parts = grads()
    ref = [torch.zeros_like(t, dtype=torch.float32) for t in (q, k, v)]
    q0 = k0 = 0
    for lq, lk in zip(lens_q, lens_k):
        if lq and lk:
            qs, ks = slice(q0, q0 + lq), slice(k0, k0 + lk)
            r = eager.attention_forward_backward(q.detach()[None, qs], k.detach()[None, ks], v.detach()[None, ks], None, None, None, causal, dout=dout[None, qs])
            ref[0][qs], ref[1][ks], ref[2][ks] = r[1][0], r[2][0], r[3][0]
        q0, k0 = q0 + lq, k0 + lk
    names = ("dq", "dk", "dv")
    for got, want, name in zip(parts, ref, names):
        assert_grad_close(got, want, name)
    again, whole = _whole(monkeypatch, grads)
    for x, y in zip(parts, again):
        assert torch.equal(x, y)
    _close(parts, whole, names)


@pytest.mark.parametrize("B,Lq,Lk,H,Hk,D,Hb,causal,dtype", [
    (1, 300, 700, 4, 2, 256, 2, True, torch.bfloat16),     # few units: cut by heads and segments
    (2, 65, 500, 2, 2, 136, 1, False, torch.float16),
    (1, 513, 513, 6, 2, 200, 6, True, torch.bfloat16),
    (1, 600, 140, 2, 1, 256, 0, True, torch.float16),      # rows without a key
    (4, 1100, 1400, 40, 20, 256, 20, True, torch.bfloat16),  # enough units of kept keys: none is cut
])
def test_compacted_above_128(B, Lq, Lk, H, Hk, D, Hb, causal, dtype):
    """The wave pairs of head dims above 128 on compacted keys."""
    from flash_sparse_attn import _cabi, flash_sparse_attn_func

    print("compacted", B, Lq, Lk, H, Hk, D, Hb, causal, dtype, flush=True)
    _cabi.set_compact_mode(_cabi.COMPACT_ALWAYS)
    q, k, v, mask, bias = make_inputs(B, Lq, Lk, H, Hk, D, (B, Hb, 1, Lk) if Hb else None, (B, Hk, 1, Lk), Lk // 2, seed=Lq + D, dtype=dtype)
    q, k, v, mask = [t.to(DEV) for t in (q, k, v, mask)]
    leaves = [t.requires_grad_(True) for t in (q, k, v)] + ([bias.to(DEV).requires_grad_(True)] if Hb else [])
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    ref = eager.attention_forward_backward(q.detach(), k.detach(), v.detach(), mask, leaves[3].detach() if Hb else None, None, causal, dout)
    out = flash_sparse_attn_func(*leaves[:3], mask, leaves[3] if Hb else None, None, causal)
    for got, want, name in zip(torch.autograd.grad(out, leaves, dout), ref[1:], ("dq", "dk", "dv", "dbias")):
        assert_grad_close(got, want, name)


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("ragged", [True, False])
def test_no_memory_for_parts(ragged, native, monkeypatch):
    """The room for parts is optional: a backward that the device has no such room for runs with whole blocks."""
    from flash_sparse_attn import _cabi, flash_sparse_attn_func, flash_sparse_attn_varlen_func

    _cabi.set_compact_mode(_cabi.COMPACT_NEVER)
    if not native:
        monkeypatch.setattr(_cabi, "host", _cabi._NoHost)
    L, H, Hk, D = 4096, 8, 2, 128
    g = torch.Generator(device=DEV).manual_seed(7)
    q = torch.randn(1, L, H, D, generator=g, device=DEV).bfloat16().requires_grad_(True)
    k, v = [torch.randn(1, L, Hk, D, generator=g, device=DEV).bfloat16().requires_grad_(True) for _ in range(2)]
    dout = torch.randn(1, L, H, D, generator=g, device=DEV).bfloat16()
    cu = torch.tensor([0, L], dtype=torch.int32, device=DEV)

    def grads():
        out = flash_sparse_attn_varlen_func(q[0], k[0], v[0], cu, cu, L, L, is_causal=True) if ragged else flash_sparse_attn_func(q, k, v, is_causal=True)
        return torch.autograd.grad(out, (q, k, v), dout[0] if ragged else dout)

    def peak():
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        got = grads()
        return got, torch.cuda.max_memory_reserved()

    parts, most = peak()
    kept, held = 64 << 20, torch.cuda.memory_allocated()  # outputs, gradients, D and the forward's: 8 + 8 + 4 + 20 MB and the allocator's pieces
    assert most > held + 2 * kept  # (or this is no such call)
    try:
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + kept) / torch.cuda.get_device_properties(0).total_memory)
        whole = grads()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    _close(parts, whole, ("dq", "dk", "dv"))
