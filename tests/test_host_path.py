"""The native host path (csrc/fdma_torch.cpp) against the general Python path it stands in for: the same kernels are
launched with the same arguments, so outputs and gradients agree bit for bit; calls it was not made for are declined."""
import pytest
import torch

DEV = "cuda"


def _host():
    from flash_sparse_attn import _cabi
    return _cabi.host


def test_declines_what_is_not_an_ordinary_device_tensor():
    q = torch.randn(1, 8, 2, 64, dtype=torch.bfloat16)
    cu = torch.tensor([0, 8], dtype=torch.int32)
    assert _host().attention(q, q, q, None, None, None, None, None, None, None, 0) is NotImplemented
    assert _host().varlen_attention(q[0], q[0], q[0], cu, cu, 8, 8, None, None, None, None, None, None) is NotImplemented
    assert _host().create_mask(q, None, 4, -1.0, None, 0) is NotImplemented
    assert _host().dyn_bias(q, q, q, None) is NotImplemented
    assert _host().attention("q", q, q, None, None, None, None, None, None, None, 0) is NotImplemented


@pytest.mark.parametrize("how", ["missing", "not an extension", "another torch", "another python"])
def test_without_a_host_path_that_fits_the_operators_warn_and_decline(how, monkeypatch, tmp_path):
    """The kernels do not depend on torch's C++ interface, so neither does the package."""
    import sys
    from flash_sparse_attn import _cabi

    if how == "missing":
        monkeypatch.setattr(_cabi, "_HOST_PATH", str(tmp_path / "_fdma_torch.so"))
    elif how == "not an extension":
        (tmp_path / "_fdma_torch.so").write_bytes(b"not a shared object")
        monkeypatch.setattr(_cabi, "_HOST_PATH", str(tmp_path / "_fdma_torch.so"))
    elif how == "another torch":
        monkeypatch.setattr(torch, "__version__", "1.13.1")
    else:
        monkeypatch.setattr(sys, "version_info", (3, 99, 0))
    with pytest.warns(RuntimeWarning, match="host path"):
        host = _cabi._load_host()
    assert host.attention(*[None] * 11) is NotImplemented and host.varlen_attention(*[None] * 13) is NotImplemented
    assert host.dyn_bias(*[None] * 4) is NotImplemented and host.create_mask(*[None] * 6) is NotImplemented


def test_the_built_host_path_fits_this_torch():
    from flash_sparse_attn import _cabi

    assert _cabi.host is not _cabi._NoHost and _cabi.host.built_for[0] == torch.__version__.split("+")[0]


@pytest.mark.gpu
def test_operators_without_the_host_path(monkeypatch):
    from flash_sparse_attn import _cabi, flash_sparse_attn_func, flash_sparse_attn_varlen_func
    from flash_sparse_attn.utils.bias import dynamic_mask_bias
    from flash_sparse_attn.utils.mask import create_mask

    q, k, v, _, _, dout = _inputs(1, 200, 200, 4, 2, 64, 1, torch.bfloat16)
    w, a = [torch.randn(*s, device=DEV).bfloat16() * 0.1 for s in ((2, 128), (2,))]
    cu = torch.tensor([0, 70, 200], dtype=torch.int32, device=DEV)
    leaves = [t.requires_grad_(True) for t in (q, k, v, w, a)]
    runs = []
    for host in (_cabi.host, _cabi._NoHost):
        monkeypatch.setattr(_cabi, "host", host)
        bias = dynamic_mask_bias(v, w, a)
        mask = create_mask(bias, None, 1, 200, 200, 64, torch.finfo(bias.dtype).min)
        out = flash_sparse_attn_func(q, k, v, mask, bias, is_causal=True)
        ragged = flash_sparse_attn_varlen_func(q[0], k[0], v[0], cu, cu, 130, 130, is_causal=True)
        runs.append((mask, out.detach(), ragged.detach()) + torch.autograd.grad((out, ragged), leaves, (dout, dout[0])))
    for x, y in zip(*runs):
        assert torch.equal(x, y)


class _NoTruth:
    def __bool__(self):
        raise ValueError("no truth value")


@pytest.mark.gpu
def test_declines_flags_without_a_truth_value():
    q, k, v, mask, bias, _ = _inputs(1, 64, 64, 2, 1, 64, 1, torch.bfloat16)
    cu = torch.tensor([0, 64], dtype=torch.int32, device=DEV)
    for at in (6, 7, 8, 9):
        args = [q, k, v, mask, bias, None, None, None, None, None, 0]
        args[at] = _NoTruth()
        assert _host().attention(*args) is NotImplemented
    for at in (8, 9, 10, 11):
        args = [q[0], k[0], v[0], cu, cu, 64, 64, None, None, None, None, None, None]
        args[at] = _NoTruth()
        assert _host().varlen_attention(*args) is NotImplemented


@pytest.mark.gpu
def test_declines_while_a_trace_records_operators():
    """torch.jit.trace sees operators of the dispatcher, not launches: a call made here would be recorded as a constant."""
    q, k, v, mask, bias, _ = _inputs(1, 64, 64, 2, 1, 64, 1, torch.bfloat16)
    seen = []

    def f(x):
        seen.append(_host().attention(x, k, v, mask, bias, None, None, None, None, None, 0) is NotImplemented)
        seen.append(_host().dyn_bias(v, torch.zeros(1, 64, dtype=x.dtype, device=DEV), bias[0, 0, 0, :1], None) is NotImplemented)
        seen.append(_host().create_mask(bias, None, 8, -1.0, None, 0) is NotImplemented)
        return x + 1

    torch.jit.trace(f, (q,), check_trace=False)
    assert seen and all(seen)
    seen.clear()
    f(q)
    assert seen == [False, False, False]


def _inputs(B, Lq, Lk, H, Hk, d, rows, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    def randn(*s): return torch.randn(*s, generator=g, device=DEV).to(dtype)
    bias = randn(B, Hk, rows, Lk)
    mask = torch.rand(bias.shape, generator=g, device=DEV) < 0.4
    return randn(B, Lq, H, d), randn(B, Lk, Hk, d), randn(B, Lk, Hk, d), mask, bias, randn(B, Lq, H, d)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,rows,dtype", [
    (2, 96, 96, 4, 2, 64, 1, torch.bfloat16),     # column mask, tile skipping
    (1, 512, 1024, 8, 2, 128, 1, torch.float16),  # column mask, compaction (forward workspace reused)
    (2, 64, 128, 4, 2, 64, 64, torch.bfloat16),   # a mask and bias row per query
    (3, 1, 4096, 8, 2, 128, 1, torch.bfloat16),   # split-KV decode with its counters
])
def test_attention_equals_the_general_path(B, Lq, Lk, H, Hk, d, rows, dtype):
    from flash_sparse_attn import flash_sparse_attn_interface as itf

    q, k, v, mask, bias, dout = _inputs(B, Lq, Lk, H, Hk, d, rows, dtype)
    causal = Lq > 1
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v, bias)]
    a = _host().attention(leaves[0], leaves[1], leaves[2], mask, leaves[3], None, causal, None, None, None, 0)
    assert a is not NotImplemented and a.grad_fn is not None
    b = itf.FlashDMAttnFunc.apply(leaves[0], leaves[1], leaves[2], mask, leaves[3], None, causal, None, None, None)
    assert torch.equal(a, b)
    if Lq > 1:
        ga = torch.autograd.grad(a, leaves, dout)
        for x, y in zip(ga, torch.autograd.grad(b, leaves, dout)):
            assert torch.equal(x, y)
        # an expanded gradient (loss = out.sum()), q without one, and a second backward through a freed graph
        c = _host().attention(q, leaves[1], leaves[2], mask, leaves[3], 0.1, causal, 0.0, False, False, 0)
        c.sum().backward()
        assert leaves[1].grad is not None and leaves[0].grad is None
        with pytest.raises(RuntimeError, match="second time"):
            c.sum().backward()
    with torch.no_grad():
        n = _host().attention(q, k, v, mask, bias, None, causal, None, None, None, 0)
        assert torch.equal(n, a.detach()) and n.grad_fn is None
    with torch.inference_mode():
        assert torch.equal(_host().attention(q, k, v, mask, bias, None, causal, None, None, None, 0), n)


@pytest.mark.gpu
def test_in_place_change_of_a_saved_input_is_noticed():
    q, k, v, mask, bias, dout = _inputs(1, 64, 64, 2, 1, 64, 1, torch.bfloat16)
    k = k.requires_grad_(True)
    out = _host().attention(q, k, v, mask, bias, None, True, None, None, None, 0)
    q.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(dout)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ragged_batch_equals_the_general_path(dtype):
    from flash_sparse_attn import flash_sparse_attn_interface as itf

    lens, H, Hk, d = [5, 130, 1, 64], 4, 2, 64
    g = torch.Generator(device=DEV).manual_seed(1)
    leaves = [torch.randn(sum(lens), h, d, generator=g, device=DEV).to(dtype).requires_grad_(True) for h in (H, Hk, Hk)]
    cu = torch.tensor([0, 5, 135, 136, 200], dtype=torch.int32, device=DEV)
    a = _host().varlen_attention(*leaves, cu, cu, 130, 130, None, True, None, None, None, None)
    b = itf.FlashAttnVarlenFunc.apply(*leaves, cu, cu, 130, 130, None, True, None, None, None, None)
    assert torch.equal(a, b)
    dout = torch.randn(a.shape, generator=g, device=DEV).to(dtype)
    for x, y in zip(torch.autograd.grad(a, leaves, dout), torch.autograd.grad(b, leaves, dout)):
        assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("L,pb", [(64, True), (131, False)])
def test_bias_producer_and_mask_builder_equal_the_general_path(L, pb):
    from flash_sparse_attn.utils import bias as B, mask as M

    g = torch.Generator(device=DEV).manual_seed(2)
    def leaf(*s): return torch.randn(*s, generator=g, device=DEV).bfloat16().requires_grad_(True)
    ins = [leaf(2, L, 4, 64), leaf(4, 256), leaf(4)] + ([leaf(4)] if pb else [])
    a = _host().dyn_bias(*ins, *([] if pb else [None]))
    b = B._DynamicMaskBias.apply(*ins, *([] if pb else [None]))
    assert a.shape == b.shape and torch.equal(a, b)
    up = torch.randn(a.shape, generator=g, device=DEV).bfloat16()
    for x, y in zip(torch.autograd.grad(a, ins, up), torch.autograd.grad(b, ins, up)):
        assert torch.equal(x, y)
    keep = _host().create_mask(a, None, 40, torch.finfo(a.dtype).min, None, 0)
    assert int(keep.sum()) == 40 * 2 * 4
    idx, cnt, count, ld = M.kept_keys_of(keep)  # the record is the one the Python side reads
    assert ld % 16 == 0 and count.tolist() == [40] * 8
    row = idx[0, :40].long()
    assert keep[0, 0, 0, row].all() and torch.equal(row, row.sort().values)
    keep[0, 0, 0, 0] = ~keep[0, 0, 0, 0]
    assert M.kept_keys_of(keep) is None


def _with_hooks(call, leaves, dout):
    """Gradients with everything that is saved moved to the host in between, and what the hooks were shown."""
    packed = []

    def pack(t):
        packed.append((t.dtype, tuple(t.shape)))
        return t.device, t.detach().cpu()

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda p: p[1].to(p[0])):
        out = call()
    assert out is not NotImplemented
    return out.detach(), torch.autograd.grad(out, leaves, dout), packed


@pytest.mark.gpu
@pytest.mark.parametrize("B,Lq,Lk,H,Hk,d,rows", [
    (2, 96, 96, 4, 2, 64, 1),      # tile skipping: no workspace
    (1, 512, 1024, 8, 2, 128, 1),  # compaction: a workspace that the backward uses again
    (1, 40, 72, 2, 2, 64, 40),     # a mask and bias row per query
])
def test_saved_tensor_hooks_see_what_the_attention_saves(B, Lq, Lk, H, Hk, d, rows):
    q, k, v, mask, bias, dout = _inputs(B, Lq, Lk, H, Hk, d, rows, torch.bfloat16)
    leaves = [t.requires_grad_(True) for t in (q, k, v, bias)]
    def call(): return _host().attention(q, k, v, mask, bias, None, True, None, None, None, 0)
    out = call()
    o, grads, packed = _with_hooks(call, leaves, dout)
    assert (torch.float32, (B, H, Lq)) in packed and len(packed) == 7  # q, k, v, mask, bias, out, LSE
    assert torch.equal(o, out)
    for a, b in zip(grads, torch.autograd.grad(out, leaves, dout)):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_saved_tensor_hooks_see_what_ragged_batch_and_bias_producer_save():
    g = torch.Generator(device=DEV).manual_seed(3)
    def leaf(*s): return torch.randn(*s, generator=g, device=DEV).bfloat16().requires_grad_(True)
    cu = torch.tensor([0, 5, 135, 136, 200], dtype=torch.int32, device=DEV)
    qkv = [leaf(200, h, 64) for h in (4, 2, 2)]
    vwa = [leaf(2, 131, 4, 64), leaf(4, 256), leaf(4)]
    for call, leaves, want, n in (
        (lambda: _host().varlen_attention(*qkv, cu, cu, 130, 130, None, True, None, None, None, None), qkv, (4, 200), 7),
        (lambda: _host().dyn_bias(*vwa, None), vwa, (2 * 131, 4), 4),
    ):
        out = call()
        dout = torch.randn(out.shape, generator=g, device=DEV).bfloat16()
        o, grads, packed = _with_hooks(call, leaves, dout)
        assert (torch.float32, want) in packed and len(packed) == n
        assert torch.equal(o, out)
        for a, b in zip(grads, torch.autograd.grad(out, leaves, dout)):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_hooks_that_drop_the_strides_of_short_rows():
    """Per-query rows of fewer than eight keys are read in whole vectors, which the strides of a slice allow and those of what
    a hook hands back do not: the general path takes such calls, which pads them."""
    from flash_sparse_attn import flash_sparse_attn_func

    q, k, v, mask, bias, dout = _inputs(1, 20, 5, 2, 1, 64, 20, torch.bfloat16)
    wide = torch.zeros(1, 1, 20, 16, dtype=torch.bool, device=DEV)
    wide[..., :5] = mask
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    def call(): return flash_sparse_attn_func(q, k, v, wide[..., :5], None, None, False)
    out = call()
    o, grads, _ = _with_hooks(call, leaves, dout)
    for a, b in zip((o,) + grads, (out,) + torch.autograd.grad(out, leaves, dout)):
        assert torch.equal(a, b)
