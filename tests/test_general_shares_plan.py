"""Shares of the general form's key tiles, asked for on the host (no GPU): a call is offered room for them only where the kernel that takes it
works on shares.  At head dims 65 to 128 the kernels of 256 query rows, which take calls of 512 such blocks or more, do not."""
import pytest


def _ask(B, Lq, Lk, H, Hk, d, bias_heads):
    from flash_sparse_attn import _cabi

    a = _cabi.BwdArgs()
    f = a.f
    f.batch, f.seqlen_q, f.seqlen_k, f.num_heads, f.num_heads_k, f.head_dim = B, Lq, Lk, H, Hk, d
    f.mask, f.num_heads_mask = 256, Hk  # (there is one, with a row per query; sizes alone are looked at)
    f.mask_strides[0], f.mask_strides[1], f.mask_strides[2] = Hk * Lq * Lk, Lq * Lk, Lk
    if bias_heads:
        f.bias, f.num_heads_bias, a.dbias = 256, bias_heads, 256
        for strides in (f.bias_strides, a.dbias_strides):
            strides[0], strides[1], strides[2] = bias_heads * Lq * Lk, Lq * Lk, Lk
    return _cabi.lib.fdma_fwd_optional_bytes(f), _cabi.lib.fdma_fwd_counter_bytes(f), _cabi.lib.fdma_bwd_optional_bytes(a)


SIZES = [(B, H, Hk) for B in (1, 3, 15, 16, 17, 31, 32, 128, 512, 1024) for H in (1, 2, 4, 8, 12, 16, 32, 64) for Hk in (1, 2, 4, 8, 32) if H % Hk == 0]


@pytest.mark.parametrize("bias_heads", [0, 1])
def test_room_only_where_a_kernel_works_on_shares(bias_heads):
    offered = 0
    for B, H, Hk in SIZES:
        for Lq in (2, 16, 31, 32, 33, 64, 129, 256, 257, 600):
            for Lk in (704, 1472, 1473, 4096):
                for d in (64, 72, 96, 128, 136, 256):
                    rows256 = 64 < d <= 128 and B * H * -(-Lq // 256) >= 512
                    forward, counters, backward = _ask(B, Lq, Lk, H, Hk, d, bias_heads)
                    offered += backward > 0
                    assert not (rows256 and (forward or counters or backward)), (B, Lq, Lk, H, Hk, d)
                    assert (counters > 0) == (forward > 0 and d <= 128)
    assert offered > 1000


@pytest.mark.parametrize("B,Lq,H,Hk,d,shares", [
    (16, 32, 32, 8, 128, 1),
    (15, 32, 32, 8, 128, 2),  # 480 blocks of 256 rows: 120 workgroups of 32 rows of four heads, two shares each
    (16, 32, 32, 8, 64, 6),   # (no kernels of 256 rows)
    (1, 32, 4, 1, 128, 8),
])
def test_either_side_of_the_line(B, Lq, H, Hk, d, shares):
    forward, counters, backward = _ask(B, Lq, 4096, H, Hk, d, 0)
    assert (forward > 0, counters > 0) == (shares > 1, shares > 1)
    assert backward == (shares * B * H * Lq * d * 4 if shares > 1 else 0)
