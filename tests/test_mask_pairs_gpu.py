"""The keep-mask builder's register form, which compares and counts two columns an instruction: rows with every kind of 16-bit value, fill
values below, at (both zeros) and above the threshold, windows of one, half and all columns, row ends inside a chunk, and the largest row
all of whose columns are kept -- against a stable sort of the ordered 16-bit keys, exactly; and the list of the row."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _keys(x):
    """Unsigned 16-bit keys in the numeric order of the floats (sign and magnitude: -0 below +0, NaN beyond the infinities)."""
    b = x.view(torch.int16).numpy().view(np.uint16).astype(np.int64)
    return np.where(b & 0x8000, ~b & 0xFFFF, b | 0x8000)


@pytest.mark.parametrize("L", [8, 13, 515, 2049, 8197, 16390, 65536])
@pytest.mark.parametrize("fill", [None, 0.0, 1.0])
@pytest.mark.parametrize("kind", ["one", "half", "all", "relu"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows(L, fill, kind, dtype):
    from flash_sparse_attn.utils.mask import create_mask, kept_keys_of

    g = torch.Generator().manual_seed(L)
    x = torch.randn(1, 2, 1, L, generator=g).to(dtype)
    odd = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), 1.0, -1.0, torch.finfo(dtype).tiny / 2], dtype=dtype)
    at = torch.rand(x.shape, generator=g) < 0.3
    x[at] = odd[torch.randint(0, len(odd), x.shape, generator=g)][at]
    pad = torch.rand(1, L, generator=g) < 0.8
    fill = torch.finfo(dtype).min if fill is None else fill
    window = {"one": 1, "half": L // 2, "all": L, "relu": 7}[kind]
    got = create_mask(x.to(DEV), pad.to(DEV), 1, 1, L, window, fill, type="relu" if kind == "relu" else "topk")
    y = x.masked_fill(~pad[:, None, None, :], fill)
    if kind == "relu":
        want = (y > 0).numpy()
    else:
        order = np.argsort(-_keys(y), axis=-1, kind="stable")[..., :window]
        want = np.zeros(y.shape, dtype=bool)
        np.put_along_axis(want, order, True, -1)
        want &= (y != torch.tensor(fill, dtype=dtype)).numpy()
    assert np.array_equal(got.cpu().numpy(), want)
    idx, cnt, count, _ = [t.cpu() if torch.is_tensor(t) else t for t in kept_keys_of(got)]
    m = torch.from_numpy(want).reshape(-1, L)
    assert torch.equal(count.long(), m.sum(-1)) and torch.equal(cnt[:, :L].long(), m.cumsum(-1))
    for i in range(2):
        assert torch.equal(idx[i, : count[i]].long(), m[i].nonzero().flatten())


@pytest.mark.parametrize("window", [1, 9, 4096, 65528, 65535, 65536])
@pytest.mark.parametrize("above", [0, 1, 9])
def test_largest_row_of_equal_values(window, above):
    """65536 ties, or nearly as many: the first ones in column order are kept, behind what lies above them."""
    from flash_sparse_attn.utils.mask import create_mask, kept_keys_of

    L = 65536
    x = torch.full((1, 1, 1, L), 0.25, dtype=torch.bfloat16)
    x[..., torch.arange(above) * 7000 + 3] = 1.0
    got = create_mask(x.to(DEV), None, 1, 1, L, window, torch.finfo(x.dtype).min, type="topk")
    want = torch.zeros(L, dtype=torch.bool)
    want[torch.argsort(-x.flatten().float(), stable=True)[:window]] = True
    assert torch.equal(got.cpu().flatten(), want)
    idx, cnt, count, _ = [t.cpu() if torch.is_tensor(t) else t for t in kept_keys_of(got)]
    assert int(count) == window and torch.equal(idx[0, :window].long(), want.nonzero().flatten()) and torch.equal(cnt[0, :L].long(), want.cumsum(0))
