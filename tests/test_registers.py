"""What the compiler says of the kernels' registers, read from the metadata that the built library carries beside them."""
import os

import pytest

msgpack = pytest.importorskip("msgpack")
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "flash-dmattn_amd", "lib", "libfdma_hip.so")


def kernels():
    data, key, found = open(LIB, "rb").read(), b"\xaeamdhsa.kernels", {}
    at = data.find(key)
    while at >= 0:
        unpacker = msgpack.Unpacker(strict_map_key=False)
        unpacker.feed(data[at - 1:at + (1 << 20)])  # (a map of a few entries starts with one byte)
        for k in unpacker.unpack()["amdhsa.kernels"]:
            found[k[".name"]] = k
        at = data.find(key, at + 1)
    return found


def test_decode_holds_its_state_in_registers():
    """No lane's state of the decode kernels goes through scratch memory: what was reloaded from there behind the loop over the keys had
    come back in some of the lanes only."""
    decode = {n: k for n, k in kernels().items() if "decode_kernel" in n}
    assert len(decode) == 2 * 3 * 6
    for name, k in decode.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name


def test_sums_of_parts_stay_apart_from_dq():
    """The compacted dQ kernels carry the sums of the dK / dV parts; neither holds the other's scalars (the sums' own loop over items has
    more than it can keep, by about fifteen; held together they were 67 to 115 too many)."""
    dq = {n: k for n, k in kernels().items() if "bwd_dq_256_kernel" in n and "ELb1EEE" in n or "bwd_dq_colmask_kernel" in n and "ELb1ELb0EEE" in n}
    assert len(dq) == 2 * (2 + 4)
    for name, k in dq.items():
        assert k[".sgpr_spill_count"] <= 20 and k[".vgpr_spill_count"] == 0, name


def test_forward_with_key_groups():
    """The forward with key groups keeps a lane's state in registers up to head dim 128; above, where O alone is 128 of them and Q 64, up
    to five do not fit (20 bytes a lane, in the kernel that reads a list's rows where they lie)."""
    fwd = {n: k for n, k in kernels().items() if "fwd_wide_kernel" in n or "fwd_96_kernel" in n or "fwd_list_kernel" in n}
    assert len(fwd) == 2 * (4 * 4 + 4 + 4 * 2)
    for name, k in fwd.items():
        most = (5, 20) if "Li256E" in name else (0, 0)
        assert (k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) <= most and k[".private_segment_fixed_size"] <= most[1], name
