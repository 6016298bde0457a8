"""Direct loads (global to LDS, issued in assembly) that nothing waits for, looked for in the AMD assembly of the library's own
source: the compiler does not know of such loads, so where LDS changes its use a wait has to stand in the source.

In the forward with key groups (fdma_fwd_wide.hip) the merge puts row sums and shares of O where the K and V tiles were.  Over every
path through a kernel: a store of the fused bias column (4 bytes) needs this wave's direct loads to have landed, a store of the merge
(16 bytes a lane, which nothing else in these kernels stores) needs a barrier after that as well, because the tiles are everybody's."""
import os
import re
import shlex
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "flash-dmattn_amd", "csrc")

NONE, LANDED, IN_FLIGHT = 0, 1, 2  # direct loads of this wave: none since the last barrier, waited for, in flight


def _assembly(name, tmp_path):
    lines = subprocess.run(["make", "-n", "-B", "-C", CSRC, name + ".o"], capture_output=True, text=True, check=True).stdout.splitlines()
    cmd = shlex.split(next(line for line in lines if name + ".hip" in line))
    if shutil.which(cmd[0]) is None:
        pytest.skip("no hipcc")
    out = str(tmp_path / (name + ".s"))
    cmd[cmd.index("-c")] = "-S"
    cmd[cmd.index("-o") + 1] = out
    subprocess.run(cmd + ["--cuda-device-only"], cwd=CSRC, check=True, timeout=600)
    with open(out) as f:
        return f.read()


def _early_stores(body):
    """(direct loads, LDS stores that some path reaches too early) of one kernel."""
    code, labels = [], {}
    for line in body.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"(\S+):$", line)
        if label:
            labels[label.group(1)] = len(code)
        elif line and not line.startswith("."):
            code.append(line)
    state, todo, early = [-1] * len(code), [(0, NONE)], set()
    while todo:
        at, s = todo.pop()
        if s <= state[at]:
            continue
        state[at] = s
        op, *args = code[at].split()
        if op.startswith("global_load_lds"):
            s = IN_FLIGHT
        elif op == "s_waitcnt" and "vmcnt(0)" in args:
            s = min(s, LANDED)
        elif op == "s_barrier" and s == LANDED:
            s = NONE
        elif op.startswith("ds_write") and s > (NONE if op == "ds_write_b128" else LANDED):
            early.add((at, code[at]))
        if op == "s_branch" or op.startswith("s_cbranch"):
            todo.append((labels[args[0]], s))
        if op not in ("s_branch", "s_endpgm") and at + 1 < len(code):
            todo.append((at + 1, s))
    return sum(c.startswith("global_load_lds") for c in code), sorted(early)


def test_no_direct_load_in_flight_at_the_merge_of_key_groups(tmp_path):
    text = _assembly("fdma_fwd_wide", tmp_path)
    kernels = re.findall(r"^(_Z\S*fwd_wide_kernel\S*):.*?\n(.*?)^\.Lfunc_end", text, re.M | re.S)
    assert len(kernels) == 32
    for name, body in kernels:
        loads, early = _early_stores(body)
        assert loads > 0 and "ds_write_b128" in body, name
        assert not early, (name, early[:3])


def test_nor_at_that_of_their_variants(tmp_path):
    """The same kernels for head dims 65 to 96, and those that read a list's rows where they lie."""
    text = _assembly("fdma_fwd_wide", tmp_path)
    kernels = re.findall(r"^(_Z\S*(?:fwd_96|fwd_list)_kernel\S*):.*?\n(.*?)^\.Lfunc_end", text, re.M | re.S)
    assert len(kernels) == 8 + 16
    for name, body in kernels:
        loads, early = _early_stores(body)
        assert loads > 0 and "ds_write_b128" in body, name
        assert not early, (name, early[:3])
