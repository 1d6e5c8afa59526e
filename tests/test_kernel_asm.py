"""Properties of the compiled kernels that no result shows: read from the AMD assembly
of this repository's own sources, built with the library's flags."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.dirname(os.path.realpath(__file__)))
PKG = os.path.join(HERE, "mojostream_amd")


def _asm(name):
    """Kernels of csrc/<name>.hip: mangled name -> instruction lines and labels."""
    if not (os.path.exists("/opt/rocm/bin/hipcc") or shutil.which("hipcc")):
        pytest.skip("hipcc not installed")
    out = os.path.join(PKG, "_build", name + ".s")
    subprocess.run(["make", "-s", "-C", PKG, out], check=True)
    kernels, cur = {}, None
    with open(out) as f:
        for line in f:
            line = line.split(";")[0].strip()
            if re.fullmatch(r"_Z\w+:", line):
                cur = kernels.setdefault(line[:-1], [])
            elif line.startswith(".Lfunc_end"):
                cur = None
            elif cur is not None and line and not (line[0] == "." and not line.endswith(":")):
                cur.append(line)
    return kernels


_READ = re.compile(r"ds_(read|load|write|store)")
_LGKM = re.compile(r"lgkmcnt\((\d+)\)")


def _in_flight_at_barriers(lines):
    """The most LDS reads and writes of a wave that can be in flight at each s_barrier,
    over all paths: a fixed point over the basic blocks."""
    blocks, names = [[]], {}
    for ln in lines:
        if ln.endswith(":"):
            if blocks[-1]:
                blocks.append([])
            names[ln[:-1]] = len(blocks) - 1
        else:
            blocks[-1].append(ln)
            if re.match(r"s_(cbranch|branch|endpgm|setpc)", ln):
                blocks.append([])
    most = [0] * len(blocks)
    found = {}
    work = list(range(len(blocks)))
    while work:
        b = work.pop()
        n, nxt = most[b], [b + 1]
        for i, ln in enumerate(blocks[b]):
            op = ln.split()[0]
            if _READ.match(op):
                n = min(n + 1, 15)  # (the counter's range)
            elif op == "s_waitcnt":
                w = _LGKM.search(ln)
                if w:
                    n = min(n, int(w.group(1)))
            elif op == "s_barrier":
                found[b, i] = max(found.get((b, i), 0), n)
            elif op == "s_endpgm":
                nxt = []
            elif op == "s_branch":
                nxt = [names[ln.split()[1]]]
            elif op.startswith("s_cbranch"):
                nxt = [b + 1, names[ln.split()[1]]]
        for t in nxt:
            if t < len(blocks) and n > most[t]:
                most[t] = n
                work.append(t)
    return list(found.values())


def test_in_flight_counts():
    """The count on hand-written blocks: a read before a barrier, one behind a wait,
    one that reaches the barrier around a loop only."""
    assert _in_flight_at_barriers(["ds_read_b128 v[0:3], v4", "s_barrier"]) == [1]
    assert _in_flight_at_barriers(["ds_read_b128 v[0:3], v4", "ds_read_b128 v[0:3], v4",
                                   "s_waitcnt vmcnt(0) lgkmcnt(1)", "s_barrier"]) == [1]
    assert _in_flight_at_barriers(["ds_read_b128 v[0:3], v4", "s_waitcnt lgkmcnt(0)",
                                   "s_barrier", "s_endpgm"]) == [0]
    assert _in_flight_at_barriers([".LBB0_1:", "s_barrier", "ds_read_b128 v[0:3], v4",
                                   "s_cbranch_scc1 .LBB0_1", "s_endpgm"]) == [15]


@pytest.mark.parametrize("source,kernel", [("flash", "k_flash"), ("gemm", "k_gemm")])
def test_lds_reads_done_at_barriers(source, kernel):
    """Loads straight into LDS refill a buffer after the barrier that follows its last
    reads: a wave must not pass that barrier with its reads in flight, since nothing
    orders them against another wave's load."""
    seen = 0
    for name, lines in _asm(source).items():
        if f"{kernel}I" not in name:
            continue
        n = _in_flight_at_barriers(lines)
        assert n and max(n) == 0, f"{name}: LDS accesses in flight at its barriers: {n}"
        seen += 1
    assert seen >= 4


def test_range_checked_loads_check_the_whole_offset():
    """The GEMV kernels rely on range-checked loads that return zeros past the end of an
    operand.  The check need not cover the scalar offset, so it has to be zero."""
    seen = 0
    for name, lines in _asm("q4").items():
        for ln in lines:
            if not ln.startswith("buffer_load"):
                continue
            ops = [o.strip() for o in ln.split(None, 1)[1].split(",")]
            soff = ops[-1].split()[0]
            assert soff == "0", f"{name}: {ln}"
            seen += "k_gemv_rows" in name
    assert seen > 100
