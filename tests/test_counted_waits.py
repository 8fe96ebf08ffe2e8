"""The kernels that wait for a part of their loads in flight
(s_waitcnt vmcnt(N), with N counted by hand in gemm_rows.hip and
frontend.hip) hold only while the compiler emits the loads that were counted.
This reads the gfx950 assembly of both files, built here from source, and
counts each pipelined loop's: loads of weights to registers and copies of
activations to LDS, per barrier. No device is needed."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "qwenscriber_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-fno-gpu-rdc", "-x", "hip", "--cuda-device-only", "-S"]

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")


def kernels(source, name, tmp_path):
    """{symbol: lines} of the kernels whose symbol holds `name`."""
    out = os.path.join(str(tmp_path), source + ".s")
    subprocess.run([HIPCC, *FLAGS, os.path.join(CSRC, source), "-o", out], check=True, capture_output=True)
    found, lines = {}, None
    with open(out) as f:
        for line in f:
            m = re.match(r"(_Z\w+):", line)
            if m:
                lines = found.setdefault(m.group(1), []) if name in m.group(1) else None
            if line.startswith(".Lfunc_end"):
                lines = None
            if lines is not None:
                lines.append(line.split(";")[0].strip())
    return found


def blocks(lines):
    """Basic blocks and their successors."""
    starts = {0} | {i for i, line in enumerate(lines) if re.match(r"\.LBB\w+:$", line)}
    starts |= {i + 1 for i, line in enumerate(lines) if re.match(r"s_c?branch|s_endpgm", line)}
    starts = sorted(i for i in starts if i < len(lines))
    index = {i: n for n, i in enumerate(starts)}
    label = {lines[i][:-1]: n for i, n in index.items() if lines[i].endswith(":")}
    body = [lines[i:j] for i, j in zip(starts, starts[1:] + [len(lines)])]
    after = []
    for n, block in enumerate(body):
        last = block[-1] if block else ""
        m = re.match(r"s_(c?)branch\w* (\.LBB\w+)", last)
        to = [label[m.group(2)]] if m else []
        if not (m and not m.group(1)) and not last.startswith("s_endpgm") and n + 1 < len(body):
            to.append(n + 1)
        after.append(to)
    return body, after


def reachable(after, n):
    seen, todo = set(), list(after[n])
    while todo:
        k = todo.pop()
        if k not in seen:
            seen.add(k)
            todo += after[k]
    return seen


def pipelined_loops(lines):
    """(barriers, loads to registers, copies to LDS, scratch accesses) of each
    loop with a barrier and matrix products."""
    body, after = blocks(lines)
    reach = [reachable(after, n) for n in range(len(body))]
    counts, done = [], set()
    for n in range(len(body)):
        if n in done or n not in reach[n]:
            continue
        loop = [k for k in reach[n] if n in reach[k]]
        done.update(loop)
        ops = [line for k in loop for line in body[k]]
        have = {key: sum(line.startswith(key) for line in ops)
                for key in ("s_barrier", "v_mfma", "global_load_lds", "global_load", "scratch", "buffer")}
        if have["s_barrier"] and have["v_mfma"]:
            counts.append((have["s_barrier"], have["global_load"] - have["global_load_lds"], have["global_load_lds"],
                           have["scratch"] + have["buffer"]))
    return counts


def test_rows_product_loads(tmp_path):
    # Codes (0 q4, 1 q5, 2 q8): groups of a weight chunk, loads of a group's.
    chunk, loads = {0: 4, 1: 2, 2: 2}, {0: 1, 1: 2, 2: 2}
    found = kernels("gemm_rows.hip", "gemm_rows_kernel", tmp_path)
    assert len(found) == 6
    for symbol, lines in found.items():
        code, waves, tiles = (int(v) for v in re.search(r"CodesE(\d)ELi(\d)ELi(\d)", symbol).groups())
        groups, copies = chunk[code], tiles * 512 // (64 * waves)
        pipelined = [c for c in pipelined_loops(lines) if c[0] == groups]
        assert pipelined == [(groups, groups * loads[code] + 1, groups * copies, 0)], (symbol, pipelined)


def test_convolution_loads(tmp_path):
    found = kernels("frontend.hip", "conv3x3s2_gelu_mfma_kernel", tmp_path)
    assert len(found) == 20
    for symbol, lines in found.items():
        rounds = int(re.search(r"kernelILi\dELi(\d)E", symbol).group(1))
        assert pipelined_loops(lines) == [(1, 18, rounds, 0)], (symbol, pipelined_loops(lines))
