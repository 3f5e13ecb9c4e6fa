"""The lanes of one wavefront hand words to each other through LDS without a
workgroup barrier in the matrix tile path: the staged V tile, and the members
of a prefix piece's query rows.  The hardware keeps a wavefront's LDS accesses
in order; the compiler does only across a fence, since no single lane reads
the words that it wrote.  So in the LLVM IR of those exchanges every change
between LDS stores and LDS loads has to have a fence in it (the IR and not the
machine code: there a fence of one wavefront leaves nothing)."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("ir") / "tile_lds_order.ll"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "xllms_amd", "csrc"), "-S", "-emit-llvm",
                    os.path.join(ROOT, "tests", "c", "tile_lds_order.hip"), "-o", str(out)],
                   check=True, timeout=300)
    return out.read_text()


def blocks_of(body):
    """{label: (LDS accesses and fences in order, successors)} of a function."""
    lines = body.splitlines()
    first = str(1 + max(map(int, re.findall(r"%(\d+)[,)]", lines[0]))))  # after the arguments
    blocks, at = {first: ([], [])}, first
    for line in lines[1:]:
        label = re.match(r"(\w[\w.]*):", line)
        if label:
            at = label.group(1)
            blocks[at] = ([], [])
        elif re.search(r"\bfence syncscope\(\"wavefront\"\) acq_rel", line):
            blocks[at][0].append("fence")
        elif re.match(r"\s*store .*addrspace\(3\)", line):
            blocks[at][0].append("store")
        elif re.match(r"\s*%\S+ = load .*addrspace\(3\)", line):
            blocks[at][0].append("load")
        blocks[at][1].extend(re.findall(r"label %([\w.]+)", line))
    return first, blocks


@pytest.mark.parametrize("name", ["v_tiles_KV_F16_32", "v_tiles_KV_F16_64", "v_tiles_KV_F16_80",
                                  "v_tiles_KV_BF16_96", "v_tiles_KV_BF16_112", "v_tiles_KV_F32_32",
                                  "prefix_members"])
def test_lds_exchange_is_fenced(listing, name):
    body = re.search(r"^define [^\n]*@%s\(.*?^}" % name, listing, re.S | re.M).group(0)
    first, blocks = blocks_of(body)
    every = [k for ops, _ in blocks.values() for k in ops]
    assert every.count("store") >= 2 and every.count("load") >= 2, every  # two tiles (pieces)
    # the accesses since the last fence, over every path
    since = {first: {"none"}}
    work = [first]
    while work:
        at = work.pop()
        ops, succ = blocks[at]
        now = set(since[at])
        for k in ops:
            if k == "fence":
                now = {"none"}
                continue
            other = "load" if k == "store" else "store"
            assert other not in now, f"{name}: a {other}, then a {k} with no fence between"
            now = {k}
        for b in succ:
            if not now <= since.get(b, set()):
                since[b] = since.get(b, set()) | now
                work.append(b)


def test_cascade_plan_has_its_lds():
    """The static LDS of the cascade's partition launch leaves the in-kernel
    plan the room of batches of 1024 to 1500 sequences (larger ones go to the
    plan kernels, two more launches)."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-device-only", "-fsyntax-only",
                        "-std=c++17", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "xllms_amd", "csrc"),
                        os.path.join(ROOT, "tests", "c", "cascade_lds_size.hip")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
