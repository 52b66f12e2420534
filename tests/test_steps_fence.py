"""Batched passes of several steps hand rows from lane to lane through LDS
(custen_amd/csrc/stencil_steps.h).  The compiler sees one lane, so only a fence
keeps its reads of other lanes' columns after the write: between every store to
LDS and the next load from it there has to be one, in what the compiler makes of
the kernels."""
import os
import re
import subprocess

import pytest

from custen_amd import build


def unfenced_loads(text):
    """Loads from LDS that some path reaches from a store to LDS without a fence."""
    blocks, name = {"": []}, ""
    for line in text.splitlines()[1:]:
        m = re.match(r"(\d+):", line)
        if m:
            name = m.group(1)
            blocks[name] = []
        else:
            blocks[name].append(line)

    def walk(lines, stored):
        bad = []
        for line in lines:
            if re.search(r"\bstore .*ptr addrspace\(3\)", line):
                stored = True
            elif "fence syncscope" in line:
                stored = False
            elif stored and re.search(r"= load .*ptr addrspace\(3\)", line):
                bad.append(line)
        return stored, bad

    bad, entered, work = [], set(), [("", False)]
    while work:
        name, stored = work.pop()
        if (name, stored) in entered:
            continue
        entered.add((name, stored))
        stored, found = walk(blocks[name], stored)
        bad += found
        work += [(b, stored) for line in blocks[name] if line.lstrip().startswith("br ")
                 for b in re.findall(r"label %(\d+)", line)]
    assert len({name for name, _ in entered}) == len(blocks)
    return bad


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="hipcc not available")
def test_lds_rows_are_fenced(tmp_path):
    ll = tmp_path / "batch.ll"
    subprocess.run([build.HIPCC, "-x", "hip", *build.COMMON, "--cuda-device-only", "-emit-llvm",
                    "-S", os.path.join(build.CSRC, "batch.hip"), "-o", str(ll)], check=True,
                   capture_output=True, timeout=120)
    kernels = re.findall(r"^define [^\n]*batchStepsKernel.*?^}", ll.read_text(), re.M | re.S)
    assert len(kernels) == 4
    for text in kernels:
        assert unfenced_loads(text) == []
        assert len(re.findall(r"\bstore .*ptr addrspace\(3\)", text)) >= 6
