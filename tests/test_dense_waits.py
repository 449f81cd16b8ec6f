"""The dense kernels that move input rows into LDS by DMA wait with s_waitcnt vmcnt(n): the transfers have landed when only
the n weight loads issued after them are in flight. That holds while at least n loads stand between the last transfer
and the wait, and the source must not leave it to chance: the weights may not be noalias, read-only kernel arguments,
whose loads count as loads of constant memory and may be moved across the transfers. Checked in the assembly that hipcc
makes of dense.hip here; needs no GPU."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "moex_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("asm") / "dense.s"
    flags = re.search(r"^HIPFLAGS = (.*?[^\\])\n", open(os.path.join(CSRC, "Makefile")).read(), re.S | re.M).group(1)
    flags = flags.replace("\\\n", " ").replace("$(ARCH)", "gfx950").split()
    subprocess.run([HIPCC, *flags, "-S", "--cuda-device-only", os.path.join(CSRC, "dense.hip"), "-o", str(out)], check=True,
                   capture_output=True)
    return out.read_text()


def _counted_waits(body):
    """(n, vector-memory loads since the last transfer) of every wait of the kernel's own asm statements, in program text"""
    got, loads, seen, own = [], 0, False, False
    for line in body.splitlines():
        t = line.strip()
        if "#ASMSTART" in t or "#ASMEND" in t:
            own = "#ASMSTART" in t
        elif t.startswith("global_load_lds"):
            loads, seen = 0, True
        elif re.match(r"(global|flat|buffer)_(load|store|atomic)", t):
            loads += 1
        elif own and seen:
            m = re.match(r"s_waitcnt.*vmcnt\((\d+)\)", t)
            if m:
                got.append((int(m.group(1)), loads))
    return got


def _kernels(text, name):
    return {m.group(1): m.group(2) for m in re.finditer(r"^(\S*%s\S*):(.*?)^\s*\.size\s" % name, text, re.S | re.M)
            if not m.group(1).startswith(".")}


def _arguments(text, kernel):
    """the metadata of the kernel's arguments, one string each"""
    block = re.search(r"\.args:((?:(?!\.args:).)*?)\.name:\s+%s\s" % re.escape(kernel), text, re.S).group(1)
    return re.split(r"\n\s+- ", block.split(".group_segment_fixed_size")[0])[0:]


@pytest.mark.parametrize("name,weights", [("gemv1_kernel", 1), ("gemm_tile_kernel", 3)])
def test_counted_waits(assembly, name, weights):
    """weights: the leading arguments whose loads the waits count"""
    found = 0
    for kernel, body in _kernels(assembly, name).items():
        waits = _counted_waits(body)
        if not waits:
            continue  # no transfers into LDS
        found += 1
        for n, loads in waits:
            assert loads >= n, (kernel, n, loads)
        args = [a for a in _arguments(assembly, kernel) if ".offset" in a]
        for a in args[:weights]:
            assert "read_only" not in a, (kernel, a)
    assert found >= 12, found
