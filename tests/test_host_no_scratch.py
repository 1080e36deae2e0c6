"""Kernels whose waits count the requests under way, with every register spoken for: nothing of theirs goes through scratch memory, whose accesses
would count among the requests and turn each wait into one for the next tile as well.  Looked for in what the compiler reports of them under the
build's own flags."""

import os
import re
import subprocess

import pytest

from ops_rec import _build

SOURCES = {"in_linear_silu_kernels_rows.hip": 6}  # (kernels in each)


def scratch_of(assembly):
    """{kernel: bytes of scratch memory per lane}, from the kernel descriptors."""
    sizes = re.findall(r"\.amdhsa_kernel (\w+)\n(?:\s+\.amdhsa_.*\n)*?\s+\.amdhsa_private_segment_fixed_size (\d+)", assembly)
    return {name: int(size) for name, size in sizes}


def spills_of(assembly):
    """{kernel: registers spilled, to scratch memory or elsewhere}, from the metadata."""
    kernels = re.findall(r"^\s+\.name:\s+(\w+)$(.*?)^\s+\.wavefront_size:", assembly, re.M | re.S)
    return {name: sum(map(int, re.findall(r"\.[sv]gpr_spill_count:\s+(\d+)", body))) for name, body in kernels}


@pytest.mark.parametrize("source", list(SOURCES))
def test_nothing_in_scratch(source, tmp_path):
    try:
        hipcc = _build.hipcc_path()
    except RuntimeError:
        pytest.skip("no hipcc on this host")
    out = tmp_path / "kernels.s"
    flags = [*_build.HIPCC_FLAGS, *_build.OPERAND_SOURCE_FLAGS[source]]
    subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", os.path.join(_build.CSRC, source), "-o", str(out)], check=True, capture_output=True,
                   timeout=300)  # fmt: skip
    text = out.read_text()
    scratch, spills = scratch_of(text), spills_of(text)
    assert len(scratch) == len(spills) == SOURCES[source], (scratch, spills)
    assert not any(scratch.values()) and not any(spills.values()), (scratch, spills)
    assert not re.search(r"^\s+scratch_", text, re.M)


def test_the_sources_are_these():
    assert set(_build.OPERAND_SOURCE_FLAGS) == set(SOURCES)


def test_the_check_sees_what_it_looks_for():
    descriptor = "\t.amdhsa_kernel _Zk\n\t\t.amdhsa_group_segment_fixed_size 64\n\t\t.amdhsa_private_segment_fixed_size 12\n"
    assert scratch_of(descriptor) == {"_Zk": 12}
    metadata = "    .name:           _Zk\n    .sgpr_spill_count: 0\n    .vgpr_spill_count: 3\n    .wavefront_size: 64\n"
    assert spills_of(metadata) == {"_Zk": 3}
