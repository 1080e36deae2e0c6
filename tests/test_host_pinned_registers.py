"""What the compiler has to keep for the kernels with sums in accumulators that assembly names (hstu_pinned_acc.hip.h), looked for in what it
makes of them with the build's own flags:

* it uses none of the accumulators that a kernel's assembly names;
* no vector instruction writes an operand of a matrix instruction in assembly in the two wait states ahead of it;
* nothing reads or writes the registers of a load in assembly between the load and the wait for it.

Each kernel's instructions are followed along its branches, the states of joining paths together.
"""

import concurrent.futures
import os
import re
import shutil
import subprocess

import pytest

from ops_rec import _build

SOURCES = {"hstu_kernels_bwd_fused.hip": 24, "hstu_kernels_fwd_pinned.hip": 4}  # (kernels in each)
_REGISTERS = {kind: re.compile(rf"(?<![\w.]){kind}(?:\[(\w+):(\w+)\]|(\d+))") for kind in "va"}


def registers(kind, text):
    """The vector (``v``) or accumulation (``a``) registers named in ``text``, as a bit mask."""
    mask = 0
    for first, last, one in _REGISTERS[kind].findall(text):
        lo, hi = (int(one), int(one)) if one else (int(first, 0), int(last, 0))
        mask |= (1 << (hi + 1)) - (1 << lo)
    return mask


def kernels(text):
    """{name: [(instruction or label, whether it stands in assembly)]}"""
    found, body, assembly = {}, None, False
    for line in text.splitlines():
        start = re.match(r"(_Z\w+):", line)
        if start:
            body = found[start[1]] = []
            continue
        if "ASMSTART" in line or "ASMEND" in line:
            assembly = "ASMSTART" in line
            continue
        line = line.split(";")[0].strip()
        if body is None or not line or (line.startswith(".") and not line.endswith(":")):
            continue
        if line.startswith(".Lfunc_end"):
            body = None
        else:
            body.append((line, assembly))
    return {name: body for name, body in found.items() if any(t == "s_endpgm" for t, _ in body)}


def steps_of(body):
    """Where each instruction leads: indices into ``body``."""
    labels = {text[:-1]: i for i, (text, _) in enumerate(body) if text.endswith(":")}
    steps = []
    for i, (text, _) in enumerate(body):
        op, _, target = text.partition(" ")
        if op == "s_endpgm":
            steps.append(())
        elif op == "s_branch":
            steps.append((labels[target.strip()],))
        elif op.startswith("s_cbranch"):
            steps.append((labels[target.strip()], i + 1))
        else:
            assert not op.startswith(("s_setpc", "s_swappc", "s_call")), text
            steps.append((i + 1,))
    return steps


def problems(body):
    pinned = 0
    for text, assembly in body:
        if assembly:
            pinned |= registers("a", text)
    wrong = {f"accumulator of the assembly's own outside it: {t}" for t, assembly in body if not assembly and registers("a", t) & pinned}
    steps = steps_of(body)
    # per instruction, on entry: vector registers written one and two wait states ago, and those that a load in assembly will fill
    state = [None] * len(body)
    state[0], todo = (0, 0, 0), [0]
    while todo:
        i = todo.pop()
        text, assembly = body[i]
        last, before, filling = state[i]
        op, _, operands = text.partition(" ")
        used = registers("v", operands)
        if op == "s_waitcnt" and "vmcnt" in text and (assembly or "vmcnt(0)" in text):
            filling = 0
        elif used & filling:
            wrong.add(f"register of a load that is under way: {text}")
        written = 0
        if op.startswith("v_") and "mfma" not in op:
            first = operands.split(",")[0]
            both = op.startswith(("v_swap", "v_permlane32_swap", "v_permlane16_swap"))
            written = registers("v", operands if both else first)
        if assembly and "mfma" in op and used & (last | before):
            wrong.add(f"operand written right ahead: {text}")
        if assembly and op.startswith("buffer_load") and " lds" not in text:
            filling |= registers("v", operands.split(",")[0])
        if text.endswith(":"):
            out = (last, before, filling)
        elif op == "s_nop":
            out = (0, last if operands.strip() == "0" else 0, filling)
        else:
            out = (written, last, filling)
        for j in steps[i]:
            joined = out if state[j] is None else tuple(a | b for a, b in zip(state[j], out))
            if joined != state[j]:
                state[j] = joined
                todo.append(j)
    return wrong


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    try:
        hipcc = _build.hipcc_path()
    except RuntimeError:
        pytest.skip("no hipcc on this host")
    directory = tmp_path_factory.mktemp("assembly")

    def one(source):
        out = directory / (source + ".s")
        flags = [*_build.HIPCC_FLAGS, *_build.SOURCE_FLAGS[source]]
        subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", os.path.join(_build.CSRC, source), "-o", str(out)], check=True,
                       capture_output=True, timeout=300)  # fmt: skip
        return kernels(out.read_text())

    with concurrent.futures.ThreadPoolExecutor() as pool:
        yield dict(zip(SOURCES, pool.map(one, SOURCES)))
    shutil.rmtree(directory, ignore_errors=True)


def test_the_sources_with_named_accumulators_are_these():
    assert set(_build.SOURCE_FLAGS) == set(SOURCES)


@pytest.mark.parametrize("source", list(SOURCES))
def test_the_compiler_keeps_clear_of_what_the_assembly_holds(source, compiled):
    found = compiled[source]
    assert len(found) == SOURCES[source]
    pinned = [name for name, body in found.items() if any(a and "mfma" in t for t, a in body)]
    assert len(pinned) == sum("kv_fused" in name or "pinned" in name for name in found)
    assert {name: wrong for name, body in found.items() if (wrong := problems(body))} == {}


CLEAN = """_Zkernel:
\tv_mov_b32_e32 v9, 0
\t;;#ASMSTART
\tbuffer_load_dwordx4 v[4:7], v9, s[0:3], 0 offen offset:0
\t;;#ASMEND
.LBB0_1:
\tv_add_f32_e32 v2, v0, v1
\t;;#ASMSTART
\ts_waitcnt vmcnt(2)
\t;;#ASMEND
\tv_mul_f32_e32 v3, v4, v5
\ts_nop 1
\t;;#ASMSTART
\tv_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]
\t;;#ASMEND
\t;;#ASMSTART
\tbuffer_load_dwordx4 v[4:7], v9, s[0:3], 0 offen offset:0
\t;;#ASMEND
\tv_mov_b32_e32 v8, v9
\ts_cbranch_scc1 .LBB0_1
\ts_endpgm
"""


@pytest.mark.parametrize(
    "old,new,expected",
    [
        ("", "", None),
        ("v_mov_b32_e32 v8, v9", "v_accvgpr_write_b32 a3, v9", "accumulator"),
        ("v_mov_b32_e32 v8, v9", "v_accvgpr_write_b32 a16, v9", None),
        ("v_mov_b32_e32 v8, v9", "v_mov_b32_e32 v8, v5", "under way"),
        ("v_add_f32_e32 v2, v0, v1", "scratch_store_dwordx4 off, v[6:9], off", "under way"),  # (reached by the branch back)
        ("s_nop 1", "s_nop 0", "right ahead"),
        ("\ts_nop 1\n", "", "right ahead"),
        ("s_nop 1", "v_permlane32_swap_b32 v8, v1", "right ahead"),
    ],
)
def test_the_check_sees_what_it_looks_for(old, new, expected):
    (body,) = kernels(CLEAN.replace(old, new) if old else CLEAN).values()
    wrong = problems(body)
    assert (not wrong) if expected is None else any(expected in w for w in wrong)
