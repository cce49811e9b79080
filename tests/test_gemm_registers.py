"""What the grouped GEMMs need of the generated code and no result shows reliably.

The column-wave kernels keep their weight fragments in registers that the compiler does not know to be in
use (the asynchronous loads and the MFMAs name them in their assembly text).  That is only sound if the compiler itself never
touches those registers and never spills in the item loop (a reload from the stack waits for every copy in flight).

In the few-rows kernels nothing but another MFMA may touch an accumulator until its MFMA has settled (19 wait states), on any
way through the code; the compiler counts an s_waitcnt as a state, which it is not when nothing is left to wait for.

Checked here on the code the build actually generates: megamoe.hip compiled to assembly with the build's own flags (no GPU
needed)."""

import os
import re
import shutil
import subprocess

import pytest

from deepep_amd import build

SOURCE = os.path.join(build.CSRC, "megamoe.hip")


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    hipcc = build._hipcc()
    if shutil.which(hipcc) is None and not os.path.exists(hipcc):
        pytest.skip("hipcc is not installed")
    out = tmp_path_factory.mktemp("isa") / "megamoe.s"
    flags = [f for f in build.FLAGS if f != "-fPIC"] + list(build.FILE_FLAGS.get("megamoe.hip", ()))
    proc = subprocess.run([hipcc, *flags, "--cuda-device-only", "-S", "-o", str(out), SOURCE], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr[-2000:]
    return out.read_text().split("\n")


def _kernels(lines, kernel="grouped_gemm_colwave_kernel"):
    """name -> (body lines, bytes of stack) of every instance of a kernel."""
    text = "\n".join(lines)
    found = {}
    for match in re.finditer(r"\.amdhsa_kernel (\S*" + kernel + r"\S*)(.*?)\.end_amdhsa_kernel", text, re.S):
        name, meta = match.group(1), match.group(2)
        start = next(i for i, line in enumerate(lines) if line.startswith(name + ":"))
        end = next(i for i in range(start, len(lines)) if lines[i].strip().startswith(".amdhsa_kernel"))
        scratch = int(re.search(r"\.amdhsa_private_segment_fixed_size\s+(\d+)", meta).group(1))
        found[name] = (lines[start:end], scratch)
    return found


def _numbers(text, file):
    singles = [int(x) for x in re.findall(r"\b" + file + r"(\d+)\b", text)]
    ranges = [int(v, 0) for pair in re.findall(r"\b" + file + r"\[(\w+):(\w+)\]", text) for v in pair]
    return singles + ranges


def test_weight_registers_belong_to_the_assembly_statements_alone(assembly):
    kernels = _kernels(assembly)
    assert len(kernels) == 6  # three tile heights x {first, second} GEMM
    for name, (body, scratch) in kernels.items():
        rows = int(re.search(r"kernelILi(\d)", name).group(1))
        # 64 / 128 rows: a64.. / a128.., right behind the accumulators; 192 rows: v192..v255
        file, first = ("v", 192) if rows == 3 else ("a", 64 * rows)
        in_statement, outside, in_loads, accumulators = False, [], set(), []
        for line in body:
            text = line.strip()
            if text.startswith(";;#ASMSTART"):
                in_statement = True
            elif text.startswith(";;#ASMEND"):
                in_statement = False
            elif in_statement:
                if text.startswith("global_load_dwordx4"):
                    in_loads.update(_numbers(text.split(",")[0], file))
                if text.startswith("v_mfma"):
                    accumulators += _numbers(text.split(",")[0], "a")
            elif any(first <= r < first + 64 for r in _numbers(text, file)):
                outside.append(text)
        assert not outside, f"{name}: the compiler uses weight registers itself: {outside[:3]}"
        assert in_loads and min(in_loads) == first and max(in_loads) == first + 63, (name, sorted(in_loads)[:4])
        assert max(accumulators) == 64 * rows - 1, f"{name}: accumulators reach a{max(accumulators)}"
        assert scratch == 0, f"{name}: {scratch} bytes of stack (a reload in the item loop waits for all copies in flight)"


SETTLED = 19  # wait states from a 16-pass MFMA to the first other instruction that may touch its result


def _registers(text):
    """(file, number) of every vector register that an instruction's operands name."""
    found = set()
    for file, low, high in re.findall(r"\b([va])\[(\d+):(\d+)\]", text):
        found.update((file, r) for r in range(int(low), int(high) + 1))
    found.update((file, int(r)) for file, r in re.findall(r"\b([va])(\d+)\b", text))
    return found


def _touched_too_early(body):
    """(MFMA, instruction, wait states between) of every non-MFMA instruction that touches an MFMA's result too early, along
    every way through the code.  s_nop N is N + 1 states, s_waitcnt none, any other instruction one."""
    code, labels = [], {}
    for line in body:
        text = line.split(";")[0].strip()
        label = re.match(r"(\.LBB\w+):", text)
        if label:
            labels[label.group(1)] = len(code)
        elif text and not text.startswith(".") and not text.endswith(":"):
            code.append(text)
    found = []
    for at, text in enumerate(code):
        if not text.startswith("v_mfma"):
            continue
        result = _registers(text.split(",")[0])
        ways, seen = [(at + 1, 0)], {}
        while ways:
            here, states = ways.pop()
            while here < len(code) and states < SETTLED and seen.get(here, SETTLED) > states:
                seen[here] = states
                step = code[here]
                if step.startswith("v_mfma"):
                    operands = step.split(None, 1)[1].split(", ")
                    if _registers(operands[0]) == result:
                        break  # written anew (or added to, which the pipe itself orders): from here on that MFMA's matter
                    if result & _registers(", ".join(operands[:3])):
                        found.append((text, step, states))
                elif result & _registers(step):
                    found.append((text, step, states))
                if step.startswith("s_endpgm"):
                    break
                target = re.match(r"s_c?branch\w*\s+(\.LBB\w+)", step)
                nop = re.match(r"s_nop (\d+)", step)
                states += int(nop.group(1)) + 1 if nop else 0 if step.startswith("s_waitcnt") else 1
                if target:
                    ways.append((labels[target.group(1)], states))
                    if step.startswith("s_branch"):
                        break
                here += 1
    return found


def test_accumulators_of_the_few_rows_kernels_settle_before_anything_else_touches_them(assembly):
    kernels = _kernels(assembly, "grouped_gemm_few_rows_kernel")
    assert len(kernels) == 4  # {one, four waves per workgroup} x {first, second} GEMM
    for name, (body, scratch) in kernels.items():
        assert sum(line.strip().startswith("v_mfma") for line in body) >= 32, name
        assert not _touched_too_early(body), (name, _touched_too_early(body)[:3])
        assert scratch == 0, f"{name}: {scratch} bytes of stack"


def test_the_check_finds_an_accumulator_that_is_touched_too_early(assembly):
    """The kernel's own waits taken out of its text (the compiler's stay): the moves and conversions behind the last MFMAs of
    some way through the code then come too early; and a small piece of code with a branch in it."""
    flagged = 0
    for body, _ in _kernels(assembly, "grouped_gemm_few_rows_kernel").values():
        without = [line for line in body if line.strip() not in ("s_nop 15",)]
        assert len(without) < len(body)
        flagged += bool(_touched_too_early(without))
    assert flagged > 0
    piece = ["v_mfma_f32_32x32x64 v[0:15], v[20:27], v[30:33], v[0:15]", "s_nop 15", "s_cbranch_scc1 .LBB0_2", "s_nop 1",
             ".LBB0_2:", "s_waitcnt vmcnt(0)", "v_mov_b32_e32 v40, v15"]
    assert [(found[1], found[2]) for found in _touched_too_early(piece)] == [("v_mov_b32_e32 v40, v15", 17)]
    assert not _touched_too_early(piece[:2] + ["s_nop 1"] + piece[2:])


def test_registers_of_the_paired_kernel_belong_to_its_assembly_statements_alone(assembly):
    """Accumulators (a0..a127, all there are with two workgroups to a CU) and weight fragments (v96..v127)."""
    kernels = _kernels(assembly, "grouped_gemm_paired_kernel")
    assert len(kernels) == 4  # {cached, streamed weights} x {first, second} GEMM
    for name, (body, scratch) in kernels.items():
        in_statement, outside, in_loads, accumulators = False, [], set(), set()
        for line in body:
            text = line.split(";")[0].strip() if not line.strip().startswith(";;#") else line.strip()
            if text.startswith(";;#ASMSTART"):
                in_statement = True
            elif text.startswith(";;#ASMEND"):
                in_statement = False
            elif in_statement:
                if text.startswith("global_load_dwordx4"):
                    in_loads.update(_numbers(text.split(",")[0], "v"))
                if text.startswith("v_mfma"):
                    accumulators.update(_numbers(text.split(",")[0], "a"))
            elif _numbers(text, "a") or any(r >= 96 for r in _numbers(text, "v")):
                outside.append(text)
        assert not outside, f"{name}: the compiler uses the kernel's own registers: {outside[:3]}"
        assert min(in_loads) == 96 and max(in_loads) == 127 and min(accumulators) == 0 and max(accumulators) == 127
        assert scratch == 0, f"{name}: {scratch} bytes of stack"
