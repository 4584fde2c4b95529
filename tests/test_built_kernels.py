"""The streaming GEMM kernels as they are built: what the compiler can not check for them, because their products and the loads beside
these are assembly it does not look into, and what it may not do to them. Read from the notes and the disassembly of the library's own
gfx950 code; no GPU needed."""
import os
import re
import shutil
import subprocess

import pytest

import skl_amd

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "llvm", "bin")
STREAMING = "gemm_mfma_ring_kernel"
PASSES = {"16x16x32_bf16": 4, "16x16x32_f16": 4, "16x16x64_i8": 4, "32x32x32_i8": 8, "32x32x64_f8f6f4": 16}  # of four cycles each


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    folder = tmp_path_factory.mktemp("code")
    library = shutil.copy(skl_amd.library_path(), folder / "library.so")
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", library], check=True, cwd=folder, capture_output=True)
    found = sorted(f for f in folder.iterdir() if f.name.endswith("gfx950") and f.stat().st_size)
    assert found
    return found


@pytest.fixture(scope="module")
def kernels(code_objects):
    """Name and instructions (mnemonic and operands, comments taken off) of every streaming kernel."""
    out = {}
    for obj in code_objects:
        text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", obj], check=True, capture_output=True, text=True).stdout
        for part in re.split(r"\n(?=[0-9a-f]{16} <)", text):
            name = re.match(r"[0-9a-f]{16} <([^>]*)>:", part)
            if name and STREAMING in name.group(1):
                out[name.group(1)] = [line.split("//")[0].strip() for line in part.split("\n")[1:] if line.startswith("\t")]
    assert len(out) > 100
    return out


def test_no_streaming_kernel_touches_scratch_memory(code_objects):
    """A scratch access behind the stores of C waits for all of them."""
    seen, bad = 0, []
    for obj in code_objects:
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", obj], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"\n  - \.agpr_count", notes)[1:]:
            value = lambda key: re.search(rf"\.{key}:\s+(\S+)", kernel).group(1)
            if STREAMING in value("name"):
                seen += 1
                if int(value("private_segment_fixed_size")) or int(value("vgpr_spill_count")):
                    bad.append(value("name"))
    assert seen > 100 and not bad, bad


def registers(operand):
    """The vector and accumulation registers of an operand, as (file, number)."""
    one = re.fullmatch(r"([va])(\d+)", operand)
    many = re.fullmatch(r"([va])\[(\d+):(\d+)\]", operand)
    if one:
        return {(one.group(1), int(one.group(2)))}
    return {(many.group(1), r) for r in range(int(many.group(2)), int(many.group(3)) + 1)} if many else set()


def operands(instruction):
    rest = instruction.split(None, 1)
    return re.findall(r"[va]\[\d+:\d+\]|\b[va]\d+\b", rest[1]) if len(rest) > 1 else []


def states(instruction):
    nop = re.fullmatch(r"s_nop (\d+)", instruction)
    return int(nop.group(1)) + 1 if nop else 1


def products(code):
    for at, instruction in enumerate(code):
        if instruction.startswith("v_mfma_"):
            yield at, PASSES[re.match(r"v_mfma_[fi]32_(\S+)", instruction).group(1)]


def latency(passes):
    """Wait states until anything but a product on the same registers may touch a product's result."""
    return passes + 4


def test_nothing_touches_a_sum_while_its_product_is_under_way(kernels):
    for name, code in kernels.items():
        for at, passes in products(code):
            result, waited = registers(operands(code[at])[0]), 0
            for instruction in code[at + 1:]:
                if waited >= latency(passes):
                    break
                if not instruction.startswith("v_mfma_"):
                    assert not any(registers(o) & result for o in operands(instruction)), (name, code[at], instruction)
                waited += states(instruction)


def test_operands_of_a_product_are_written_two_states_ahead(kernels):
    """By vector instructions; what comes from LDS is waited for."""
    for name, code in kernels.items():
        for at, _ in products(code):
            read, waited = set().union(*(registers(o) for o in operands(code[at])[1:])), 0
            for instruction in reversed(code[:at]):
                if waited >= 2:
                    break
                waited += states(instruction)
                if instruction.startswith("v_") and not instruction.startswith(("v_mfma_", "v_cmp")):
                    assert not registers(operands(instruction)[0] if operands(instruction) else "") & read, (name, instruction, code[at])


def test_the_loop_is_not_left_with_a_product_under_way(kernels):
    """From the last product of a loop to its end: what the compiler puts behind the loop may read any sum."""
    loops = 0
    for name, code in kernels.items():
        marks = list(products(code))
        for (at, passes), following in zip(marks, [m[0] for m in marks[1:]] + [len(code)]):
            waited = 0
            for instruction in code[at + 1:following]:
                if instruction.startswith("s_cbranch"):
                    loops += 1
                    assert waited >= latency(passes), (name, code[at], waited)
                    break
                waited += states(instruction)
    assert loops >= len(kernels)


def test_every_load_to_lds_has_its_m0_written_in_front_of_it(kernels):
    """Where loads are part of assembly, which writes M0 unseen, no M0 is held from one load to another."""
    seen = 0
    for name, code in kernels.items():
        loads = [at for at, x in enumerate(code) if re.match(r"(global_load_lds|buffer_load_\S+ .*\blds\b)", x)]
        if any(code[at].startswith("buffer_load") for at in loads):
            assert all(code[at].startswith("buffer_load") for at in loads), name  # all of them the compiler's
            continue
        for at in loads:
            seen += 1
            writes = [x for x in code[max(at - 2, 0):at] if re.match(r"s_\S+ m0,", x)]
            assert len(writes) == 1 and re.match(r"s_\S+ m0,", code[at - 2]), (name, code[at - 3:at + 1])
    assert seen


def test_both_ways_of_the_stores_are_there(kernels):
    """Stores of C through the caches and past them differ in one bit, and the compiler makes one of two branches that differ in it alone."""
    for name, code in kernels.items():
        past = sum(x.startswith("global_store_dwordx4") and x.endswith(" nt") for x in code)
        through = sum(x.startswith("global_store_dwordx4") and not x.endswith(" nt") for x in code)
        assert past and through, (name, past, through)
