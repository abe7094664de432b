"""What the source does not give by itself, checked on the machine code of the built library. The compiler counts no wait states in front
of an SMFMAC in inline assembly: no vector instruction writes an operand of one of gemm_kernel's less than two wait states in front of
it. Layers without a bias pass none of a bias's code in front of wide_kernel's barrier. The first image's eight loads of tokens are spaced."""
import os
import re
import subprocess

import pytest

from onebitsparsemul_amd import build as native_build

NEEDED = 2  # wait states from a vector instruction's write to an SMFMAC's read of the register
REGISTER = re.compile(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+))")


def registers(text):
    return {(kind, i) for kind, low, high, one in REGISTER.findall(text) for i in range(int(low or one), int(high or one) + 1)}


def too_close(code):
    """(SMFMAC, write) line pairs of one function's code, [(address, instruction, operands, branch target or None)]"""
    at = {line[0]: i for i, line in enumerate(code)}
    jumps = {}
    for i, (_, _, _, target) in enumerate(code):
        if target in at:
            jumps.setdefault(at[target], []).append(i)

    def writes(i, operands, states):
        """vector instructions that write one of `operands` and reach instruction i within less than `states` wait states"""
        falls = [i - 1] if i > 0 and code[i - 1][1] not in ("s_branch", "s_endpgm") else []
        for j in falls + jumps.get(i, []):
            _, name, rest, _ = code[j]
            if name.startswith("v_") and "mfma" not in name and "smfmac" not in name:
                if registers(rest if "swap" in name else rest.split(",")[0]) & operands:
                    yield j
                    continue
            passed = int(rest, 0) + 1 if name == "s_nop" else 1
            if passed < states:
                yield from writes(j, operands, states - passed)

    return [(code[i][1:3], code[j][1:3]) for i, line in enumerate(code) if "smfmac" in line[1]
            for j in writes(i, registers(line[2]), NEEDED)]


def functions(text):
    """name and code of each function of a disassembly"""
    for part in re.split(r"^(?=[0-9a-f]{16} <)", text, flags=re.M)[1:]:
        head, *lines = part.splitlines()
        start, code = int(head[:16], 16), []
        for line in lines:
            found = re.match(r"\s+(\w+)(.*?)\s*// ([0-9A-F]{12}): [0-9A-F ]+(?:<[^+>]+(?:\+0x([0-9a-f]+))?>)?", line)
            if found:
                branch = found[1].startswith(("s_cbranch", "s_branch"))
                code.append((int(found[3], 16), found[1], found[2], start + int(found[4] or "0", 16) if branch else None))
        yield head[18:-2], code


def test_the_check_finds_a_write_that_is_too_close():
    smfmac = (12, "v_smfmac_f32_32x32x32_f16", " a[0:15], v[6:9], v[10:17], v5", None)
    for write in ((0, "v_mov_b64_e32", " v[4:5], v[2:3]", None), (0, "v_accvgpr_write_b32", " a15, v1", None)):
        wait = (4, "s_setprio", " 1", None)
        assert too_close([write, smfmac]) and too_close([write, wait, smfmac])
        assert not too_close([write, wait, (8, "s_nop", " 0", None), smfmac]) and not too_close([write, (4, "s_nop", " 1", None), smfmac])
        # around a loop
        assert too_close([(8, "s_nop", " 3", None), smfmac, write, (20, "s_cbranch_scc1", " 1", 12)])
    assert not too_close([(0, "v_mov_b32_e32", " v4, v5", None), smfmac])


def disassembly(source, folder):
    """functions() of one object of the built library"""
    llvm = os.path.join(os.path.dirname(native_build.HIPCC), "..", "llvm", "bin")
    subprocess.run(["ar", "x", native_build.STATIC_LIB, source], cwd=folder, check=True)
    subprocess.run([os.path.join(llvm, "llvm-objdump"), "--offloading", source], cwd=folder, check=True, stdout=subprocess.DEVNULL)
    (device,) = [name for name in os.listdir(folder) if name.endswith("gfx950")]
    return functions(subprocess.run([os.path.join(llvm, "llvm-objdump"), "-d", device], cwd=folder, check=True, capture_output=True,
                                    text=True).stdout)


@pytest.mark.parametrize("source", ["onebit_gemm.o", "onebit_gemm_tokens.o"])
def test_operands_of_inline_smfmacs_are_written_early_enough(source, tmp_path):
    kernels = {name: code for name, code in disassembly(source, tmp_path) if "gemm_kernel" in name}
    assert len(kernels) >= 18 and sum("smfmac" in line[1] for code in kernels.values() for line in code) > 2000
    assert sum(line[3] is not None for code in kernels.values() for line in code) > 100  # branches with their targets
    for name, code in kernels.items():
        assert not too_close(code), name


def test_layers_without_a_bias_pass_none_of_its_code_in_front_of_the_barrier(tmp_path):
    """wide_kernel's token-major form: a bias is read by loads that are not taken for LDS reads, on a path of its own: behind the barrier
    that calls without one pass, in front of its own, where the reads of the sums do not wait for it"""
    kernels = [(name, code) for name, code in disassembly("onebit_wide_tokens.o", tmp_path) if "wide_kernel" in name]
    assert len(kernels) >= 24
    for name, code in kernels:
        names = [line[1] for line in code]
        # (the copies of x go to LDS: global_load_lds_...)
        bias = [i for i, n in enumerate(names) if n.startswith(("flat_load", "global_load_dword", "global_load_ushort"))]
        assert bias and not any(names[i].startswith("flat") for i in bias) and min(bias) > names.index("s_barrier"), name
        behind = [n for n in names[min(bias):] if n == "s_barrier" or n.startswith("ds_read")]
        assert behind[0] == "s_barrier", name


def test_eight_loads_of_tokens_are_spaced_ahead_of_the_loop(tmp_path):
    """skinny_kernel on eight wavefronts, thirteen to sixteen tokens: all at once they cost 3 % (10624 x 5024 with 16 6.91 us, 6.63 spaced)"""
    found = 0
    for name, code in disassembly("onebit_skinny_tokens.o", tmp_path):
        if re.search(r"skinny_kernelILi8ELi[24]ELi40E", name):
            lines = [line[1] + line[2] for line in code if line[1] == "s_nop" or line[1].startswith("buffer_load_dwordx4")]
            text = " ".join("n" if line.split() == ["s_nop", "15"] else "l" if line.startswith("buffer") else "" for line in lines)
            assert "n l n l n l n l n l n l n l" in re.sub(" +", " ", text), name
            found += 1
    assert found == 4  # 64- and 128-row groups, fp16 and bf16
