"""What inline assembly in the kernels writes is declared: the compiler keeps values in every register that a statement
does not name, m0 and the condition codes among them."""

import re
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "distie_amd" / "csrc"

# registers that an instruction may name as its destination without an operand of the statement standing for them
FIXED = re.compile(r"\b(m0|vcc|exec|s\d+|v\d+|a\d+|s\[\d+:\d+\]|v\[\d+:\d+\]|a\[\d+:\d+\])$")


def statements(text):
    """-> (template, clobbers) of every asm statement"""
    for match in re.finditer(r"\basm\s+(?:volatile\s*)?\(", text):
        depth, end, quoted = 1, match.end(), False
        while depth:
            c = text[end]
            if c == '"' and text[end - 1] != "\\":
                quoted = not quoted
            if not quoted:
                depth += (c == "(") - (c == ")")
            end += 1
        body = text[match.end():end - 1]
        parts, at, quoted = [""], 0, False
        while at < len(body):                       # split at the colons outside of strings
            c = body[at]
            if c == '"' and body[at - 1:at] != "\\":
                quoted = not quoted
            if c == ":" and not quoted:
                parts.append("")
            else:
                parts[-1] += c
            at += 1
        parts += [""] * (4 - len(parts))
        template = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', parts[0])).replace("\\n", "\n").replace("\\t", " ")
        yield template, re.findall(r'"([^"]*)"', parts[3])


def undeclared(text):
    missing = []
    for template, clobbers in statements(text):
        for line in re.split(r"[\n;]", template):
            words = line.strip().split(None, 1)
            if len(words) < 2 or words[0].startswith(("s_waitcnt", "s_nop", "global_store", "ds_write")):
                continue
            target = FIXED.match(words[1].split(",")[0].strip())
            if target and target.group(1) not in clobbers:
                missing.append((line.strip(), target.group(1)))
    return missing


@pytest.mark.parametrize("path", sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")), ids=lambda path: path.name)
def test_registers_written_by_inline_assembly_are_declared(path):
    assert undeclared(path.read_text()) == []


def test_the_check_sees_an_undeclared_register():
    text = 'asm volatile("s_mov_b32 m0, %0\\n\\ts_nop 0\\n\\tglobal_load_lds_dwordx4 %1, off" ::"s"(at), "v"(p) : "memory"MORE);'
    assert [target for _, target in undeclared(text.replace("MORE", ""))] == ["m0"]
    assert undeclared(text.replace("MORE", ', "m0"')) == []


def test_what_other_workgroups_write_is_looked_for_in_memory_each_time(tmp_path):
    """In the compiler's own terms: wherever the kernel asks for such words, the same stretch of code says that memory may have
    changed, so that no look stands for the next one."""
    from distie_amd.csrc import build

    out = tmp_path / "layer_chain.ll"
    subprocess.run([build._hipcc(), *build.HIP_FLAGS, "-x", "hip", "--offload-device-only", "-emit-llvm", "-S",
                    str(CSRC / "layer_chain.hip"), "-o", str(out)], check=True, capture_output=True)
    kernels = [body[:body.index("\n}")] for body in re.split(r"^define ", out.read_text(), flags=re.MULTILINE)[1:]
               if "layer_chain_kernel" in body.split("\n", 1)[0]]
    assert len(kernels) == 6
    for body in kernels:
        blocks = [b for b in re.split(r"^\d+:.*\n", body, flags=re.MULTILINE) if "call" in b and "llvm.amdgcn.raw.buffer.load" in b]
        assert len(blocks) >= 4                        # x of a sum, x of a norm, and twice what a sum is added to
        assert all('asm sideeffect "", "~{memory}"' in b[:b.index("llvm.amdgcn.raw.buffer.load")] for b in blocks)
