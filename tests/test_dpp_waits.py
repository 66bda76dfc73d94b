"""
Inline assembly with DPP operands (lane broadcasts within rows): such an operand
may not be written by the two vector instructions before it, and the compiler,
which does not look into the assembly, may place the copy or reload of an operand
right before a statement. Every statement therefore holds two instructions or
wait states in front of its first DPP instruction, and none of its own writes of
a DPP operand comes closer. Read from the sources, with their macros expanded;
no GPU.
"""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "tad_dftd4_amd" / "csrc"


def _statements(path):
    """Instruction lists of the asm statements that hold a DPP instruction."""
    text = re.sub(r"^\s*#\s*(include|pragma).*$", "", path.read_text(), flags=re.M)
    text = subprocess.run(["g++", "-E", "-P", "-w", "-x", "c++", "-"], input=text, text=True,
                          capture_output=True, check=True).stdout
    for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", text):
        code = re.match(r'(?:\s*"(?:[^"\\]|\\.)*")*', text[m.end():]).group()
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', code)).replace("\\t", " ")
        ins = [i.strip() for i in code.split("\\n") if i.strip()]
        if any("_dpp" in i for i in ins):
            yield ins


def test_dpp_operands_are_waited_for():
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    found = 0
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")):
        for ins in _statements(path):
            found += 1
            slots, written = 0, {}  # wait states so far; operand -> slot after its write
            for i in ins:
                op, _, rest = i.partition(" ")
                if op == "s_nop":
                    slots += int(rest) + 1
                    continue
                args = [a.strip().split(" ")[0].lstrip("-") for a in rest.split(",")]
                if op.endswith("_dpp"):
                    assert slots - written.get(args[1], 0) >= 2, f"{path.name}: {ins}"
                slots += 1
                written[args[0]] = slots
    assert found >= 3
