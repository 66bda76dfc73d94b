"""
Inline assembly with DPP operands (lane broadcasts within rows): such an operand
may not be written by the two vector instructions before it, and the compiler,
which does not look into the assembly, may place the copy or reload of an operand
right before a statement. Every statement therefore holds two instructions or
wait states in front of its first DPP instruction, and none of its own writes of
a DPP operand comes closer. Read from the sources; no GPU.
"""

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "tad_dftd4_amd" / "csrc"
FMAC = re.compile(r'D4_FMAC\("([^"]*)", "([^"]*)", "([^"]*)", "([^"]*)"\)')


def _statements(text):
    """Instruction lists of the asm statements that hold a DPP instruction."""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"\basm\s*(?:volatile\s*)?\(", text):
        body = text[m.end():text.index(";\n", m.end())]
        body = FMAC.sub(r'"v_fmac_f64_dpp \1, \2, \3 row_newbcast:\4\\n\\t"', body)
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', re.split(r"\n\s*:", body)[0]))
        ins = [i.strip() for i in code.replace("\\t", " ").split("\\n") if i.strip()]
        if any("_dpp" in i for i in ins):
            yield ins


def test_dpp_operands_are_waited_for():
    found = 0
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.h")):
        for ins in _statements(path.read_text()):
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
    assert found >= 11
