"""What inline assembly writes it has to tell the compiler, and what the compiler's hazard recogniser does for an
instruction it has to do by itself: both go unnoticed until a build in which something else uses the register."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tsne-cuda_amd", "csrc")


def statements():
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".h")):
            continue
        with open(os.path.join(CSRC, name)) as f:
            text = f.read()
        for at in re.finditer(r"\basm\s+volatile\s*\(", text):
            end, depth, quoted = at.end(), 1, False
            while depth:
                c = text[end]
                quoted ^= c == '"' and text[end - 1] != "\\"
                depth += 0 if quoted else (c == "(") - (c == ")")
                end += 1
            yield name, text[at.end():end - 1]


def parts(statement):
    """(instructions, operands and clobbers) of a statement."""
    code = re.match(r'\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', statement)
    lines = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', code.group(1))).replace("\\t", " ").split("\\n")
    return [line.split(None, 1) for line in lines if line.strip()], statement[code.end():]


FOUND = [(name, s) for name, s in statements() if parts(s)[0]]


def test_statements_are_found():
    assert any("global_load_lds" in s for _, s in FOUND)


@pytest.mark.parametrize("name,statement", FOUND)
def test_fixed_registers_are_clobbered(name, statement):
    """A register that an instruction writes by name (m0, vcc, exec, s7, v[0:3]) is among the clobbers."""
    instructions, rest = parts(statement)
    clobbers = set(re.findall(r'"([^"]*)"', rest.split(":")[-1]))
    for mnemonic, operands in ((i + [""])[:2] for i in instructions):
        written = operands.split(",")[0].strip()
        if re.match(r"(m0|vcc|exec|scc|[sva]\d|[sva]\[)", written) and not mnemonic.startswith(("s_cmp", "global_store")):
            assert written in clobbers, "%s: '%s %s' writes %s behind the compiler's back" % (name, mnemonic, operands, written)


@pytest.mark.parametrize("name,statement", FOUND)
def test_addresses_of_loads_are_formed_on_the_scalar_unit(name, statement):
    """A memory instruction's scalar address comes from a scalar instruction of the same statement."""
    instructions, _ = parts(statement)
    scalar = set()
    for mnemonic, operands in ((i + [""])[:2] for i in instructions):
        operands = [o.strip() for o in operands.split(",")]
        if mnemonic.startswith(("global_", "buffer_", "flat_")):
            assert scalar & set(operands[1:]), "%s: address of '%s' may come from a vector instruction" % (name, mnemonic)
        elif mnemonic.startswith("s_"):
            scalar.add(operands[0])
