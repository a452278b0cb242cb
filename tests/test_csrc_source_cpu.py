"""The kernels' and entry points' source: what the compiler does not check.

The compiler treats an asm statement as one opaque instruction.  A register it writes
must be named as clobbered, and the wait states that the hardware asks for between its
operands' writers and its own memory instruction must be inside it.  An entry point may
be called by any thread, so a value that a function keeps is initialised where it is
declared.
"""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "hybrid_llm_amd" / "csrc"
ASM = re.compile(r"\basm\s+volatile\s*\((.*?)\)\s*;", re.S)


def _statements():
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.hpp")):
        for m in ASM.finditer(path.read_text()):
            yield path.name, m.group(1)


def _template(stmt: str) -> list[str]:
    """The instructions of a statement (its leading string literals)."""
    text = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', stmt.split(":")[0]))
    return [i.strip() for i in re.split(r"\\n|\\t|;", text) if i.strip()]


def test_m0_writes_are_clobbers():
    seen = 0
    for name, stmt in _statements():
        if any(re.match(r"s_mov_b32\s+m0\b", i) for i in _template(stmt)):
            seen += 1
            assert '"m0"' in stmt.rsplit(":", 1)[1], (name, stmt)
    assert seen >= 2  # the LDS copies of the gated delta rule


def test_buffer_loads_wait_for_their_descriptor():
    """Five wait states between a VALU write of an SGPR and a vector memory instruction
    that reads it: whatever the compiler placed before the statement, its own
    instructions before the load must make them up."""
    seen = 0
    for name, stmt in _statements():
        waits = 0
        for ins in _template(stmt):
            if ins.startswith("buffer_load"):
                seen += 1
                assert waits >= 5, (name, stmt)
            nop = re.match(r"s_nop\s+(\d+)", ins)
            waits += int(nop.group(1)) + 1 if nop else 1
    assert seen >= 2


def test_function_statics_are_initialised_once():
    """A function-local ``static`` scalar that is filled in later is read and written by
    every thread that calls; const ones are initialised under the language's guard."""
    for path in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.hpp")) + sorted(CSRC.glob("*.cpp")):
        for line in path.read_text().splitlines():
            assert not re.match(r"\s+static\s+(int|bool|long long|unsigned|void\s*\*)\s+\w+\s*=", line), (
                path.name, line)
