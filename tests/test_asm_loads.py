"""Loads written in inline asm (csrc/): the compiler takes an asm statement's outputs as written when the statement ends, so a load
that returns a register must be waited for in its own statement."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "csrc"
LOAD = re.compile(r"\b(global_load|flat_load|buffer_load|scratch_load|ds_read|ds_load|s_load|s_buffer_load)_(?!lds)\w+")


def statements(text):
    for m in re.finditer(r"\basm\s*(?:volatile|__volatile__)?\s*\(", text):
        depth, i, quoted = 1, m.end(), False
        while depth:
            c = text[i]
            if c == '"' and text[i - 1] != "\\":
                quoted = not quoted
            elif not quoted:
                depth += (c == "(") - (c == ")")
            i += 1
        yield text[m.start():i]


def test_loads_wait_in_their_own_statement():
    seen = 0
    for f in sorted(CSRC.rglob("*")):
        if f.suffix not in (".hip", ".h", ".cpp"):
            continue
        for s in statements(f.read_text()):
            code = " ".join(re.findall(r'"((?:[^"\\]|\\.)*)"', s))
            loads = LOAD.findall(code)
            if not loads:
                continue
            seen += 1
            last = max(m.end() for m in LOAD.finditer(code))
            assert "s_waitcnt" in code[last:], f"{f.name}: {s[:120]}"
            assert all('"=&' in o for o in re.findall(r'"=[^"]*"', s)), f"{f.name}: outputs share registers with addresses"
    assert seen  # (the fused GEMM epilogues')
