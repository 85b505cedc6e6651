"""The kernels' inline assembly names every register it uses by number or name
among its clobbers (an operand's register is the compiler's choice), or, m0,
which no clobber list takes, keeps it at its start and puts it back at its
end."""
import os
import re
import subprocess

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "physim_amd",
                   "csrc", "pg_kernels.h")


def statements():
    """(code, clobbers) of every asm statement, macros expanded."""
    text = open(SRC).read()
    text = re.sub(r"^\s*#\s*include.*$", "", text, flags=re.M)
    out = subprocess.run(["g++", "-E", "-P", "-x", "c++", "-"], input=text, text=True,
                         capture_output=True, check=True).stdout
    for m in re.finditer(r"\basm\s+volatile\s*\(|\basm\s*\(", out):
        depth, i, quoted = 1, m.end(), False
        parts = [""]  # the statement split at its colons
        while depth:
            c = out[i]
            if c == '"' and out[i - 1] != "\\":
                quoted = not quoted
            if not quoted:
                depth += {"(": 1, ")": -1}.get(c, 0)
            if c == ":" and not quoted and depth == 1:
                parts.append("")
            elif depth:
                parts[-1] += c
            i += 1
        code = "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', parts[0]))
        yield code.replace("\\n", "\n").replace("\\t", " "), set(
            re.findall(r'"([^"]*)"', parts[3])) if len(parts) > 3 else set()


def registers(code):
    named = set()
    for line in code.split("\n"):
        line = re.sub(r"%\[?\w+\]?|Lw\w*%?=?|/\*.*?\*/", " ", line)
        for kind, a, b in re.findall(r"\b([sva])\[(\d+):(\d+)\]", line):
            named |= {f"{kind}{r}" for r in range(int(a), int(b) + 1)}
        named |= set(re.findall(r"\b([sv]\d+|m0|vcc|exec)\b", line))
    return named


def test_named_registers_are_clobbered():
    seen = 0
    for code, clobbers in statements():
        used = registers(code)
        seen += len(used)
        first, last = code.strip().split("\n")[0], code.strip().split("\n")[-1]
        keep = re.fullmatch(r"\s*s_mov_b32 (%\[\w+\]), m0\s*", first)
        if keep and re.fullmatch(rf"\s*s_mov_b32 m0, {re.escape(keep[1])}\s*", last) \
                and code.count(keep[1]) == 2:
            used -= {"m0"}
        assert used <= clobbers, (sorted(used - clobbers), code[:200])
    assert seen >= 3 * 20  # (the walk's loop in its three forms is among them)
