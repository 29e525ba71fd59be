"""Rules of the device sources that no run can show: a breach works until the compiler's register
allocation happens to change."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _asm_blocks():
    for path in sorted(glob.glob(os.path.join(ROOT, "fastermoe_amd", "csrc", "*"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"\basm\s+volatile\s*\((.*?)\)\s*;", text, flags=re.S):
            yield os.path.basename(path), m.group(1)


def test_inline_asm_names_the_special_registers_it_writes():
    """m0 (the LDS address of a direct-to-LDS load) and scc (the result of scalar compares and additions) in the
    clobber list of every asm statement that changes them."""
    seen = 0
    for name, body in _asm_blocks():
        strings = re.findall(r'"((?:[^"\\]|\\.)*)"', body)
        code = [line.strip() for s in strings for line in re.split(r"\\n(?:\\t)?", s)]
        if any(re.match(r"s_\w+\s+m0\b", line) for line in code):
            seen += 1
            assert "m0" in strings, f"{name}: {body}"
        if any(re.match(r"s_(cmp|add|sub|and|or|lshl|lshr)\w*\s", line) for line in code):
            assert "scc" in strings, f"{name}: {body}"
    assert seen >= 3
