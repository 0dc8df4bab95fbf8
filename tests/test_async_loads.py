"""What the compiler has to be told about the kernels' inline assembly, checked in the sources: it neither counts the
asynchronous loads into LDS nor sees which registers an asm statement writes unless the statement says so, and it keeps no
distance between instructions inside one."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mamba_amd", "csrc")


def _asm_statements():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h*"))):
        src = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"\basm\s+volatile\s*\((.*?)\)\s*;", src, flags=re.S):
            yield os.path.basename(path), m.group(1)


def test_asm_that_writes_m0_says_so():
    writers = [(f, a) for f, a in _asm_statements() if re.search(r"s_mov_b32 m0\b", a)]
    assert writers
    for f, a in writers:
        assert '"m0"' in a.rsplit(":", 1)[1], f"{f}: {a}"


def test_asm_that_reads_memory_through_a_scalar_base_waits_for_it():
    # five wait states from a vector instruction that writes a scalar register to a vector memory instruction that reads it
    # (gfx9): every instruction before the access is one, s_nop n is n + 1
    seen = 0
    for f, a in _asm_statements():
        text = "".join(re.findall(r'"([^"]*)"', a.split(":")[0])).replace("\\t", "")
        states = 0
        for inst in filter(None, text.split("\\n")):
            if re.match(r"(global|buffer|flat|scratch)_", inst) and re.search(r'"s"', a):
                seen += 1
                assert states >= 5, f"{f}: {text}"
            m = re.match(r"s_nop (\d+)", inst)
            states += int(m.group(1)) + 1 if m else 1
    assert seen
