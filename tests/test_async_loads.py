"""What the compiler has to be told about the kernels' inline assembly, checked in the sources: it neither counts the
asynchronous loads into LDS nor sees which registers an asm statement writes unless the statement says so."""
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
