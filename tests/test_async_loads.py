"""What the compiler has to be told about the kernels' inline assembly, checked in the sources: it neither counts the
asynchronous loads into LDS nor sees which registers an asm statement writes unless the statement says so, and it keeps no
distance between instructions inside one."""
import glob
import os
import re
import subprocess

import pytest

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


def _fewest_behind(lines):
    """Over the paths from an asynchronous load to a counted wait of the source (async_done): the fewest vector memory
    operations on the way, less the number that the wait lets stay in flight.  A path ends where the source waits for
    everything; the compiler's own waits, of which it may make fewer, are left out of account.  A branch over an empty set
    of lanes is not taken: at a full chunk every wave has lanes in every store and add, by the conditions in the source."""
    label = {m.group(1): k for k, l in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", l))}
    best, todo = None, [(0, k + 1) for k, l in enumerate(lines) if l.startswith("global_load_lds")]
    seen = {}
    while todo:
        n, k = min(todo)
        todo.remove((n, k))
        while k < len(lines) and seen.get(k, n + 1) > n:
            seen[k] = n
            l = lines[k]
            m = re.match(r"s_waitcnt vmcnt\((\d+)\)", l)
            if m and lines[k - 1] == ";;#ASMSTART":
                if int(m.group(1)) > 0:
                    best = n - int(m.group(1)) if best is None else min(best, n - int(m.group(1)))
                break
            if re.match(r"(global|flat|buffer|scratch)_(load|store|atomic)", l):
                n += 1
            elif m := re.match(r"s_(c?branch)(\w*)\s+(\.LBB\w+)", l):
                if m.group(1) == "branch":
                    k = label[m.group(3)]
                    continue
                if m.group(2) != "_execz":
                    todo.append((n, label[m.group(3)]))
            elif l.startswith("s_endpgm"):
                break
            k += 1
    return best


def _kernels(name, kernel, tmp_path):
    from mamba_amd import build
    out = tmp_path / "k.s"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, name + ".hip"),
                    "-o", str(out)], check=True, capture_output=True)
    for m in re.finditer(r"^(_Z\w*%s\w*):(.*?)^\s*\.section" % kernel, out.read_text(), flags=re.S | re.M):
        lines = [l.split("; ")[0].strip() for l in m.group(2).splitlines()]
        yield m.group(1), [l for l in lines if l and not re.match(r"\.(?!LBB)|;(?!;#ASM)", l)]


@pytest.mark.parametrize("name,kernel", [("ssd_dx_fused", "bwd_dx_fused_kernel"), ("ssd_scan_group", "chunk_scan_fwd_group_kernel")])
def test_counted_waits_cover_the_loads(name, kernel, tmp_path):
    counted = 0
    for kernel_name, lines in _kernels(name, kernel, tmp_path):
        assert any(l.startswith("global_load_lds") for l in lines)
        counted += sum(lines[k] == ";;#ASMSTART" and bool(re.match(r"s_waitcnt vmcnt\([1-9]", lines[k + 1])) for k in range(len(lines) - 1))
        behind = _fewest_behind(lines)
        assert behind is None or behind >= 0, kernel_name
    assert counted


def _operations(lines):
    """(kind, count) of what a wait on vector memory counts, of the source's own waits, and of barriers, in order."""
    for k, l in enumerate(lines):
        if m := re.match(r"global_load_lds_dword(x4)?\b", l):
            yield "rows" if m.group(1) else "table", 1
        elif re.match(r"(global|flat|buffer|scratch)_(load|store|atomic)", l):
            yield "other", 1
        elif (m := re.match(r"s_waitcnt vmcnt\((\d+)\)", l)) and lines[k - 1] == ";;#ASMSTART":
            yield "wait", int(m.group(1))
        elif l.startswith("s_barrier"):
            yield "barrier", 0


def test_counted_waits_of_the_state_walk(tmp_path):
    # A ring of stages: the rows that a stage waits for were asked for `ahead` stages before, the table's entries in the chunk's
    # first stage.  Over three rounds of the loop over the chunks, each wait leaves no more in flight than what came behind them.
    seen = 0
    for name, lines in _kernels("ssd_fwd", "chunk_state_passing_fwd_kernel", tmp_path):
        heads, stages = map(int, re.search(r"ILi(\d)ELi(\d)E", name).groups())
        ahead = 2 if heads == 1 else 3
        label = {m.group(1): k for k, l in enumerate(lines) if (m := re.match(r"(\.LBB\w+):", l))}
        back = [(label[m.group(1)], k) for k, l in enumerate(lines) if (m := re.match(r"s_c?branch\w*\s+(\.LBB\w+)", l)) and label[m.group(1)] < k]
        body = next(ops for a, b in back if len(ops := list(_operations(lines[a:b]))) > 8)
        done, asked, table, waits = 0, [[]], [], 0     # operations so far; those of each stage's rows; of the table
        for turn in range(3):
            for k, (kind, n) in enumerate(body):
                if kind in ("rows", "table", "other"):
                    done += 1
                    (asked[-1] if kind == "rows" else table if kind == "table" else []).append(done)
                elif kind == "wait":
                    waits += 1
                    if body[k + 1][0] == "barrier":
                        if len(asked) > ahead:
                            assert done - asked[-ahead][-1] >= n > 0, (name, turn, k)
                        asked.append([])
                    else:
                        assert done - table[-1] >= n > 0, (name, turn, k)
        assert waits == 3 * (stages + 1) and len({len(a) for a in asked[1:]}) == 1, name
        seen += 1
    assert seen == 8
