"""Wait states between a matrix product and the first other use of its result registers, over
all paths of the built kernels' control flow.

The hardware does not hold back a vector, LDS or memory instruction that touches the result of
a matrix product still in the pipeline; the compiler places enough instructions or s_nop between
them.  After v_mfma_f32_16x16x32 it needs 8 wait states (what it inserts in straight-line code).
Where some blocks between a product and the use rewrite only part of the accumulators it has
missed the shortest path, so the distance is checked here and not taken for granted.
"""
import heapq
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from platoanalyze_amd import build

NEED = 8


def registers(operand):
    m = re.search(r"\b([va])\[(\d+):(\d+)\]", operand)
    if m:
        return {(m[1], k) for k in range(int(m[2]), int(m[3]) + 1)}
    m = re.search(r"\b([va])(\d+)\b", operand)
    return {(m[1], int(m[2]))} if m else set()


def functions(text):
    """Per function its instructions [(opcode, operands)] and their successors."""
    out, name = {}, None
    for line in text.splitlines():
        line = line.split(";")[0].rstrip()
        if re.match(r"\w+:$", line):
            name = line[:-1]
            out[name] = ([], {})
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and re.match(r"\.LBB\w+:$", line):
            out[name][1][line[:-1]] = len(out[name][0])
        elif name and re.match(r"\t[a-z]", line):
            op, _, rest = line.strip().partition(" ")
            out[name][0].append((op, [o.strip() for o in rest.split(",")] if rest else []))
    for name, (code, labels) in out.items():
        following = []
        for i, (op, ops) in enumerate(code):
            if op == "s_endpgm":
                following.append([])
            elif op == "s_branch":
                following.append([labels[ops[0]]])
            else:
                following.append([i + 1] + ([labels[ops[0]]] if op.startswith("s_cbranch") else []))
        out[name] = code, following
    return out


def distances(text, limit=24):
    """(function, product, use, wait states) of each product whose result is used within `limit`
    wait states on some path.  A product that accumulates in place takes the result over."""
    found = []
    for name, (code, following) in functions(text).items():
        for i, (op, ops) in enumerate(code):
            if not op.startswith("v_mfma"):
                continue
            result, seen = registers(ops[0]), set()
            queue = [(0, j) for j in following[i]]
            while queue:
                d, j = heapq.heappop(queue)
                if d > limit or j in seen or j >= len(code):
                    continue
                seen.add(j)
                op2, ops2 = code[j]
                if any(registers(o) & result for o in ops2):
                    a = [registers(o) for o in ops2]
                    if op2.startswith("v_mfma") and a[0] == a[3] == result and not (a[1] | a[2]) & result:
                        continue
                    found.append((name, " ".join([op, *ops]), " ".join([op2, *ops2]), d))
                    break
                step = int(ops2[0]) + 1 if op2 == "s_nop" else 1
                for k in following[j]:
                    heapq.heappush(queue, (d + step, k))
    return found


def test_distances_follow_the_shortest_path():
    text = """kernel:
\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]
\ts_cbranch_scc1 .LBB0_2
\tv_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[4:7], a[4:7]
\ts_nop 7
\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]
\ts_nop 5
.LBB0_2:
\ts_nop 1
\tv_accvgpr_read_b32 v8, a2
\ts_endpgm
.Lfunc_end0:
"""
    assert [d for *_, d in distances(text)] == [3, 8]  # the branch taken; the last product


@pytest.mark.skipif(not shutil.which(build.HIPCC), reason="needs hipcc")
def test_matrix_results_are_read_after_their_wait_states(tmp_path):
    sources = [s for s in sorted(Path(build.CSRC).glob("*.hip")) if "__builtin_amdgcn_mfma" in s.read_text()]
    assert sources
    for s in sources:
        asm = tmp_path / (s.stem + ".s")
        subprocess.run([build.HIPCC, *build.HIP_FLAGS, "-I", str(build.ROOT / "include"), "-I", str(build.CSRC), "-x", "hip",
                        "-S", "--cuda-device-only", str(s), "-o", str(asm)], check=True, capture_output=True)
        text = asm.read_text()
        assert text.count("v_mfma") > 0
        short = [f for f in distances(text) if f[3] < NEED]
        assert not short, short[:5]
