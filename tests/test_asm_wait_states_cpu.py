"""Wait states around vector instructions of inline asm, in the assembly that hipcc makes of the kernels.  hipcc keeps the states that matrix products need
between a writer and a reader only where it sees both; next to asm the source has to.  Counted as the hardware's manual does, an instruction one state and
s_nop n n + 1, along every path, without the time that a product itself takes."""
import collections
import os
import re
import shlex
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "aphrodite_engine_amd", "csrc")
PRODUCTS = ("v_mfma", "v_smfma")
BEHIND_ASM = 2                          # states between asm's result and a product, a lane swap or a lane choice that reads it

Step = collections.namedtuple("Step", "line asm op text writes reads states")


def _behind(product):
    """States between a product and a vector instruction on its result: its passes and four.  16-bit products of 16x16x32 and 32x32x16 take 8 passes at most."""
    return 12 if re.search(r"_(16x16x32|32x32x16)_b?f16", product) else 20


def _registers(operand):
    m = re.match(r"-?\|?([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", operand.strip())
    if not m:
        return frozenset()
    return frozenset((m[1], i) for i in (range(int(m[2]), int(m[3]) + 1) if m[2] else [int(m[4])]))


def _steps(text):
    """{kernel: [label or Step]}"""
    kernels, into, asm = {}, None, False
    for line, s in enumerate(text.splitlines(), 1):
        if "#ASMSTART" in s or "#ASMEND" in s:
            asm = "#ASMSTART" in s
        elif m := re.match(r"(_Z[\w.$]+):", s):
            into = kernels.setdefault(m[1], [])
        elif into is not None and (m := re.match(r"(\.L\w+):", s)):
            into.append(m[1])
        elif into is not None and (s := s.split(";")[0].strip()) and not s.startswith("."):
            op, _, rest = s.partition(" ") if " " in s else s.partition("\t")
            ops = [_registers(o) for o in re.split(r",(?![^\[]*\])", rest)]
            vector = op.startswith("v_")
            writes = ops[0] if vector and not op.startswith(("v_cmp", "v_readlane", "v_readfirstlane")) or op.startswith(("ds_read", "buffer_load", "global_load")) else frozenset()
            reads = frozenset().union(*(ops if not writes or op.startswith(("v_fmac", "v_swap")) or "swap" in op else ops[1:])) if vector else frozenset()
            if "swap" in op:
                writes |= ops[1]
            into.append(Step(line, asm, op, s, writes, reads, int(rest, 0) + 1 if op == "s_nop" else 1))
    return kernels


def _too_near(text):
    found = []
    for kernel, steps in _steps(text).items():
        at = {s: i for i, s in enumerate(steps) if isinstance(s, str)}
        ahead = collections.defaultdict(list)
        for i, s in enumerate(steps):
            if not isinstance(s, str) and s.op.startswith(("s_branch", "s_cbranch")):
                ahead[at[s.text.split()[-1]]].append(i)
            if i + 1 < len(steps) and (isinstance(s, str) or s.op not in ("s_branch", "s_endpgm", "s_setpc_b64")):
                ahead[i + 1].append(i)

        def writer(i, registers, which, states):
            """A step that ``which`` picks and that wrote one of the registers fewer than ``states`` ahead of step i, on some path."""
            seen, todo = {}, [(i, 0, registers)]
            while todo:
                j, d, left = todo.pop()
                for k in ahead[j]:
                    s, e, rest = steps[k], d, left
                    if not isinstance(s, str):
                        if s.writes & left and which(s) and d < states(s):
                            return s
                        e, rest = d + s.states, left - s.writes
                    if rest and e < 20 and seen.get((k, rest), 20) > e:
                        seen[k, rest] = e
                        todo.append((k, e, rest))

        for i, s in enumerate(steps):
            if isinstance(s, str) or not s.op.startswith("v_"):
                continue
            w = None
            if s.asm:
                w = writer(i, s.reads | s.writes, lambda x: x.op.startswith(PRODUCTS), lambda x: _behind(x.op))
            if not w and (s.op.startswith(PRODUCTS) or "permlane" in s.op):
                w = writer(i, s.reads, lambda x: x.asm and x.op.startswith("v_") and not x.op.startswith(PRODUCTS), lambda x: BEHIND_ASM)
            if not w and "row_" in s.text:
                w = writer(i, _registers(s.text.split(",")[1]), lambda x: x.asm and x.op.startswith("v_"), lambda x: BEHIND_ASM)
            if w:
                found.append(f"{kernel}: '{w.text}' (line {w.line}) too near '{s.text}' (line {s.line})")
    return found


def test_the_count():
    def kernel(between, ahead="v_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], 0", asm="v_max3_f32 v30, v3, v4, v5"):
        return f"_Zk:\n\t{ahead}\n{between}\t;;#ASMSTART\n\t{asm}\n\t;;#ASMEND\n\ts_endpgm\n"
    far = "\ts_nop 11\n"
    assert _too_near(kernel("")) and not _too_near(kernel(far)) and _too_near(kernel("\ts_nop 10\n"))
    assert _too_near(kernel(far, ahead="v_mfma_f32_32x32x2_f32 v[0:15], v20, v24, 0"))
    # a jump past the states, and a register written anew
    assert _too_near(kernel("\ts_cbranch_scc1 .L1\n" + far + ".L1:\n"))
    assert not _too_near(kernel("\tv_mov_b32_e32 v3, 0\n", asm="v_max3_f32 v30, v3, v31, v32"))
    back = kernel("", ahead="s_nop 0", asm="v_pk_mul_f16 v21, v21, s6").replace("\ts_endpgm", "{}\tv_mfma_f32_16x16x32_f16 v[0:3], v[20:23], v[24:27], 0\n\ts_endpgm")
    assert _too_near(back.format("\tv_and_b32_e32 v9, 15, v9\n")) and not _too_near(back.format("\ts_nop 1\n"))


@pytest.mark.skipif(not shutil.which("hipcc") and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")
@pytest.mark.parametrize("name", ["flash_attn_short", "wna16_gemm", "mixers/delta_rule_chunked"])
def test_states_around_inline_asm(name, tmp_path):
    folder, file = os.path.split(os.path.join(CSRC, name))
    lines = subprocess.run(["make", "-n", "-B", f"build/{file}.o"], cwd=folder, check=True, capture_output=True, text=True).stdout.splitlines()
    command = [a for a in shlex.split(next(x for x in lines if f"{file}.hip" in x)) if a != "-c"]
    out = tmp_path / "kernels.s"
    command[command.index("-o") + 1] = str(out)
    subprocess.run(command + ["-S", "--offload-device-only", "-w"], cwd=folder, check=True, capture_output=True)
    found = _too_near(out.read_text())
    assert not found, "\n".join(found[:10])
