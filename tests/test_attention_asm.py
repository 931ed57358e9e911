"""The attention core's in-place rescale against the matrix cores' wait states (CPU only).

`attention_block` (neo-theano_amd/csrc/tq_attention.hip) multiplies its accumulators in
inline asm, where the compiler places none of the wait states that a vector instruction
needs after the MFMA that writes its register (19 at most) and an MFMA after the vector
instruction (2).  This compiles the kernels to gfx950 assembly with the library's flags
and walks, in every instance, all paths back and on from each of these multiplies until
the states are held, and fails on an MFMA that touches its register before that."""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "neo-theano_amd"))

NEED_AFTER_MFMA, NEED_BEFORE_MFMA = 19, 2


def _regs(text):
    out = set()
    for lo, hi, one in re.findall(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b", text):
        out |= {int(one)} if one else set(range(int(lo), int(hi) + 1))
    return out


def _parse(body):
    """[(text, in asm)], and the instructions that can run after and before each."""
    code, asm, labels = [], False, {}
    for raw in body.split("\n"):
        if "#ASMSTART" in raw or "#ASMEND" in raw:
            asm = "#ASMSTART" in raw
            continue
        line = raw.split(";")[0].strip()
        label = re.fullmatch(r"(\.LBB\w+):", line)
        if label:
            labels[label.group(1)] = len(code)
        elif line and not line.startswith(".") and not line.endswith(":"):
            code.append((line, asm))
    after = [[] for _ in code]
    for i, (line, _) in enumerate(code):
        op = line.split()[0]
        if op.startswith(("s_cbranch", "s_branch")):
            after[i].append(labels[line.split()[-1]])
        if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(code):
            after[i].append(i + 1)
    before = [[] for _ in code]
    for i, targets in enumerate(after):
        for t in targets:
            if t < len(code):
                before[t].append(i)
    return code, after, before


def _states(line):
    m = re.fullmatch(r"s_nop (\d+)", line)
    return int(m.group(1)) + 1 if m else 1


def hazards(body):
    """Multiplies in inline asm with an MFMA on their register on some path before its wait
    states are held; and the count of these multiplies."""
    code, after, before = _parse(body)
    found, count = [], 0
    for i, (line, in_asm) in enumerate(code):
        if not in_asm or not line.startswith("v_mul_f32"):
            continue
        count += 1
        reg = _regs(line.split(",")[0])
        for edges, need in ((before, NEED_AFTER_MFMA), (after, NEED_BEFORE_MFMA)):
            todo, seen = [(j, 0) for j in edges[i]], {}
            while todo:
                j, held = todo.pop()
                if held >= need or seen.get(j, need) <= held:
                    continue
                seen[j] = held
                if code[j][0].startswith("v_mfma") and reg & _regs(code[j][0]):
                    found.append(line)
                    break
                todo += [(t, held + _states(code[j][0])) for t in edges[j] if t < len(code)]
    return found, count


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    import build
    if not os.path.exists(build.HIPCC) and not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("asm") / "tq_attention.s"
    flags = [f for f in build.HIP_FLAGS if f not in ("-fPIC", "-Wall")]
    r = subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(build.CSRC, "tq_attention.hip"),
                        "-o", str(out)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    return {m.group(1): m.group(2) for m in
            re.finditer(r"^(_Z\w*k_attention\w*):.*?\n(.*?)\.Lfunc_end", out.read_text(), re.S | re.M)}


def test_every_rescale_is_far_from_the_products(kernels):
    assert len(kernels) == 9, sorted(kernels)
    for name, body in sorted(kernels.items()):
        found, count = hazards(body)
        assert count in (16, 32, 48, 64), (name, count)  # 16 for every 32 of the head dimension
        assert found == [], name


MFMA = "\tv_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], v[0:15]\n"
MUL = "\t;;#ASMSTART\n\tv_mul_f32 v3, v50, v3\n\t;;#ASMEND\n"
FILL = "\tv_add_f32 v40, v41, v42\n"


def test_model_flags_a_near_product():
    assert hazards(MFMA + FILL * 18 + MUL) == (["v_mul_f32 v3, v50, v3"], 1)
    assert hazards(MFMA + FILL * 19 + MUL) == ([], 1)
    assert hazards(MFMA + "\ts_nop 15\n" + FILL * 3 + MUL) == ([], 1)
    assert hazards(MFMA.replace("v[0:15]", "v[60:75]") + MUL) == ([], 1)
    assert hazards(MUL + FILL + MFMA) == (["v_mul_f32 v3, v50, v3"], 1)
    assert hazards(MUL + FILL * 2 + MFMA) == ([], 1)
    # round a loop: the product at its end is near the multiply at its head
    for fill, near in ((9, True), (18, False)):
        loop = ".LBB0_1:\n" + MUL + FILL * 30 + MFMA + FILL * fill + "\ts_cbranch_scc1 .LBB0_1\n\ts_endpgm\n"
        assert bool(hazards(loop)[0]) == near
