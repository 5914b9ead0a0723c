"""Wait states in the built gfx950 code that the compiler cannot see to: it does not look
inside inline assembly, so an instruction there may come too early after a matrix
instruction. Reads the disassembly of the library; no GPU needed."""
import collections
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "pil2-proofman_amd", "libpil2_commit_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

# passes of four cycles; instructions before a VALU write to the SrcC registers, and
# before a VALU access to the result
PASSES = {"v_mfma_i32_16x16x64_i8": 4, "v_mfma_i32_32x32x32_i8": 8}
SRCC_WAIT = {4: 3, 8: 7}
RESULT_WAIT = {4: 8, 8: 12}
# instructions whose second operand is a result too (a carry mask)
TWO_RESULTS = re.compile(r"v_(mad_[ui]64_[ui]32|(add|sub|subrev|addc|subb|subbrev)_co_u32)")

Instruction = collections.namedtuple("Instruction", "op operands writes reads address target")


def _registers(operand):
    if operand == "vcc":
        return {("s", 106), ("s", 107)}
    m = re.fullmatch(r"-?\|?([vs])(?:(\d+)|\[(\d+):(\d+)\])\|?", operand)
    if not m:
        return set()
    first, last = (m[2], m[2]) if m[2] else (m[3], m[4])
    return {(m[1], i) for i in range(int(first), int(last) + 1)}


def _instruction(op, operands, address, target):
    sets = [_registers(o) for o in operands]
    n = 2 if TWO_RESULTS.match(op) else 1
    writes, reads = set().union(*sets[:n]), set().union(*sets[n:])
    if op.startswith(("v_permlane32_swap", "v_swap")):
        writes = reads = writes | reads
    elif op.startswith(("v_fmac", "v_writelane")):
        reads = reads | writes
    if not op.startswith("v_"):  # of the others only the results of scalar instructions count
        reads = set()
        if not op.startswith("s_") or op.startswith(("s_cmp", "s_bitcmp", "s_cbranch", "s_waitcnt", "s_nop")):
            writes = set()
    return Instruction(op, operands, writes, reads, address, target)


def functions(disassembly):
    """Name -> instructions of every function in llvm-objdump's text."""
    out, code = collections.OrderedDict(), None
    for line in disassembly.split("\n"):
        m = re.match(r"[0-9a-f]+ <(.+)>:", line)
        if m:
            code = out.setdefault(m[1], [])
            continue
        m = re.match(r"\t(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):(.*)", line)
        if not m:
            continue
        operands = [o.strip().split(" ")[0] for o in re.split(r",\s*(?![^\[]*\])", m[2])] if m[2] else []
        target = None
        if m[1].startswith(("s_cbranch", "s_branch")):
            t = re.search(r"\+0x([0-9a-f]+)>", m[4])
            target = int(t[1], 16) if t else 0
        code.append(_instruction(m[1], operands, int(m[3], 16), target))
    return out


def early(code, at, start, rules):
    """The VALU instructions that come too early after code[start] (at: places by address).
    rules: (name, registers, instructions in between, whether writes count, reads)."""
    most = max(r[2] for r in rules)
    found, seen, paths = [], set(), [(start + 1, 0, tuple(r[1] for r in rules))]
    while paths:
        k, waited, sets = paths.pop()
        while k < len(code) and waited < most and (k, waited) not in seen:
            seen.add((k, waited))
            i = code[k]
            if i.op.startswith("v_mfma"):  # hands the registers over: the compiler's business
                sets = tuple(s - i.writes for s in sets)
            elif i.op.startswith("v_"):
                for (name, _, wait, w, r), s in zip(rules, sets):
                    if waited < wait and s & ((i.writes if w else set()) | (i.reads if r else set())):
                        found.append("%s after %d: %s %s" % (name, waited, i.op, ", ".join(i.operands)))
                sets = tuple(s - i.writes for s in sets)
            else:
                sets = tuple(s - i.writes for s in sets)
            waited += int(i.operands[0], 0) + 1 if i.op == "s_nop" else 1
            if i.op in ("s_endpgm", "s_setpc_b64", "s_swappc_b64"):
                break
            if i.target is not None:
                paths.append((at[code[0].address + i.target], waited, sets))
                if i.op == "s_branch":
                    break
            k += 1
    return found


def matrix_hazards(code):
    out, at = [], {i.address: k for k, i in enumerate(code)}
    for k, i in enumerate(code):
        if not i.op.startswith("v_mfma"):
            continue
        p = PASSES[i.op]  # a matrix instruction not listed needs its passes here
        result, srcc = _registers(i.operands[0]), _registers(i.operands[3])
        out += early(code, at, k, [("result", result, RESULT_WAIT[p], True, True),
                               ("SrcC", srcc - result, SRCC_WAIT[p], True, False)])
    return out


def disassemble(path, directory):
    """Text of every gfx950 code object in the file."""
    here = os.path.join(str(directory), "code")
    with open(path, "rb") as f, open(here, "wb") as g:
        g.write(f.read())
    subprocess.run([OBJDUMP, "--offloading", here], check=True, capture_output=True, cwd=str(directory))
    parts = sorted(p for p in os.listdir(str(directory)) if p.endswith("gfx950"))
    assert parts, "no gfx950 code in " + path
    return [subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(str(directory), p)], check=True,
                           capture_output=True, text=True).stdout for p in parts]


@pytest.fixture(scope="module")
def code(tmp_path_factory):
    out = collections.OrderedDict()
    for text in disassemble(LIB, tmp_path_factory.mktemp("isa")):
        out.update(functions(text))
    return out


def test_rules_see_an_early_write():
    """The rules themselves, on one sequence with each fault and one without."""
    def run(*lines):
        text = "0000000000001000 <k>:\n" + "".join(
            "\t%s // %012X: 00\n" % (l, 0x1000 + 8 * k) for k, l in enumerate(lines))
        return matrix_hazards(functions(text)["k"])

    mfma = "v_mfma_i32_16x16x64_i8 v[4:7], v[10:13], v[14:17], v[0:3]"
    late = "v_mad_i64_i32 v[2:3], s[0:1], v20, 1, v[22:23]"
    assert run(mfma, late) and run(mfma, "s_nop 1", late) and not run(mfma, "s_nop 2", late)
    dead = "v_mov_b32_e32 v6, v30"
    assert run(mfma, "s_nop 6", dead) and not run(mfma, "s_nop 7", dead)
    # round a loop
    loop = "s_cbranch_scc1 65533 // 000000001008: BF85FFFD <k+0x0>"
    text = "0000000000001000 <k>:\n\t%s // 000000001000: 00\n\t%s // 000000001008: 00\n\t%s\n" % (
        dead, mfma, loop.replace("1008", "1010"))
    assert matrix_hazards(functions(text)["k"])


def test_matrix_registers_are_not_overwritten_early(code):
    matrix = [f for f, c in code.items() if any(i.op.startswith("v_mfma") for i in c)]
    assert len(matrix) > 40
    bad = ["%s: %s" % (f, h) for f in matrix for h in matrix_hazards(code[f])]
    assert not bad, "%d early accesses:\n%s" % (len(bad), "\n".join(bad[:20]))


# VALU instructions between a VALU write of scalar registers (a carry mask) and a VALU
# read of them
MASK_WAIT = 2


def mask_hazards(code):
    out, at = [], {i.address: k for k, i in enumerate(code)}
    for k, i in enumerate(code):
        masks = {r for r in i.writes if r[0] == "s"} if i.op.startswith("v_") else set()
        if masks:
            out += early(code, at, k, [("mask", masks, MASK_WAIT, False, True)])
    return out


def test_carry_masks_are_not_read_early(code):
    bad = ["%s: %s" % (f, h) for f, c in code.items() for h in mask_hazards(c)]
    assert not bad, "%d early reads:\n%s" % (len(bad), "\n".join(bad[:20]))


# Factors whose halves the compiler knows in part, so that it leaves out a multiply-add of
# the chain that the masks' distances are counted in
KNOWN = ["(uint64_t)(uint32_t)a[i]", "a[i] << 32", "7", "0x7000000000000000ull"]
PRODUCTS = ["gl_mulk1(x, {f}, 0, 0)", "gl_mulk1({f}, x, 0, 0)", "gl_mulk1({f}, {f}, 0, 0)", "gl_mulk1(x, {f}, k, k)",
            "gl_mul(x, {f})", "gl_mul({f}, {f})", "gl_mul_nc(x, {f})"]


def test_products_by_known_factors_keep_the_distance(tmp_path):
    import build
    calls = [p.format(f=f) for p in PRODUCTS for f in KNOWN]
    calls += ["gl_mulk1<true>(x, %s, 0, 0)" % f for f in ("(uint64_t)k", "(uint64_t)k << 32", "7")]
    src, obj = tmp_path / "k.hip", tmp_path / "k.co"
    src.write_text('#include "gl_field.h"\n' + "".join(
        'extern "C" __global__ void k%d(uint64_t *a, uint32_t k)\n{\n    const int i = threadIdx.x;\n'
        "    const uint64_t x = a[i + 64];\n    a[i] = %s;\n}\n" % (n, c) for n, c in enumerate(calls)))
    subprocess.run(["hipcc"] + build.FLAGS + ["-w", "--offload-device-only", "--no-gpu-bundle-output", "-c", "-I",
                                              build.CSRC, str(src), "-o", str(obj)], check=True, capture_output=True)
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True,
                          text=True).stdout
    kernels = functions(text)
    assert set(kernels) == {"k%d" % n for n in range(len(calls))}
    bad = {c: mask_hazards(kernels["k%d" % n]) for n, c in enumerate(calls)}
    assert not any(bad.values()), {c: h for c, h in bad.items() if h}
