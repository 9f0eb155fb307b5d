"""The attention kernels read LDS operands in inline assembly that the compiler does not count (att_common.hpp): it may copy,
spill or reuse a register whose read has not arrived.  Whether it did is looked up in the built kernels: along every path,
LDS operations in the order they were issued, trimmed by each wait to what it leaves outstanding (LDS completes in order), and
no instruction that touches the destination of an outstanding read.  The same for results of vector instructions, which
inline assembly may place in front of a matrix instruction without the two wait states between them."""
import os
import re
import subprocess

import pytest

from blockedattention_amd import build

LLVM = "/opt/rocm/llvm/bin/"
REGISTER = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")
LINE = re.compile(r"\t(\S+)(.*?)\s*// 0*([0-9A-F]+):(?: [0-9A-F]{8})+(?: <(.+)\+0x([0-9a-f]+)>)?$")


def registers(text):
    out = set()
    for kind, one, lo, hi in REGISTER.findall(text):
        base = 512 if kind == "a" else 0
        out.update(range(base + int(one or lo), base + int(one or hi) + 1))
    return frozenset(out)


def kernels(source, tmp):
    """name -> [(address, opcode, destination registers, all registers, operand text, branch target)]"""
    obj = os.path.join(build.OBJDIR, source + ".o")
    if not os.path.exists(obj):
        pytest.skip("kernels are not built")
    fat, code = str(tmp / "fat"), str(tmp / "code")
    subprocess.check_call([LLVM + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, obj, str(tmp / "rest")])
    subprocess.check_call([LLVM + "clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--output=" + code,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
    text = subprocess.run([LLVM + "llvm-objdump", "-d", code], check=True, capture_output=True, text=True).stdout
    out, start = {}, 0
    for line in text.split("\n"):
        head = re.match(r"([0-9a-f]+) <(.+)>:", line)
        if head:
            start, body = int(head[1], 16), out.setdefault(head[2], [])
            continue
        m = LINE.match(line)
        if m:
            op, args = m[1], m[2]
            target = start + int(m[5], 16) if m[5] and op.startswith(("s_branch", "s_cbranch")) else None
            written = registers(args if "swap" in op else args.split(",")[0])
            body.append((int(m[3], 16), op, written, registers(args), args, target))
    return out


def step(flight, ins):
    """Outstanding LDS operations after an instruction (their destinations, oldest first), and whether it touched one early."""
    _, op, dst, regs, args, _ = ins
    if op == "s_waitcnt":
        m = re.search(r"lgkmcnt\((\d+)\)", args)
        if m:
            flight = flight[max(0, len(flight) - int(m[1])):]
    elif op.startswith("ds_"):
        read = "read" in op or "permute" in op or "swizzle" in op or "rtn" in op
        early = any((regs - dst if read else regs) & r for r in flight)
        flight = flight + (dst if read else frozenset(),)
        while flight and not flight[0]:
            flight = flight[1:]
        return flight[-16:], early
    else:
        return flight, any(regs & r for r in flight)
    return flight, False


def faults(body):
    at = {ins[0]: i for i, ins in enumerate(body)}
    heads = {at[i[5]] for i in body if i[5] is not None}
    found, seen, work = [], set(), [(0, ())]
    while work:
        i, flight = work.pop()
        while i < len(body):
            if i in heads:
                if (i, flight) in seen:
                    break
                seen.add((i, flight))
            flight, early = step(flight, body[i])
            if early:
                found.append(body[i])
            if body[i][5] is not None:
                work.append((at[body[i][5]], flight))
            if body[i][1] in ("s_branch", "s_endpgm"):
                break
            i += 1
    # a vector instruction's result in a matrix instruction: two wait states
    recent = []
    for ins in body:
        op = ins[1]
        if op.startswith("v_mfma"):
            read = registers(ins[4].split(",", 1)[1])
            if any(read & r for r in recent):
                found.append(ins)
        written = ins[2] if op.startswith("v_") and not op.startswith("v_mfma") else frozenset()
        recent = (recent + [written] * (int(ins[4]) + 1 if op == "s_nop" else 1))[-2:]
    return found


@pytest.mark.parametrize("source", ["attention", "attention_backward"])
def test_no_register_is_touched_before_its_read_arrives(source, tmp_path):
    bodies = kernels(source, tmp_path)
    assert bodies and any(i[1].startswith("ds_read") for b in bodies.values() for i in b)
    wrong = {name: [f"{i[0]:x}: {i[1]}{i[4]}" for i in faults(body)][:4] for name, body in bodies.items()}
    assert not {name: w for name, w in wrong.items() if w}


def test_planted_mistakes_are_found():
    def ins(at, op, args, target=None):
        return (at, op, registers(args.split(",")[0]), registers(args), args, target)
    read, use = ins(0, "ds_read_b128", " v[4:7], v1 offset:64"), ins(8, "v_mov_b32_e32", " v9, v6")
    end, wait = ins(90, "s_endpgm", ""), lambda n: ins(4, "s_waitcnt", f" lgkmcnt({n})")
    other = ins(2, "ds_read_b64", " v[10:11], v1")
    assert faults([read, use, end]) and faults([read, ins(4, "s_waitcnt", " vmcnt(0)"), use, end])
    assert faults([other, read, wait(1), use, end]) and not faults([read, other, wait(1), use, end])
    # only where the branch is taken, and only on the second round of a loop
    assert faults([read, ins(2, "s_cbranch_scc0", " 2", 8), wait(0), use, end])
    assert faults([ins(1, "s_nop", " 0"), use, ins(10, "ds_read_b32", " v6, v1"), ins(12, "s_cbranch_scc0", " 2", 1), end])
    mul, nop = ins(1, "v_mul_f32_e32", " v8, v8, v1"), lambda n: ins(2, "s_nop", f" {n}")
    product = ins(5, "v_mfma_f32_16x16x32_f16", " v[20:23], v[12:15], v[16:19], v[8:11]")
    assert faults([mul, nop(0), product, end]) and not faults([mul, nop(1), product, end])
