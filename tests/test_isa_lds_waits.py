"""The built code objects: every transposing LDS read (ds_read_b64_tr_b16, the
persistent tile's row-major B fragments) is waited for before anything touches
its result.

LDS operations of a wavefront complete in order and nothing in the hardware
holds back an instruction that reads a result still on its way: on every path
from such a read an `s_waitcnt lgkmcnt(n)` has to come first, with n at most
the LDS operations issued after it.
"""
import glob
import os
import re
import subprocess

import pytest


REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
REG = re.compile(r"(?<!\w)([va])(?:(\d+)|\[(\d+):(\d+)\])(?![\w\[])")


def regs(text):
    out = set()
    for f, one, lo, hi in REG.findall(text):
        out |= {(f, i) for i in range(int(one or lo), int(one or hi) + 1)}
    return out


def kernels(path, tmp):
    """{kernel: [(address, mnemonic, operands)]} of a code object built here."""
    elf = os.path.join(tmp, "co.elf")
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--type=o", "--unbundle",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={path}", f"--output={elf}"], check=True)
    text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", elf], check=True, capture_output=True,
                          text=True).stdout
    out, cur = {}, None
    for line in text.splitlines():
        head = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if head:
            cur = out.setdefault(head[1], [])
        elif cur is not None and "//" in line:
            ins, code = line.split("//", 1)
            op, _, rest = ins.strip().partition(" ")
            cur.append((int(code.split(":")[0], 16), op, rest))
    return out


def early_touches(ins):
    """(read, toucher) pairs: an instruction that a path reaches after a
    transposing read, that names a register of its result, before a wait
    that completes the read."""
    at = {a: i for i, (a, _, _) in enumerate(ins)}
    succ = []
    for i, (a, op, rest) in enumerate(ins):
        s = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        if op.startswith(("s_branch", "s_cbranch")):
            off = int(rest.split()[0])
            s.append(at[a + 4 + 4 * (off - 65536 if off >= 32768 else off)])
        succ.append([x for x in s if x < len(ins)])
    named = [regs(rest) for _, _, rest in ins]
    bad = []
    for i, (_, op, rest) in enumerate(ins):
        if not op.startswith("ds_read_b64_tr"):
            continue
        dst = regs(rest.split(",")[0])
        seen, todo = {}, [(j, 0) for j in succ[i]]  # (next instruction, LDS operations issued since)
        while todo:
            j, c = todo.pop()
            if seen.get(j, 1 << 30) <= c:
                continue
            seen[j] = c
            _, o, r = ins[j]
            if o == "s_waitcnt":
                m = re.search(r"lgkmcnt\((\d+)\)", r)
                if m and int(m[1]) <= c:
                    continue
            if named[j] & dst:
                bad.append((" ".join(ins[i][1:]), " ".join(ins[j][1:])))
                continue
            c += o.startswith("ds_")
            todo += [(k, min(c, 16)) for k in succ[j]]
    return bad


def test_transposing_reads_are_waited_for(tmp_path):
    path = os.path.join(REPO, "triton-ext_amd", "_build", "gemm_bf16.hsaco")
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")) or not os.path.exists(path):
        pytest.skip(f"needs {path} and llvm-objdump")
    found = 0
    for name, ins in kernels(path, str(tmp_path)).items():
        found += any(op.startswith("ds_read_b64_tr") for _, op, _ in ins)
        bad = early_touches(ins)
        assert not bad, (name, len(bad), bad[:4])
    assert found >= 18, found  # persist_kn at three tiles, with 16-bit (4 pairs of types) and fp32 outputs (2)


def test_no_load_is_issued_in_inline_asm():
    """A load in inline asm stands with its wait in the same block, or not at
    all: the compiler takes its result as there at once, may copy or reuse the
    registers while the load is on its way, and does not count it."""
    srcs = [p for p in glob.glob(os.path.join(REPO, "triton-ext_amd", "csrc", "**", "*"), recursive=True)
            if p.endswith((".hip", ".h", ".cpp"))]
    assert len(srcs) > 10
    for p in srcs:
        with open(p) as f:
            text = f.read()
        for m in re.finditer(r"\basm\b[^;]*?\((\s*\"(?:[^\"\\]|\\.)*\")+", text):
            code = m[0]
            if re.search(r"\b(global|buffer|flat|scratch)_load|\bds_read|\bds_load|\bs_load|_rtn", code):
                assert "s_waitcnt" in code, (os.path.relpath(p, REPO), code)
