"""The grouped matmul's 16 x 16 x 32 matrix instructions are inline assembly, so the compiler does not know what they are
and inserts no wait states around them.  These checks read the gfx950 code of the built library: an ordinary vector
instruction that writes a register one of them reads is at least two instructions away, one that touches a result at
least 18 (the longest matrix instruction's), and the clearing of the accumulators is separated from the first product by
a wait that the source asks for, not only by what the compiler happened to put there."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from mindspeed_amd import _lib

MFMA = "v_mfma_f32_16x16x32"
WRITE_STATES, RESULT_STATES = 2, 18
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def _code_objects(path):
    """The gfx950 code objects of a library: every offload bundle in it lists (offset, size, target) per member."""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        (members,) = struct.unpack_from("<Q", data, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(members):
            offset, size, name = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + name]
            p += 24 + name
            if target.endswith(b"gfx950") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(magic, at + len(magic))


def _registers(text):
    """Vector registers named in an operand list, as (file, number)."""
    out = set()
    for file, lo, hi, single in re.findall(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        for r in range(int(lo or single), int(hi or single) + 1):
            out.add((file, r))
    return out


class _Instruction:
    def __init__(self, text):
        self.op, _, rest = text.partition(" ")
        operands = re.split(r",\s*(?![^\[]*\])", rest)
        self.matrix = self.op.startswith("v_mfma")
        self.vector = self.op.startswith("v_") and not self.matrix
        self.states = int(operands[0], 0) + 1 if self.op == "s_nop" else 1
        self.target = operands[0].strip() if self.op.startswith(("s_branch", "s_cbranch")) else None
        self.ends = self.op in ("s_branch", "s_endpgm", "s_setpc_b64")
        memory = self.op.startswith(("ds_", "global_", "buffer_", "flat_", "scratch_"))
        self.named = _registers(rest) if self.vector or self.matrix or memory else set()
        swap = self.op.startswith("v_swap") or self.op.startswith("v_permlane")
        self.written = (self.named if swap else _registers(operands[0])) if self.vector or self.matrix else set()
        self.read = _registers(",".join(operands[1:])) if self.matrix else set()


def _kernels(assembly):
    """name -> (instructions, predecessors of each instruction)."""
    found, name = {}, None
    for line in assembly.splitlines():
        head = re.match(r"^(?:[0-9a-f]+ )?<([^>]+)>:", line)
        if head and not re.match(r"^L\d+$", head.group(1)):
            name, code, labels = head.group(1), [], {}
            found[name] = (code, labels)
        elif head:
            labels[head.group(1)] = len(code)
        elif name and line.startswith(("\t", " ")) and line.split("//")[0].strip():
            code.append(_Instruction(re.sub(r"\s+", " ", line.split("//")[0].strip())))
    for name, (code, labels) in found.items():
        before = [[i - 1] if i and not code[i - 1].ends else [] for i in range(len(code))]
        for i, ins in enumerate(code):
            if ins.target is not None:
                before[labels[ins.target.strip("<>")]].append(i)
        found[name] = (code, before)
    return found


def _behind(code, before, at, states):
    """Instructions that can run fewer than `states` wait states ahead of instruction `at`, on any path."""
    todo, best = [(p, 0) for p in before[at]], {}
    while todo:
        i, passed = todo.pop()
        if passed >= states or best.get(i, states) <= passed:
            continue
        best[i] = passed
        todo += [(p, passed + code[i].states) for p in before[i]]
    return best


def _violations(code, before):
    bad = []
    for i, ins in enumerate(code):
        if ins.op.startswith(MFMA):
            for j in _behind(code, before, i, WRITE_STATES):
                if code[j].vector and code[j].written & ins.read:
                    bad.append(("operand written too late", j, i))
        elif ins.named:
            for j in _behind(code, before, i, RESULT_STATES):
                if code[j].op.startswith(MFMA) and code[j].written & ins.named:
                    bad.append(("result touched too early", j, i))
    return bad


def _unguarded_entries(code, before):
    """Products that an ordinary write of their accumulator can reach, on any path, without an s_nop of two states or more
    (or an earlier product on the same accumulator) in between."""
    bad = []
    for i, ins in enumerate(code):
        if not ins.op.startswith(MFMA):
            continue
        todo, met = list(before[i]), set()
        while todo:
            j = todo.pop()
            if j in met:
                continue
            met.add(j)
            other = code[j]
            if (other.op == "s_nop" and other.states >= WRITE_STATES) or (other.matrix and other.written & ins.written):
                continue
            if other.vector and other.written & ins.written:
                bad.append((j, i))
                break
            todo += before[j]
    return bad


def test_the_check_sees_planted_hazards():
    def check(*lines):
        text = "\n".join(["0000 <k>:"] + [l if l.startswith("<") else "\t" + l for l in lines])
        code, before = _kernels(text)["k"]
        return [v[0] for v in _violations(code, before)], len(_unguarded_entries(code, before))

    product = MFMA + "_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"
    late, early = ["operand written too late"], ["result touched too early"]
    assert check("v_mov_b32_e32 v2, v9", "s_nop 0", product) == (late, 0)
    assert check("v_mov_b32_e32 v2, v9", "s_nop 1", product) == ([], 0)
    assert check("v_accvgpr_write_b32 a3, 0", "s_mov_b32 s0, 1", "s_mov_b32 s1, 1", product) == ([], 1)
    assert check("v_accvgpr_write_b32 a3, 0", "s_nop 1", product, product) == ([], 0)
    assert check("v_mov_b32_e32 v20, v9", product, "s_nop 15", "v_accvgpr_read_b32 v1, a2") == (early, 0)
    assert check(product, "s_nop 15", "s_nop 15", "v_accvgpr_read_b32 v1, a2") == ([], 0)
    assert check(product, "s_nop 15", "ds_write_b128 v40, a[0:3]") == (early, 0)
    # over a loop's back edge
    assert check("<L0>:", product, "s_add_u32 s0, s0, 1", "v_mov_b32_e32 v6, v9", "s_cbranch_scc1 <L0>", "s_endpgm") == (late, 0)


def test_built_matrix_kernels_keep_their_distances(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    seen = 0
    for n, code_object in enumerate(_code_objects(_lib.LIB_PATH)):
        path = tmp_path / f"{n}.co"
        path.write_bytes(code_object)
        assembly = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--symbolize-operands", str(path)], check=True,
                                  capture_output=True, text=True).stdout
        if MFMA not in assembly:
            continue
        for name, (code, before) in _kernels(assembly).items():
            products = sum(i.op.startswith(MFMA) for i in code)
            if products:
                seen += products
                assert not _violations(code, before), (name, _violations(code, before)[:3])
                assert not _unguarded_entries(code, before), (name, _unguarded_entries(code, before)[:3])
    assert seen >= 1000
