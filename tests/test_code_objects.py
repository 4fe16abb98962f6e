"""What the compiler made of the attention kernels, read from the built library: matrix results are never touched early, and kernels
that were measured without scratch memory have none.  No GPU needed."""
import os
import re
import shutil
import struct
import subprocess
from collections import defaultdict

import pytest

from baselinebenchmark_amd import _cabi

LLVM = "/opt/rocm/llvm/bin"
pytestmark = [pytest.mark.sage_attention,
              pytest.mark.skipif(not shutil.which("llvm-objdump", path=LLVM), reason="needs ROCm's llvm-objdump")]

MFMA_PASSES = {"32x32x32_i8": 8, "16x16x64_i8": 4, "32x32x16_f16": 8, "16x16x32_f16": 4, "32x32x64_f8f6f4": 16, "16x16x128_f8f6f4": 8}


@pytest.fixture(scope="module")
def code_objects(sage_lib, tmp_path_factory):
    """The gfx950 code objects of the library, one per source file, as files."""
    data, out, at = _cabi.LIB_PATH.read_bytes(), [], 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entries, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(entries):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            if data[p + 24:p + 24 + n].endswith(b"gfx950"):
                path = tmp_path_factory.mktemp("co") / f"{len(out)}.co"
                path.write_bytes(data[at + offset:at + offset + size])
                out.append(path)
            p += 24 + n
        at += 24
    assert out
    return out


def registers(operand):
    """Vector registers that an operand names."""
    m = re.match(r"-?\|?([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", operand)
    if not m:
        return frozenset()
    lo, hi = (m[2], m[3]) if m[2] else (m[4], m[4])
    return frozenset((m[1], r) for r in range(int(lo), int(hi) + 1))


class Kernel:
    def __init__(self, name, lines):
        self.name, self.addresses, self.text = name, [], []
        for line in lines:   # "\tv_add_f32 v0, v1, v2   // 000000001A00: ..."
            text, _, note = line.partition("//")
            self.text.append(text.strip())
            self.addresses.append(int(note.split(":")[0], 16))
        self.index = {a: i for i, a in enumerate(self.addresses)}
        self.targets = {}
        for i, (text, line) in enumerate(zip(self.text, lines)):
            if text.startswith(("s_branch", "s_cbranch")):
                self.targets[i] = int(re.search(r"\+0x([0-9a-f]+)>", line)[1], 16) if "+0x" in line else 0
        self.memo = {}

    def uses(self, i):
        """(registers touched, other than as an accumulator that a matrix instruction goes on with; wait states that pass)."""
        if i not in self.memo:
            op, _, rest = self.text[i].partition(" ")
            operands = [o.strip() for o in re.split(r",\s*(?![^\[]*\])", rest)]
            if op == "s_nop":
                self.memo[i] = frozenset(), int(operands[0], 0) + 1
            elif op.startswith("v_mfma"):
                self.memo[i] = frozenset().union(*(registers(o) for k, o in enumerate(operands) if k not in (0, 3))), 1
            else:
                self.memo[i] = frozenset().union(*map(registers, operands)), 1
        return self.memo[i]

    def early(self):
        """Instructions that touch a matrix result before it is there, on any path: a result of an N-pass instruction needs N + 4 wait
        states, and nothing but the instructions in between makes them pass."""
        found = []
        base = self.addresses[0]
        for i, text in enumerate(self.text):
            if not text.startswith("v_mfma"):
                continue
            need = next(p for shape, p in MFMA_PASSES.items() if shape in text) + 4
            result = registers(text.partition(" ")[2])
            todo, seen = [(i + 1, 0)], {}
            while todo:
                j, states = todo.pop()
                if states >= need or j >= len(self.text) or seen.get(j, need) <= states:
                    continue
                seen[j] = states
                op = self.text[j].partition(" ")[0]
                if op.startswith("v_mfma") and registers(self.text[j].partition(" ")[2]) == result:
                    continue   # (a later result in the same place: it is followed on its own)
                touched, passed = self.uses(j)
                if touched & result:
                    found.append(f"{self.name}: `{self.text[j]}` {states} states after `{text}`, needs {need}")
                    continue
                if j in self.targets:
                    todo.append((self.index[base + self.targets[j]], states + passed))
                if op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                    todo.append((j + 1, states + passed))
        return found


def kernels(path, wanted):
    text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
    name, lines = None, []
    for line in text.splitlines():
        m = re.match(r"^[0-9a-f]+ <(\S+)>:$", line)
        if m:
            if name and lines and wanted in name:
                yield Kernel(name, lines)
            name, lines = m[1], []
        elif line.startswith("\t") and "//" in line:
            lines.append(line)
    if name and lines and wanted in name:
        yield Kernel(name, lines)


def test_no_matrix_result_is_touched_before_it_is_there(code_objects):
    # (the compiler counts its own scheduling markers as wait states)
    found, seen = [], defaultdict(int)
    for path in code_objects:
        for k in kernels(path, "attn"):
            seen["kernels"] += 1
            seen["products"] += sum(t.startswith("v_mfma") for t in k.text)
            found += k.early()
    assert seen["kernels"] > 100 and seen["products"] > 10000, dict(seen)
    assert not found, "\n".join(found[:20])


def scratch_bytes(path):
    """Bytes of scratch memory a lane, by kernel."""
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(path)], capture_output=True, text=True, check=True).stdout
    return dict(re.findall(r"\.name: +(\S+)\n(?:(?! +- \.agpr_count)[^\n]*\n)*? +\.private_segment_fixed_size: (\d+)", notes))


def attention_kernel(D, NW, pv, causal, msum, mask, ksub):
    """Start of the mangled name of the variants of sage::attn_kernel with these template arguments."""
    return f"_ZN4sage11attn_kernelILi{D}ELi{NW}ELi128ELi{pv}ELb{int(causal)}ELb{int(msum)}ELi{mask}ELi{ksub}E"


def test_kernels_that_lose_by_scratch_memory_have_none(code_objects):
    # 128 rows, FP8 P.V, head_dim 64, interleaved K scales: with LSE up to 1.46 times as long as with 256 rows when they spilled
    wanted = [attention_kernel(64, 4, 1, causal, msum, 0, 3) for causal, msum in ((False, False), (True, False), (True, True))]
    masked = attention_kernel(64, 4, 1, False, False, 3, 1)   # ... and with a packed mask, whose LDS leaves room for two workgroups only
    seen = {name: int(n) for path in code_objects for name, n in scratch_bytes(path).items() if name.startswith((*wanted, masked))}
    assert len(seen) == 2 * len(wanted) + 1   # (with INT8 and with floating-point Q)
    assert not any(seen.values()), seen


def test_no_kernel_that_no_call_reaches(code_objects):
    # 256 rows where the calls of a kind take 128 at every size: interleaved scales (FP8 P.V with LSE; FP16, head_dim 64, causal), masks with one K scale
    # per 32 keys (all but boolean ones over FP16 P.V)
    unreachable = [attention_kernel(D, 8, 1, causal, False, 0, 3) for D in (64, 128) for causal in (False, True)] + [attention_kernel(64, 8, 0, True, False, 0, 3)]
    unreachable += [attention_kernel(D, 8, pv, False, False, mask, 1) for D in (64, 128) for pv in (0, 1) for mask in (3, 4, 5) if mask == 5 or pv == 1]
    names = [name for path in code_objects for name in scratch_bytes(path)]
    assert any(name.startswith(attention_kernel(128, 8, 0, False, False, 3, 1)) for name in names)
    assert not [name for name in names if name.startswith(tuple(unreachable))]


def test_the_walk_sees_an_early_use_on_every_path():
    def at(*texts):
        return [f"\t{t}  // {0x100 + 8 * i:012X}:" + (f" <k+0x{8 * int(t.split()[1]):x}>" if "branch" in t else "") for i, t in enumerate(texts)]
    product = "v_mfma_i32_16x16x64_i8 v[0:3], v[8:11], v[12:15], 0"
    copy = "v_mov_b32_e32 v20, v3"
    assert Kernel("k", at(product, "s_nop 6", copy, "s_endpgm")).early()
    assert not Kernel("k", at(product, "s_nop 7", copy, "s_endpgm")).early()
    assert not Kernel("k", at(product, "s_nop 0", "v_mfma_i32_16x16x64_i8 v[0:3], v[8:11], v[12:15], v[0:3]", "s_nop 7", copy, "s_endpgm")).early()
    assert Kernel("k", at(product, "s_cbranch_scc1 4", "s_nop 7", "s_endpgm", copy, "s_endpgm")).early()
    assert Kernel("k", at(copy, product, "s_nop 3", "s_branch 0")).early()
    assert not Kernel("k", at(copy, product, "s_nop 6", "s_branch 0")).early()
