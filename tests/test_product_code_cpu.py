"""The compiled code of the matrix products whose loops count on instructions that hipcc does not know or may leave out (csrc/ob_mm.h): every
``ob_dense_wr / mm``, ``ob_t16_wr / mm`` and ``ob_t32_wr / mm`` kernel of the built objects, disassembled.

- ``ob_wr_loop``'s waits in front of its barriers count the loads of later steps.  hipcc drops a load whose result is never used, and a count that includes it lets the
  barrier pass before a tile has landed.  Along every path through the kernel the waits in front of barriers alone, without the others that hipcc happens to
  place, must leave at most the transfers of NST - 2 steps on their way.
- The MFMAs are inline assembly, so hipcc does not keep the two wait states that an operand written by the vector unit needs before an MFMA reads it, and a register
  kept in scratch would be fetched in front of one."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from onebit_amd import build as B

LIBS = {"onebit_hybrid.hip": (B.LIB_HYBRID, B.SOURCES_HYBRID), "onebit_train.hip": (B.LIB, B.SOURCES)}
KERNEL = re.compile(r"ob_(dense|t16|t32)_(wr|mm)_kernel")


def _objdump():
    tool = shutil.which("llvm-objdump", path=os.path.join(os.path.dirname(os.path.realpath(B._hipcc())), "..", "lib", "llvm", "bin") + ":/opt/rocm/llvm/bin")
    return tool or pytest.skip("no llvm-objdump")


class Kernel:
    """Instructions of one function: ``text[i]`` = (mnemonic, operands), ``target[i]`` = index a branch goes to or None."""

    def __init__(self, name, base, lines):
        self.name, self.text, self.target, at, to = name, [], [], {}, []
        for addr, line, dest in lines:
            at[addr - base] = len(self.text)
            op, _, rest = line.partition(" ")
            self.text.append((op, rest.strip()))
            to.append(dest)
        self.target = [at.get(d) if d is not None else None for d in to]

    def args(self):
        return [int(v) for v in re.findall(r"L[ib](\d+)E", self.name)]


def _kernels(src, tmp, KERNEL=KERNEL):
    lib, sources = LIBS.get(src, (B.LIB, B.SOURCES))
    if not os.path.exists(B._obj(src)):
        B.build(lib=lib, sources=sources)
    data = open(B._obj(src), "rb").read()
    at = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    (n,), p = struct.unpack_from("<Q", data, at + 24), at + 32
    for _ in range(n):
        off, size, idlen = struct.unpack_from("<QQQ", data, p)
        if b"gfx950" in data[p + 24:p + 24 + idlen]:
            break
        p += 24 + idlen
    co = os.path.join(str(tmp), src + ".co")
    open(co, "wb").write(data[at + off:at + off + size])
    out, name = [], None
    proc = subprocess.Popen([_objdump(), "-d", "--no-show-raw-insn", co], stdout=subprocess.PIPE, text=True)
    for line in proc.stdout:
        m = re.match(r"([0-9a-f]+) <(\S+)>:", line)
        if m:
            base, name = int(m[1], 16), m[2] if KERNEL.search(m[2]) else None
            if name:
                out.append((name, base, []))
            continue
        m = name and re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):(?:.*<[^>]*?(?:\+0x([0-9a-f]+))?>)?", line)
        if m:
            dest = (int(m[3], 16) if m[3] else 0) if m[1].startswith(("s_cbranch", "s_branch")) else None
            out[-1][2].append((int(m[2], 16), m[1], dest))
    assert proc.wait() == 0
    return [Kernel(*k) for k in out]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("code")
    return [k for src in LIBS for k in _kernels(src, tmp)]


def _vmcnt(ops):
    m = re.search(r"vmcnt\((\d+)\)", ops)
    return int(m[1]) if m else None


def _late_transfers(k, most):
    """Largest number of transfers to the LDS that may still be on their way behind a barrier, by the waits directly in front of barriers.  ``most``: those allowed;
    paths end where the loop drains everything, or at the first barrier with more."""
    worst, seen, todo = 0, set(), [(0, ())]
    while todo:
        i, queue = todo.pop()
        while (i, queue) not in seen:
            seen.add((i, queue))
            op, ops = k.text[i]
            if op == "s_endpgm":
                break
            if op.startswith("global_load_lds"):
                queue = (queue + ("T",))[-64:]
            elif re.match(r"(global|flat|buffer|scratch)_(load|store|atomic)", op):
                queue = (queue + ("L",))[-64:]
            elif op == "s_waitcnt" and _vmcnt(ops) is not None:
                if k.text[i + 1][0] == "s_barrier":
                    queue = queue[-_vmcnt(ops):] if _vmcnt(ops) else ()
                    worst = max(worst, queue.count("T"))
                    if worst > most:
                        return worst
                elif _vmcnt(ops) == 0 and k.text[i + 1] == ("s_nop", "15"):
                    break                                                # the end of the loop: everything has landed
            if k.target[i] is not None:
                if op == "s_branch":
                    i = k.target[i]
                    continue
                todo.append((k.target[i], queue))
            i += 1
    return worst


def test_barriers_wait_for_the_tile_they_publish(kernels):
    checked = 0
    for k in kernels:
        if "_wr_" not in k.name:
            continue
        a = k.args()
        mt = a[1] if "dense" in k.name else a[-1]
        nst, per = (a[2], (mt + 3) // 4) if "dense" in k.name else (5 if mt < 8 else 4, mt // 4)
        late = _late_transfers(k, (nst - 2) * per)
        assert late <= (nst - 2) * per, f"{k.name}: {late} transfers on their way behind a barrier, {(nst - 2) * per} are of later steps"
        assert late == (nst - 2) * per, f"{k.name}: the steady step waits for more than it has to"
        checked += 1
    assert checked >= 30


def _regs(ops, kind="v"):
    out = set()
    for m in re.finditer(rf"\b{kind}(?:(\d+)|\[(\d+):(\d+)\])", ops):
        out |= {int(m[1])} if m[1] else set(range(int(m[2]), int(m[3]) + 1))
    return out


def _operands_are_ready(kernels, scratch="scratch_"):
    products = 0
    for k in kernels:
        mf = [i for i, (op, _) in enumerate(k.text) if op.startswith("v_mfma")]
        products += len(mf)
        assert not any(op.startswith(scratch) for op, _ in k.text[mf[0]:mf[-1]]), f"{k.name}: a register in scratch between products"
        for i in mf:
            parts = re.findall(r"[va]\[\d+:\d+\]", k.text[i][1])
            assert len(parts) == 4 and parts[0] == parts[3] and parts[0][0] == "a" and parts[1][0] == parts[2][0] == "v", (k.name, k.text[i])
            operands, sums, states, j = _regs(parts[1]) | _regs(parts[2]), _regs(parts[0], "a"), 0, i - 1
            while states < 2 and j >= 0:                                 # (an operand may also come from in front of a branch: the loop's first product)
                op, ops = k.text[j]
                if op.startswith("v_") and not op.startswith(("v_mfma", "v_cmp", "v_readfirstlane")):
                    to = ops.split(",")[0]
                    assert not _regs(to) & operands and not _regs(to, "a") & sums, f"{k.name}: {op} {ops} in front of {k.text[i]}"
                states += 1 + (int(ops) if op == "s_nop" else 0)
                j -= 1
    return products


def test_operands_are_not_written_in_front_of_their_products(kernels):
    assert _operands_are_ready(kernels) > 5000


@pytest.fixture(scope="module")
def one_bit(tmp_path_factory):
    """The 1-bit LDS-DMA product (csrc/ob_gemm2.h, ob_gemm3_body): single, grouped and K-sliced, every tile."""
    return _kernels("onebit_hip.hip", tmp_path_factory.mktemp("one_bit"), re.compile(r"ob_gemm3(g|ks)?_f16_kernel"))


def _tile(k):
    rt, wn = k.args()[-2:]
    per = (128 if wn == 4 else 32 * rt) // 32                            # transfers of a wave and step; wn / 2 more for a quad's weights
    return rt, wn, 2 * per + wn // 2


def test_one_bit_products_wait_for_the_tile_they_publish(one_bit):
    assert len({k.name for k in one_bit}) == 20
    for k in one_bit:
        most = _tile(k)[2]
        late = _late_transfers(k, most)
        assert late == most, f"{k.name}: {late} transfers on their way behind a barrier, {most} are of later steps"


def test_one_bit_operands_are_not_written_in_front_of_their_products(one_bit):
    assert _operands_are_ready(one_bit, "scratch_load") > 5000             # (the largest tile stores what its epilogue reads, in front of its last steps)


def test_small_float32_train_product_computes_one_transform_an_operand(tmp_path):
    """ob_tgemm_kernel's forward instance: the weights' signs are two comparisons of each of a thread's eight elements, the activations' products none."""
    ks = _kernels("onebit_train.hip", tmp_path, re.compile(r"ob_tgemm_kernel(ILb1ELb1ELi1ELi3|\d)"))
    assert len(ks) == 1
    assert sum(bool(re.match(r"v_cmpx?_n?(gt|lt|ge|le)_f32", op)) for op, _ in ks[0].text) == 16
