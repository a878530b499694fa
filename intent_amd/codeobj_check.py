"""Static checks on the gfx950 code object this package builds.

Some pipelines issue LDS DMA (``buffer_load_dword[x4] ... lds``) as inline
assembly that the compiler's wait-count pass does not track (``lds_dma<B,
true>`` and ``lds_store16`` in ``csrc/mfma_pipe.h``). They order every read of
DMA-written LDS with their own ``s_waitcnt`` and barriers, which holds only
while the compiler issues no vector memory operations of its own inside their
loops; a spill reload there would bring its own wait and break that ordering
without any error. Inline assembly also gets no hazard padding from the
compiler. ``check_code_object`` therefore rejects

* scratch use (a non-zero private segment, SGPR or VGPR spills, or any
  ``scratch_*`` instruction) in a kernel that issues untracked LDS DMA (names
  in ``UNTRACKED_DMA_KERNELS``: the packed-weight MoE projections, whose DMA
  comes from ``csrc/w4pk.h``);

and, in every kernel that contains an LDS DMA,

* an LDS DMA fewer than 1 wait state after the SALU write of M0 it uses;
* an LDS DMA fewer than 5 wait states after a VALU write of an SGPR it reads
  (buffer resource or offset).

The wait states are the gfx9 hazard table's (an instruction counts one,
``s_nop N`` counts N + 1).

In every kernel with MFMAs it also rejects an MFMA whose A, B or scale operand
was written while lanes were masked off. MFMAs ignore EXEC and read their
operands from all 64 lanes, but the reads and decodes that produce those operands
obey it. The compiler may move an MFMA with no other use below a per-lane branch
(the rows past M of an epilogue), which is harmless by itself and does happen; it
would be wrong if the operand's own instruction moved with it, since the masked
lanes would then leave their part of the operand stale. Nothing in the source
rules that out everywhere, so the built code is checked, but for
``WAVE_UNIFORM_KERNELS``.

The input is a code object built here from this repository's own sources.
"""
from __future__ import annotations

import re
import subprocess
from dataclasses import dataclass, field
from pathlib import Path

LLVM_BIN = Path("/opt/rocm/llvm/bin")
TARGET = "hipv4-amdgcn-amd-amdhsa--gfx950"

# Kernels whose LDS DMA is the inline-assembly form (the compiler's wait pass
# does not see it). Substrings of the mangled names.
UNTRACKED_DMA_KERNELS = ("moe_gate_up_pk_kernel", "moe_down_pk_kernel")

# Kernels whose K loop the compiler takes for divergent (its bounds come from threadIdx.x >> 6), though
# every lane of a wave agrees: the loads and MFMAs of a step are masked as a whole or not at all.
# Substrings of the mangled names.
WAVE_UNIFORM_KERNELS = ("_117w4a16_gemv_kernel", "_117w8a16_gemv_kernel")

M0_WAIT = 1
VALU_SGPR_WAIT = 5

_TARGET = re.compile(r"<[^>+]+(?:\+0x([0-9a-f]+))?>")
_LABEL = re.compile(r"^[0-9a-f]+ <(?P<name>[^>]+)>:\s*$")
_DMA = re.compile(r"^buffer_load_(dword|dwordx4|ubyte|ushort|sbyte|sshort)\b.*\blds\b")
_SREG = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\b(vcc)\b|\b(m0)\b")


class CodeObjectError(RuntimeError):
    """A kernel of the built library breaks a rule its inline assembly relies on."""


@dataclass
class KernelReport:
    name: str
    dma: int = 0
    scratch_ops: int = 0
    private_segment: int = 0
    spills: int = 0
    problems: list = field(default_factory=list)


def _tool(name: str) -> str:
    path = LLVM_BIN / name
    return str(path) if path.exists() else name


def _run(cmd) -> str:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise CodeObjectError(f"{cmd[0]} failed: {proc.stderr.strip()}")
    return proc.stdout


def extract_device_code(binary: Path, out: Path) -> Path:
    """The gfx950 code object bundled in a host object or shared library."""
    out = Path(out)
    fatbin = out.with_suffix(".fatbin")
    _run([_tool("llvm-objcopy"), f"--dump-section=.hip_fatbin={fatbin}", str(binary), str(out.with_suffix(".host"))])
    _run([_tool("clang-offload-bundler"), "--unbundle", "--type=o", f"--input={fatbin}", f"--targets={TARGET}",
          f"--output={out}"])
    fatbin.unlink(missing_ok=True)
    out.with_suffix(".host").unlink(missing_ok=True)
    return out


def _sregs(text: str) -> set:
    regs = set()
    for m in _SREG.finditer(text):
        if m.group(1) is not None:
            regs.update(f"s{i}" for i in range(int(m.group(1)), int(m.group(2)) + 1))
        elif m.group(3) is not None:
            regs.add(f"s{m.group(3)}")
        elif m.group(4):
            regs.update(("vcc",))
        else:
            regs.add("m0")
    return regs


def _operands(inst: str) -> list:
    parts = inst.split(None, 1)
    if len(parts) < 2:
        return []
    ops, depth, cur = [], 0, ""
    for ch in parts[1]:
        if ch == "[":
            depth += 1
        elif ch == "]":
            depth -= 1
        if ch == "," and depth == 0:
            ops.append(cur.strip())
            cur = ""
        else:
            cur += ch
    if cur.strip():
        ops.append(cur.strip())
    return ops


_CARRY_OUT = re.compile(r"^v_(add|sub|subrev|addc|subb|subbrev)_co_u32|^v_mad_(u64_u32|i64_i32)|^v_div_scale")


def _valu_sgpr_writes(inst: str) -> set:
    """SGPRs (and vcc) a VALU instruction writes."""
    op = inst.split(None, 1)[0]
    ops = _operands(inst)
    if not op.startswith("v_") or not ops:
        return set()
    if op.startswith(("v_readfirstlane", "v_readlane")):
        return _sregs(ops[0])
    if op.startswith(("v_cmp", "v_cmpx")):
        return {"vcc"} if op.endswith("_e32") else _sregs(ops[0])
    if _CARRY_OUT.match(op):
        if op.endswith("_e32"):
            return {"vcc"}
        return _sregs(ops[1]) if len(ops) > 1 else set()
    return set()


def _wait_states(inst: str) -> int:
    if inst.startswith("s_nop"):
        ops = _operands(inst)
        return int(ops[0], 0) + 1 if ops else 1
    return 1


def _dma_sgpr_reads(inst: str) -> set:
    ops = _operands(inst)
    regs = set()
    for o in ops[1:]:
        regs |= _sregs(o)
    return regs


def _check_kernel(name: str, insts: list, meta: dict) -> KernelReport:
    rep = KernelReport(name)
    rep.private_segment = meta.get("private_segment_fixed_size", 0)
    rep.spills = meta.get("sgpr_spill_count", 0) + meta.get("vgpr_spill_count", 0)
    for i, inst in enumerate(insts):
        if inst.startswith("scratch_"):
            rep.scratch_ops += 1
        if not _DMA.match(inst):
            continue
        rep.dma += 1
        reads = _dma_sgpr_reads(inst)
        waits = 0
        m0_seen = False
        for j in range(i - 1, -1, -1):
            prev = insts[j]
            if not m0_seen and re.match(r"^s_\w+\s+m0\b", prev):
                m0_seen = True
                if waits < M0_WAIT:
                    rep.problems.append(f"LDS DMA {waits} wait states after the M0 write: {prev!r} -> {inst!r}")
            hit = _valu_sgpr_writes(prev) & reads
            if hit and waits < VALU_SGPR_WAIT:
                rep.problems.append(
                    f"LDS DMA reads {sorted(hit)} {waits} wait states after a VALU write: {prev!r} -> {inst!r}")
            waits += _wait_states(prev)
            if waits >= VALU_SGPR_WAIT and m0_seen:
                break
            if prev.startswith(("s_endpgm", "s_branch", "s_cbranch", "s_setpc")):
                break
    if rep.dma and any(k in name for k in UNTRACKED_DMA_KERNELS):
        if rep.private_segment:
            rep.problems.append(f"private segment of {rep.private_segment} bytes")
        if rep.spills:
            rep.problems.append(f"{rep.spills} register spills")
        if rep.scratch_ops:
            rep.problems.append(f"{rep.scratch_ops} scratch instructions")
    return rep


_BRANCH = ("s_cbranch", "s_branch", "s_endpgm", "s_setpc")
_VREG = re.compile(r"^([va])(?:(\d+)|\[(\d+):(\d+)\])$")
# Vector instructions whose first operand is not a destination.
_NO_DEST = re.compile(r"^(ds_write|ds_store|global_store|buffer_store|flat_store|scratch_store|global_atomic|"
                      r"buffer_atomic|ds_add|v_cmp|v_readfirstlane|v_readlane|v_nop)")


def _vregs(operand: str) -> set:
    m = _VREG.match(operand)
    if not m:
        return set()
    lo, hi = (m.group(2), m.group(2)) if m.group(2) else (m.group(3), m.group(4))
    return {m.group(1) + str(i) for i in range(int(lo), int(hi) + 1)}


class _Masked:
    """Lanes masked off on some path to a point: the SGPR pairs that hold the EXEC to restore, each
    with those outstanding when it was saved, and the vector registers written since."""

    def __init__(self, saved=None, written=()):
        self.saved = dict(saved or {})
        self.written = set(written)

    def merge(self, other) -> bool:
        before = ({k: set(v) for k, v in self.saved.items()}, len(self.written))
        for reg, outer in other.saved.items():
            self.saved[reg] = self.saved.get(reg, frozenset()) | outer
        self.written |= other.written
        return before != ({k: set(v) for k, v in self.saved.items()}, len(self.written))

    def _restore(self, reg: str) -> None:
        if reg not in self.saved:
            return
        for inner in [k for k, outer in self.saved.items() if k == reg or reg in outer]:
            del self.saved[inner]

    def _save(self, reg: str) -> None:
        self._restore(reg)
        self.saved[reg] = frozenset(self.saved)

    def step(self, inst: str):
        """Applies one instruction; the operands an MFMA reads that were written under a mask."""
        op, _, rest = inst.partition(" ")
        if op.startswith("s_") and "exec" in inst:
            ops = _operands(inst)
            if "saveexec" in op:
                if not op.startswith("s_and_saveexec"):  # the other side of a branch: EXEC is whole between
                    self._restore(ops[1])
                self._save(ops[0])
            elif op == "s_xor_b64" and ops[1] == "exec" and ops[0] != "exec" and ops[2] in self.saved:
                self.saved[ops[0]] = self.saved.pop(ops[2])  # the lanes of the other side, kept for its saveexec
            elif ops[0] == "exec" and op in ("s_or_b64", "s_mov_b64"):
                for reg in ops[1:]:
                    self._restore(reg)
                self._restore("exec")
            elif ops[0] == "exec" and op == "s_andn2_b64":  # lanes that left a loop
                self.saved.setdefault(ops[2], frozenset(self.saved))
            elif ops[0] == "exec" and op == "s_and_b64" and not self.saved:
                self._save("exec")
            if not self.saved:
                self.written.clear()
            return set()
        if not self.saved or not op.startswith(("v_", "ds_", "global_", "buffer_", "flat_", "scratch_")):
            return set()
        ops = _operands(inst)
        if op.startswith("v_mfma"):
            reads = set()
            for o in ops[1:3] + ops[4:]:
                reads |= _vregs(o.split(" ")[0])
            stale = reads & self.written
            self.written -= _vregs(ops[0])  # written in every lane
            return stale
        if ops and not _NO_DEST.match(op) and " lds" not in inst:
            self.written |= _vregs(ops[0])
        return set()


def masked_mfma_operands(insts: list) -> list:
    """The MFMAs of a kernel, (address, text, branch target address or None) per instruction, that
    read an A, B or scale operand written while lanes were masked off."""
    if not any(text.startswith("v_mfma") for _, text, _ in insts):
        return []
    index = {addr: i for i, (addr, _, _) in enumerate(insts)}
    starts = {0}
    for i, (_, text, target) in enumerate(insts):
        if text.startswith(_BRANCH):
            starts.add(i + 1)
            if target in index:
                starts.add(index[target])
    order = sorted(x for x in starts if x < len(insts))
    ends = dict(zip(order, order[1:] + [len(insts)]))
    state = {0: _Masked()}
    work = [0]
    while work:
        first = work.pop()
        cur = _Masked(state[first].saved, state[first].written)
        for i in range(first, ends[first]):
            cur.step(insts[i][1])
        _, last, target = insts[ends[first] - 1]
        following = []
        if not last.startswith(("s_branch", "s_endpgm", "s_setpc")) and ends[first] < len(insts):
            following.append(ends[first])
        if last.startswith(("s_branch", "s_cbranch")) and target in index:
            following.append(index[target])
        for nxt in following:
            if nxt not in state:
                state[nxt] = _Masked(cur.saved, cur.written)
                work.append(nxt)
            elif state[nxt].merge(cur):
                work.append(nxt)
    problems = []
    for first in order:
        if first not in state:
            continue  # padding
        cur = _Masked(state[first].saved, state[first].written)
        for i in range(first, ends[first]):
            stale = cur.step(insts[i][1])
            if stale:
                problems.append(f"operand {sorted(stale)} was written with lanes masked off: {insts[i][1]!r}")
    return problems


def _metadata(code_object: Path) -> dict:
    notes = _run([_tool("llvm-readelf"), "--notes", str(code_object)])
    meta, cur = {}, None
    for line in notes.splitlines():
        s = line.strip()
        m = re.match(r"^-?\s*\.name:\s+(\S+)", s)
        if m:
            cur = meta.setdefault(m.group(1), {})
            continue
        m = re.match(r"^-?\s*\.(private_segment_fixed_size|sgpr_spill_count|vgpr_spill_count):\s+(\d+)", s)
        if m and cur is not None:
            cur[m.group(1)] = int(m.group(2))
    return meta


def check_code_object(code_object: Path) -> list:
    """Reports for every kernel of a gfx950 code object; raises CodeObjectError
    listing every kernel that breaks a rule above."""
    meta = _metadata(code_object)
    dis = _run([_tool("llvm-objdump"), "-d", "--no-show-raw-insn", str(code_object)])
    kernels, name, insts, base = [], None, [], 0
    for line in dis.splitlines():
        m = _LABEL.match(line)
        if m:
            if name is not None:
                kernels.append((name, insts))
            name, insts, base = m.group("name"), [], int(line.split(" ", 1)[0], 16)
            continue
        s, _, comment = (part.strip() for part in line.partition("//"))
        if name is not None and s:
            addr = int(comment.split(":")[0], 16) if ":" in comment else -1
            to = _TARGET.search(comment)
            insts.append((addr, s, base + int(to.group(1) or "0", 16) if to else None))
    if name is not None:
        kernels.append((name, insts))
    reports = []
    for n, ins in kernels:
        reports.append(_check_kernel(n, [text for _, text, _ in ins], meta.get(n, {})))
        if not any(k in n for k in WAVE_UNIFORM_KERNELS):
            reports[-1].problems.extend(masked_mfma_operands(ins))
    bad = [r for r in reports if r.problems]
    if bad:
        lines = []
        for r in bad:
            lines.append(f"{r.name}:")
            lines.extend(f"  {p}" for p in r.problems[:8])
        raise CodeObjectError("kernels break their scratch, hazard or mask rules:\n" + "\n".join(lines))
    return reports


def check_binary(binary: Path, workdir: Path) -> list:
    """check_code_object on the device code of a host object or shared library."""
    workdir = Path(workdir)
    workdir.mkdir(parents=True, exist_ok=True)
    co = extract_device_code(binary, workdir / (Path(binary).stem + ".gfx950.co"))
    return check_code_object(co)
