"""CPU check of the built prefill and LM-head code for what the compiler cannot see in their inline
assembly. prefill_kernel writes its MFMAs out, and the compiler adds no wait states to instructions it does
not know: the order of the stream has to keep a result from being touched before it is written and an
operand from being read right after a vector instruction wrote it. Its loads to LDS set M0 themselves:
nothing else in those kernels may use M0. Each kernel's code is followed along all its branches."""
import re
import subprocess
from pathlib import Path

import pytest

from pagedkv import _lib

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
# wait states (instructions, or 4 cycles) until an MFMA's result may be touched by anything but the next
# accumulation: its passes and 4 more; an MFMA issues when the one before it has left the first pass, so
# it covers its predecessor's passes
PASSES = {"v_mfma_f32_32x32x16_bf16": 8, "v_mfma_f32_4x4x4_16b_bf16": 2}
AFTER_VALU = 2  # wait states between a vector instruction and an MFMA that reads its result

_REG = re.compile(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b")


def _regs(text):
    out = set()
    for kind, lo, hi, kind1, one in _REG.findall(text):
        out |= {kind + str(i) for i in range(int(lo), int(hi) + 1)} if kind else {kind1 + one}
    return out


class Insn:
    def __init__(self, text):
        self.op, _, rest = text.partition(" ")
        self.text = text
        self.ops = [o.strip() for o in re.split(r",(?![^\[]*\])", rest)] if rest else []
        self.mfma = "mfma" in self.op
        # what it writes comes first, except for stores and loads to LDS, which write no register
        store = "store" in self.op or "_write" in self.op or "lds_dword" in self.op
        first = self.ops[:1] if not store else []
        if self.op.startswith("v_permlane32_swap"):
            first = self.ops[:2]
        self.dst = set().union(*[_regs(o) for o in first]) if first else set()
        self.src = set().union(*[_regs(o) for o in self.ops[len(first):]]) if self.ops[len(first):] else set()
        if re.match(r"v_(fmac|dot2c|mac|permlane|accvgpr_write)|.*d16_hi", self.op):
            self.src |= self.dst
        self.states = int(self.ops[0], 0) + 1 if self.op == "s_nop" else 1

    @property
    def valu(self):
        return self.op.startswith("v_") and not self.mfma


def _step(insn, state, report):
    """state: (register -> wait states that its MFMA result still needs, register -> states since a vector
    instruction wrote it); both are moved on past insn."""
    pend, wrote = state
    if insn.mfma:
        acc = _regs(insn.ops[0])
        for r in _regs(insn.ops[1]) | _regs(insn.ops[2]) | (_regs(insn.ops[3]) - acc):
            if wrote.get(r, AFTER_VALU) < AFTER_VALU:
                report(f"{r} read {wrote[r]} states after a vector write: {insn.text}")
            if pend.get(r, 0) > 0:
                report(f"{r} is an operand {pend[r]} states before its result is written: {insn.text}")
        for r in acc & _regs(insn.ops[3]):
            if wrote.get(r, AFTER_VALU) < AFTER_VALU:
                report(f"{r} accumulated {wrote[r]} states after a vector write: {insn.text}")
    else:
        for r in insn.src | insn.dst:
            if pend.get(r, 0) > 0:
                report(f"{r} touched {pend[r]} states early: {insn.text}")
    states = PASSES[insn.op] if insn.mfma else insn.states
    for r in [r for r in pend if pend[r] <= states]:
        del pend[r]
    for r in pend:
        pend[r] -= states
    for r in [r for r in wrote if wrote[r] + states >= AFTER_VALU]:
        del wrote[r]
    for r in wrote:
        wrote[r] += states
    if insn.mfma:
        for r in insn.dst:
            pend[r] = PASSES[insn.op] + 4
            wrote.pop(r, None)
    elif insn.valu:
        for r in insn.dst:
            wrote[r] = 0


def check_stream(code):
    """code: [(address, text, branch target or None)] of one kernel. Violations, along every path."""
    insns = [Insn(t) for _, t, _ in code]
    at = {a: i for i, (a, _, _) in enumerate(code)}
    heads = {0} | {at[t] for _, _, t in code if t is not None} | \
        {i + 1 for i, (_, _, t) in enumerate(code) if t is not None and i + 1 < len(code)}
    found, seen = {}, {}
    work = [(0, ({}, {}))]
    while work:
        i, (pend, wrote) = work.pop()
        if i in seen:  # join: the longest remaining wait, the most recent write
            p0, w0 = seen[i]
            if all(p0.get(r, 0) >= n for r, n in pend.items()) and all(w0.get(r, 9) <= n for r, n in wrote.items()):
                continue
            pend = {r: max(pend.get(r, 0), p0.get(r, 0)) for r in {*pend, *p0}}
            wrote = {r: min(wrote.get(r, 9), w0.get(r, 9)) for r in {*wrote, *w0}}
        seen[i] = (dict(pend), dict(wrote))
        state = (dict(pend), dict(wrote))
        while True:
            _step(insns[i], state, lambda m, i=i: found.setdefault(i, m))
            op, target = insns[i].op, code[i][2]
            if target is not None:
                work.append((at[target], (dict(state[0]), dict(state[1]))))
            if op in ("s_branch", "s_endpgm", "s_setpc_b64") or i + 1 == len(code):
                break
            i += 1
            if i in heads:
                work.append((i, state))
                break
    return list(found.values())


def check_m0(code):
    """M0 is set only right before a load to LDS, and used by nothing else."""
    bad = []
    for i, (_, text, _) in enumerate(code):
        if re.search(r"\bm0\b", text) and not text.startswith("s_mov_b32 m0, "):
            bad.append(text)
        if text.startswith("s_mov_b32 m0, ") and not (code[i + 1][1].startswith("s_nop") and
                                                      code[i + 2][1].startswith("global_load_lds_dwordx4")):
            bad.append(text + " without its load")
        if "load_lds" in text and not any(t.startswith("s_mov_b32 m0, ") for _, t, _ in code[max(0, i - 6):i]):
            bad.append(text + " without its M0")
    return bad


def _kernels(tmp, wanted):
    """Disassembled kernels of libpagedkv.so whose symbols contain `wanted`."""
    lib = tmp / "lib.so"
    lib.symlink_to(_lib.LIB_PATH)
    subprocess.run([OBJDUMP, "--offloading", lib.name], cwd=tmp, check=True, capture_output=True)
    out = {}
    for obj in sorted(tmp.glob("lib.so.*gfx950")):
        if wanted.encode() not in obj.read_bytes():
            continue
        text = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True, text=True).stdout
        for m in re.finditer(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^\s*$|\Z)", text, re.M | re.S):
            name, body = m.groups()
            if wanted not in name:
                continue
            code = []
            for line in body.splitlines():
                insn, _, tail = line.partition("//")
                addr = re.match(r"\s*([0-9A-Fa-f]+):", tail)
                if not insn.strip() or not addr:
                    continue
                insn = re.sub(r"\s+", " ", insn.strip())
                branch = None
                if re.match(r"s_(c?branch)", insn):
                    b = re.search(r"<\S+?\+0x([0-9a-fA-F]+)>|<(\S+)>", tail)
                    branch = (int(b.group(1), 16) if b and b.group(1) else 0)
                code.append((int(addr.group(1), 16), insn, branch))
            base = code[0][0]
            out[name] = [(a - base, t, b) for a, t, b in code]
    return out


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not OBJDUMP.exists():
        pytest.skip("llvm-objdump not installed")
    _lib.lib()
    cache = {}

    def get(wanted):
        if wanted not in cache:
            cache[wanted] = _kernels(tmp_path_factory.mktemp("code"), wanted)
        return cache[wanted]

    return get


def test_prefill_kernel_wait_states(kernels):
    found = kernels("14prefill_kernelI")
    assert len(found) == 16
    for name, code in found.items():
        mfmas = sum("mfma" in t for _, t, _ in code)
        assert mfmas > 200, f"{name}: {mfmas} MFMAs"
        assert not check_stream(code), name


def test_m0_belongs_to_the_loads_to_lds(kernels):
    for wanted, count in (("14prefill_kernelI", 16), ("lm_head_split", 3)):
        found = kernels(wanted)
        assert len(found) == count
        for name, code in found.items():
            assert any("load_lds" in t for _, t, _ in code), name
            assert not check_m0(code), name


def _code(text):
    lines = [line.strip() for line in text.strip().splitlines()]
    return [(4 * i, re.sub(r" -> \d+$", "", line), 4 * int(line.split("-> ")[1]) if "->" in line else None)
            for i, line in enumerate(lines)]


@pytest.mark.parametrize("text,bad", [
    # an operand written one instruction before
    ("v_mov_b32_e32 v4, 0\nv_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\ns_endpgm", 1),
    ("v_mov_b32_e32 v4, 0\ns_nop 1\nv_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\ns_endpgm", 0),
    # a result read after 11 and after 12 wait states
    ("v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\ns_nop 10\nv_add_f32_e32 v0, v16, v1\ns_endpgm", 1),
    ("v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\ns_nop 11\nv_add_f32_e32 v0, v16, v1\ns_endpgm", 0),
    # accumulation in place needs none; an accumulator that LDS data overwrites does
    ("v_mfma_f32_32x32x16_bf16 a[16:31], v[4:7], v[8:11], 0\n"
     "v_mfma_f32_32x32x16_bf16 a[16:31], v[4:7], v[8:11], a[16:31]\ns_endpgm", 0),
    ("v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\nds_read_b128 v[16:19], v0\ns_endpgm", 1),
    # only along the back edge of a loop
    ("s_nop 0\nv_add_f32_e32 v0, v16, v1\ns_nop 15\nv_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\n"
     "s_cbranch_scc1 1 -> 1\ns_endpgm", 1),
    ("s_nop 0\nv_add_f32_e32 v0, v16, v1\nv_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], 0\n"
     "s_nop 11\ns_cbranch_scc1 1 -> 1\ns_endpgm", 0),
])
def test_checker_sees_planted_violations(text, bad):
    assert len(check_stream(_code(text))) == bad


def test_checker_sees_planted_m0_uses():
    load = "s_mov_b32 m0, s3\ns_nop 0\nglobal_load_lds_dwordx4 v1, s[2:3] offset:1024\n"
    assert not check_m0(_code(load + "s_endpgm"))
    assert check_m0(_code(load + "s_mov_b32 s4, m0\ns_endpgm"))
    assert check_m0(_code("global_load_lds_dwordx4 v1, s[2:3]\ns_endpgm"))
    assert check_m0(_code("s_mov_b32 m0, -1\nv_nop\nv_nop\ns_endpgm"))
