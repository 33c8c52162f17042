"""CPU: checks of the assembly of every kernel, for what no result shows
reliably: the wait states that gfx950 leaves to software, and spills.

Wait states.  The compiler keeps them for its own instructions, but does not
see those inside an asm statement, and may put its copies right before or
behind one; so the whole listing is checked, along every path.

Rules (wait states between the two; an instruction in between counts one, s_nop
n counts n + 1; AMD CDNA3 ISA guide, required software wait states, and LLVM's
GCNHazardRecognizer for gfx940 and later):
  VALU writes a VGPR            -> DPP or v_permlane reads it            2
                                -> v_readlane / v_readfirstlane reads it 1
  transcendental writes a VGPR  -> other VALU reads it                   1
  VALU writes an SGPR or VCC    -> VALU reads it                         2
                                -> v_readlane / v_writelane lane select  4
                                -> v_div_fmas reads VCC                  4
                                -> vector memory reads it                5
  VALU writes EXEC              -> DPP                                   5"""
import concurrent.futures as cf
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "gpu-pcg-tracking_amd"))
import build as recipe  # noqa: E402

FAR = 8  # more wait states than any rule asks for
TRANS = ("v_rcp_", "v_rsq_", "v_sqrt_", "v_exp_", "v_log_", "v_sin_", "v_cos_")
DPP = re.compile(r"\b(quad_perm|row_\w+|wave_\w+):|\brow_mirror\b|\brow_half_mirror\b")
REG = re.compile(r"\b(vcc|exec)(?:_lo|_hi)?\b|(?<![\w.])([vsa])(?:(\d+)\b|\[(\d+):(\d+)\])")


def _regs(text):
    out = set()
    for m in REG.finditer(text):
        if m.group(1):
            out.add(m.group(1))
        elif m.group(3):
            out.add(m.group(2) + m.group(3))
        else:
            out.update(m.group(2) + str(k) for k in range(int(m.group(4)), int(m.group(5)) + 1))
    return out


class Inst:
    """Registers written and read, by kind, of one line of assembly."""

    def __init__(self, line, text):
        self.line, self.text = line, text
        self.op, _, rest = text.partition(" ")
        ops = [o.strip() for o in rest.split(",")] if rest else []
        self.dpp = bool(DPP.search(rest)) and self.op.startswith("v_")
        self.valu = self.op.startswith("v_")
        self.trans = self.op.startswith(TRANS)
        self.lane_op = self.op.startswith(("v_readlane", "v_readfirstlane", "v_writelane"))
        n_dst = 0
        if self.valu and ops and self.op != "v_nop":
            n_dst = 1
            if self.op.startswith("v_div_scale") or "_co_" in self.op or self.op.startswith(("v_mad_u64_u32", "v_mad_i64_i32")):
                n_dst = 2
        dst, src = ops[:n_dst], ops[n_dst:]
        self.writes = set().union(*map(_regs, dst)) if dst else set()
        self.reads = set().union(*map(_regs, src)) if src else set()
        if "swap" in self.op and self.valu:
            self.writes = self.reads = _regs(rest)
        if self.op.startswith(("v_fmac", "v_writelane", "v_dot2c", "v_mac")):
            self.reads = self.reads | self.writes
        if self.op.startswith("v_cmpx"):
            self.writes = self.writes | {"exec"}
        if self.op.startswith("v_div_fmas"):
            self.reads = self.reads | {"vcc"}
        self.dpp_src = _regs(src[0]) if self.dpp and src else set()
        self.mem = self.op.startswith(("global_", "buffer_", "flat_", "scratch_"))
        self.mem_reads = _regs(rest) if self.mem else set()
        self.select = _regs(src[1]) if self.op.startswith(("v_readlane", "v_writelane")) and len(src) > 1 else set()

    @property
    def advance(self):
        m = re.match(r"s_nop\s+(0x[0-9a-f]+|\d+)", self.text)
        return int(m.group(1), 0) + 1 if m else 1

    def needs(self):
        """(register, wait states, written by a transcendental only)"""
        for r in self.dpp_src:
            yield r, 2, False
        if self.dpp:
            yield "exec", 5, False
        if self.valu:
            scalar = {r for r in self.reads if r[0] == "s" or r == "vcc"}
            for r in scalar:
                yield r, 4 if r in self.select or (r == "vcc" and self.op.startswith("v_div_fmas")) else 2, False
            vector = self.reads - scalar - {"exec"}
            for r in vector:
                if self.op.startswith(("v_readlane", "v_readfirstlane")):
                    yield r, 1, False
                if self.op.startswith("v_permlane"):
                    yield r, 2, False
                if not self.trans:
                    yield r, 1, True
        for r in self.mem_reads:
            if r[0] == "s" or r == "vcc":
                yield r, 5, False


def _blocks(text):
    """Basic blocks of each function: {label: (instructions, successors)}."""
    funcs, blocks, name, cur = [], None, None, None
    for no, raw in enumerate(text.splitlines(), 1):
        line = raw.split(";")[0].strip()
        if not line:
            continue
        if line.startswith(".type") and "@function" in line:
            blocks = {}
            funcs.append((line.split()[1].split(",")[0], blocks))
            name = None
        m = re.match(r"([\w.$]+):", line)
        if m and blocks is not None:
            prev, name = name, m.group(1)
            cur = blocks[name] = ([], [])
            if prev is not None and blocks[prev][1] is not None and not _ends(blocks[prev][0]):
                blocks[prev][1].append(name)
            continue
        if blocks is None or cur is None or line.startswith("."):
            if line.startswith((".section", ".size")):
                blocks, cur = None, None
            continue
        for part in line.split("\n"):
            inst = Inst(no, re.sub(r"\s+", " ", part))
            cur[0].append(inst)
            if inst.op.startswith(("s_cbranch", "s_branch")):
                cur[1].append(inst.text.split()[-1])
                prev, name = name, f"{name}+{no}"
                cur = blocks[name] = ([], [])
                if inst.op != "s_branch":
                    blocks[prev][1].append(name)
    return funcs


def _ends(insts):
    return bool(insts) and insts[-1].op.startswith(("s_endpgm", "s_branch", "s_setpc", "s_trap"))


def hazards(text):
    """[(function, line, text, register, wait states found, needed)]"""
    found = []
    for func, blocks in _blocks(text):
        # by register: (wait states since a VALU wrote it, since a transcendental one did)
        start = {b: None for b in blocks}
        if not blocks:
            continue
        first = next(iter(blocks))
        start[first] = {}
        todo = [first]
        bad = {}
        while todo:
            b = todo.pop()
            state = dict(start[b])
            for inst in blocks[b][0]:
                for reg, need, trans in inst.needs():
                    have = state.get(reg, (FAR, FAR))[1 if trans else 0]
                    if have < need:
                        bad[(inst.line, reg, need)] = (func, inst.line, inst.text, reg, have, need)
                step = inst.advance
                state = {r: (a + step, t + step) for r, (a, t) in state.items() if a + step < FAR}
                if inst.valu:
                    for r in inst.writes:
                        state[r] = (0, 0 if inst.trans else FAR)
                elif inst.mem or inst.op.startswith(("ds_", "s_")):
                    # what something else writes comes with its own wait or needs none
                    for r in _regs(inst.text.split(" ", 1)[1].split(",")[0]) if " " in inst.text else ():
                        if inst.op.startswith(("ds_write", "global_store", "buffer_store", "scratch_store", "s_cmp",
                                               "s_bitcmp", "s_waitcnt", "s_nop", "s_cbranch", "s_branch")):
                            break
                        state.pop(r, None)
            for s in blocks[b][1]:
                if s not in start:
                    continue
                if start[s] is None:
                    start[s] = dict(state)
                    todo.append(s)
                    continue
                old, changed = start[s], False
                for r, (a, t) in state.items():
                    oa, ot = old.get(r, (FAR, FAR))
                    if a < oa or t < ot:
                        old[r] = (min(a, oa), min(t, ot))
                        changed = True
                if changed:
                    todo.append(s)
        found += bad.values()
    return found


def _listing(src):
    cmd = [recipe.HIPCC, *recipe.COMMON, *recipe.DEVICE_FLAGS, "--offload-device-only", "-S", "-o", "-", src]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return r.stdout


@pytest.mark.parametrize("code,count", [
    ("v_mov_b32_e32 v1, v2\n v_add_f32_dpp v3, v1, v4 row_ror:1 row_mask:0xf bank_mask:0xf", 1),
    ("v_mov_b32_e32 v1, v2\n s_nop 0\n v_add_f32_dpp v3, v1, v4 row_ror:1 row_mask:0xf bank_mask:0xf", 1),
    ("v_mov_b32_e32 v1, v2\n s_nop 1\n v_add_f32_dpp v3, v1, v4 row_ror:1 row_mask:0xf bank_mask:0xf", 0),
    ("v_mov_b32_e32 v4, v2\n v_add_f32_dpp v3, v1, v4 row_ror:1 row_mask:0xf bank_mask:0xf", 0),  # not the DPP operand
    ("v_readlane_b32 s4, v1, 3\n v_mov_b32_e32 v9, v8\n v_mul_f32_e32 v2, s4, v3", 1),
    ("v_readlane_b32 s4, v1, 3\n s_nop 1\n v_mul_f32_e32 v2, s4, v3", 0),
    ("v_mov_b32_e32 v1, v2\n v_readlane_b32 s4, v1, 3", 1),
    ("v_mov_b32_e32 v1, v2\n s_nop 0\n v_permlane16_swap_b32 v3, v1", 1),
    ("v_rcp_f32_e32 v1, v2\n v_mul_f32_e32 v3, v1, v1", 1),
    ("v_rcp_f32_e32 v1, v2\n s_nop 0\n v_mul_f32_e32 v3, v1, v1", 0),
    # the write at the loop's end, the read at its start
    ("s_nop 7\n.LBB0_1:\n v_add_f32_dpp v3, v1, v4 row_ror:1 row_mask:0xf bank_mask:0xf\n v_mov_b32_e32 v1, v2\n"
     " s_cbranch_scc1 .LBB0_1", 1),
])
def test_the_check_itself(code, count):
    assert len(hazards(f".type f,@function\nf:\n {code}\n s_endpgm\n")) == count


@pytest.fixture(scope="module")
def listings():
    srcs = [s for s in recipe.sources() if s.endswith(".hip")]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        out = dict(zip(map(os.path.basename, srcs), ex.map(_listing, srcs)))
    assert sum(text.count("\ts_endpgm") for text in out.values()) > 30
    return out


def test_kernels_keep_the_wait_states(listings):
    found = [(name, *h) for name, text in listings.items() for h in hazards(text)]
    for h in found[:40]:
        print(h)
    assert not found, f"{len(found)} reads too close to a write"


def narrow_spills(text):
    """[(line, text)] of register spills ahead of the s_or_b64 exec of their block,
    which store the lanes of the branch that ends there and no others."""
    found, block = [], []
    for no, line in enumerate(text.splitlines(), 1):
        if re.match(r"[\w.$]+:|; %bb\.", line):
            block = []
        if "Folded Spill" in line or ("Reload Reuse" in line and "v_accvgpr_write" in line):
            block.append((no, line.strip()))
        if re.match(r"\s*s_or_b64 exec, exec,", line):
            found += block
            block = []
    return found


def test_spills_store_every_lane(listings):
    """The compiler has put the spill of a value for all lanes ahead of the end
    of a branch that only some had taken; reloaded for the others it was
    whatever the slot held (a team kernel then stored knots of lambda in wrong
    places)."""
    assert narrow_spills("; %bb.1:\n\tscratch_store_dword off, v1, off ; 4-byte Folded Spill\n"
                         "\ts_or_b64 exec, exec, s[0:1]\n") != []
    assert narrow_spills("; %bb.1:\n\ts_or_b64 exec, exec, s[0:1]\n"
                         "\tscratch_store_dword off, v1, off ; 4-byte Folded Spill\n") == []
    found = [(name, *f) for name, text in listings.items() for f in narrow_spills(text)]
    assert not found, found
