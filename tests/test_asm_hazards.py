"""The attention kernels' inline assembly in the compiled code.

The compiler knows neither that an inline MFMA is one nor that an inline LDS
read lands later than its statement, so it inserts no wait states and no waits
for them.  The kernels keep the distances by their layout; these tests read the
gfx950 assembly that this tree's sources compile to and check that they hold:

* no VALU instruction writes an operand of an MFMA in the two instructions
  before it (the compiler keeps that distance for the MFMAs it knows);
* no VALU instruction touches an MFMA's result sooner than RESULT_STATES
  wait states after it, and no other MFMA takes it as an A or B operand;
* no instruction touches the destination of an LDS read before a wait that
  covers it (LDS operations return in order).
"""
import os
import re
import subprocess

import pytest

from dsa_amd import build

OPERAND_STATES = 2
# a 16x16x32 bf16 MFMA takes four passes; its result is there after at most four more
RESULT_STATES = 8
MFMA_STATES = 4  # passes that a following MFMA waits for the unit

_REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def _regs(text):
    out = set()
    for m in _REG.finditer(text):
        if m.group(4) is not None:
            out.add((m.group(1), int(m.group(4))))
        else:
            out.update((m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1))
    return out


def _is_valu(op):
    return op.startswith("v_") and not op.startswith("v_mfma") and not op.startswith("v_nop")


def _parse(line):
    """(opcode, [operands]) of an instruction line, or None."""
    line = line.split(";")[0].strip()
    if not line or line.endswith(":") or line.startswith("."):
        return None
    op, _, rest = line.partition(" ")
    op = op.split("\t")[0]
    rest = line[len(op):]
    return op, [x.strip() for x in re.split(r",(?![^\[]*\])", rest)]


def _written(op, args):
    if not args or not args[0]:
        return set()
    if op.startswith(("ds_write", "ds_store", "buffer_store", "global_store", "flat_store", "scratch_store", "s_")):
        return set()
    if " lds" in " ".join(args) or "_lds_" in op:
        return set()
    if "swap" in op:
        return _regs(args[0]) | _regs(args[1])
    return _regs(args[0])


def violations(lines):
    """Broken distances in a kernel's instructions, in text order.  Behind a jump
    the state is that of the first jump to the label that follows."""
    found = []
    recent = []    # (wait states, opcode, registers a VALU instruction wrote)
    results = {}   # register of an MFMA result -> wait states since
    in_flight = []  # destinations of LDS reads, oldest first (empty: another LDS operation)
    at_label, reached = {}, True
    for n, line in enumerate(lines):
        label = re.match(r"\s*(\.L\w+):", line)
        if label and not reached:
            recent, results, in_flight = at_label.get(label.group(1), ([], {}, []))
            recent, results, in_flight = list(recent), dict(results), list(in_flight)
            reached = True
        ins = _parse(line)
        if ins is None:
            continue
        op, args = ins
        if op.startswith(("s_branch", "s_cbranch")):
            at_label.setdefault(args[0], (list(recent), dict(results), list(in_flight)))
        if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
            reached = False
        if op == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", line)
            if m:
                keep = int(m.group(1))
                in_flight = in_flight[len(in_flight) - keep:] if keep and len(in_flight) > keep else (in_flight if keep else [])
            elif "cnt(" not in line:  # a plain number: taken as a full wait only where its LDS field is 0
                value = int(line.split()[-1], 0)
                if (value >> 8) & 0xF == 0:
                    in_flight = []
        touched = set().union(*[_regs(a) for a in args]) if args else set()
        for dst in in_flight:
            if dst & touched:
                found.append((n, "LDS read in flight", line.strip()))
        written = _written(op, args)
        mfma = op.startswith("v_mfma")
        if mfma:
            reads = set().union(*[_regs(a) for a in args[1:4]])
            states = 0
            for cost, what, regs in reversed(recent):
                if states >= OPERAND_STATES:
                    break
                if regs & reads:
                    found.append((n, f"{what} writes an operand {states} states before", line.strip()))
                states += cost
            early = (_regs(args[1]) | _regs(args[2])) & set(results)
            if any(results[r] < RESULT_STATES for r in early):
                found.append((n, "MFMA result as an operand", line.strip()))
        elif _is_valu(op):
            for r in touched & set(results):
                if results[r] < RESULT_STATES:
                    found.append((n, f"MFMA result {results[r]} states after", line.strip()))
                    break
        cost = 1
        if op == "s_nop":
            cost = int(args[0], 0) + 1
        elif mfma:
            cost = MFMA_STATES
        results = {r: s + cost for r, s in results.items() if s + cost < RESULT_STATES}
        if mfma:
            results.update({r: 0 for r in written})
        recent.append((cost if not mfma else 1, op, written if _is_valu(op) else set()))
        del recent[:-8]
        if op.startswith("ds_"):
            reads_lds = op.startswith(("ds_read", "ds_load"))
            in_flight.append(_regs(args[0]) if reads_lds else set())
    return found


def kernels(asm):
    """{demangled-enough name: instruction lines} of the code object's functions."""
    out, name = {}, None
    for line in asm.splitlines():
        m = re.match(r"^(_Z\w+):", line)
        if m:
            name = m.group(1)
            out[name] = []
        elif name and line.startswith(".Lfunc_end"):
            name = None
        elif name:
            out[name].append(line)
    return out


@pytest.fixture(scope="module")
def attention_asm(tmp_path_factory):
    if not os.path.exists(build.hipcc()):
        pytest.skip("no hipcc")
    path = str(tmp_path_factory.mktemp("asm") / "attention.s")
    subprocess.run([build.hipcc(), *build.COMMON_FLAGS, *build.OPT_FLAGS, "--cuda-device-only", "-S", "-o", path,
                    os.path.join(build.CSRC_DIR, "dsa_attention.hip")], check=True, stderr=subprocess.DEVNULL)
    with open(path) as f:
        return kernels(f.read())


@pytest.mark.parametrize("kernel,args,mfmas", [("dsa_attn_ring_kernel", "ILi4ELi1ELb1E", 100),
                                               ("dsa_attn_ring_kernel", "ILi4ELi1ELb0E", 100),
                                               ("dsa_attn_ring_kernel", "ILi8ELi1ELb1E", 100),
                                               ("dsa_attn_ring_kernel", "ILi8ELi1ELb0E", 100),
                                               ("dsa_attn_ring_kernel", "ILi8ELi4ELb1E", 18),
                                               ("dsa_attn_ring_kernel", "ILi8ELi4ELb0E", 18),
                                               ("dsa_attn_wave_kernel", "ILb1E", 50),
                                               ("dsa_attn_wave_kernel", "ILb0E", 50)])
def test_attention_kernels_keep_their_distances(attention_asm, kernel, args, mfmas):
    names = [n for n in attention_asm if kernel + args in n]
    assert len(names) == 1, names
    lines = attention_asm[names[0]]
    assert sum(" v_mfma" in ln or "\tv_mfma" in ln for ln in lines) >= mfmas
    found = violations(lines)
    assert not found, f"{len(found)} broken distances, the first ones: {found[:5]}"


@pytest.mark.parametrize("text,broken", [
    # a copy right before an MFMA that reads it, one instruction further, two
    ("v_mov_b32_e32 v4, v9\nv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", 1),
    ("v_mov_b32_e32 v4, v9\ns_add_u32 s0, s0, s1\nv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", 1),
    ("v_mov_b32_e32 v4, v9\ns_nop 1\nv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", 0),
    ("v_mov_b32_e32 v12, v9\nv_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]", 0),
    # an accumulator read too early, and behind enough wait states
    ("v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]\nv_accvgpr_read_b32 v1, a2", 1),
    ("v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]\ns_nop 7\nv_accvgpr_read_b32 v1, a2", 0),
    # an LDS read's destination before its wait: copied, overwritten, waited for in part, in full
    ("ds_read_b128 v[4:7], v1\nv_mov_b32_e32 v20, v5\ns_waitcnt lgkmcnt(0)", 1),
    ("ds_read_b128 v[4:7], v1\nv_mov_b32_e32 v5, 0\ns_waitcnt lgkmcnt(0)", 1),
    ("ds_read_b128 v[4:7], v1\nds_read_b32 v8, v1\ns_waitcnt lgkmcnt(1)\nv_mov_b32_e32 v20, v5\nv_mov_b32_e32 v21, v8", 1),
    ("ds_read_b128 v[4:7], v1\nds_read_b32 v8, v1\ns_waitcnt lgkmcnt(0)\nv_mov_b32_e32 v20, v5\nv_mov_b32_e32 v21, v8", 0),
    ("buffer_load_dwordx4 v4, s[0:3], 0 offen lds\nv_mov_b32_e32 v4, 0", 0),
    # the two sides of a branch
    ("s_cbranch_vccnz .LBB0_1\nds_read_b32 v1, v2\ns_branch .LBB0_2\n.LBB0_1:\nv_mov_b32_e32 v1, -1\n.LBB0_2:\ns_endpgm", 0),
    ("ds_read_b32 v1, v2\ns_cbranch_vccnz .LBB0_1\ns_branch .LBB0_2\n.LBB0_1:\nv_mov_b32_e32 v1, -1\n.LBB0_2:\ns_endpgm", 1),
])
def test_the_check_sees_broken_distances(text, broken):
    assert len(violations(text.splitlines())) == broken
