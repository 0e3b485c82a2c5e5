"""The built kernels' own code, read on the CPU: no register is touched while a load into it is under way, and no result of a
matrix product before the wait states that it needs have passed, on any path through a kernel.

Reads from LDS by inline assembly are values that the compiler takes to be there at once: it may copy them to other registers
before the wait that the source puts in front of their use.  And it has left out wait states behind a matrix product where one way
round a branch is shorter than the other.  Neither shows in a source file, and the results are wrong only now and then.

Rules (quarter-rate issue slots, as s_nop counts them): a result of v_mfma_f32_16x16x32_bf16 (4 passes) may be read 8 slots later, of
v_mfma_f32_32x32x16_bf16 (8 passes) 12, of v_mfma_f32_32x32x2_f32 (16 passes) 18, and overwritten by the vector ALU one slot earlier
(loads take longer than that to arrive); the next product is issued when the one before it has gone through its passes.  vmcnt and lgkmcnt count vector memory and LDS
operations, which complete in order; scalar loads complete in any order.  What the vector ALU writes may be read across lanes
(DPP, permlane) 2 slots later and, from a scalar register, by a memory address 5 slots later."""
import concurrent.futures
import os
import re
import shutil
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pre-tjax_amd", "libptj.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
RANGE, ONE, COMMA = re.compile(r"\b([vas])\[(\d+):(\d+)\]"), re.compile(r"\b([vas])(\d+)\b"), re.compile(r",(?![^\[]*\])")
NO_RESULT = re.compile(r"s_(cmp|bitcmp|cbranch|branch|barrier|setprio|endpgm|sleep)")
CARRY_OUT = re.compile(r"v_(add|sub|subrev|addc|subb)_co_|v_mad_(u64_u32|i64_i32)|v_div_scale")


def registers(text):
    found = [(k, i) for k, a, b in RANGE.findall(text) for i in range(int(a), int(b) + 1)]
    found += [(k, int(i)) for k, i in ONE.findall(text)]
    return found + ([("s", 106), ("s", 107)] if "vcc" in text else [])


class Instruction:
    def __init__(self, text):
        self.text, (self.op, _, rest) = text, text.partition(" ")
        op, operands = self.op, [x.strip() for x in COMMA.split(rest)]
        self.wait = self.counter = self.load = None
        self.slots, self.passes, self.factors = 1, 0, ()
        self.out = self.into = ()
        vector, lds = re.match(r"(global|buffer|flat|scratch)_", op), op.startswith("ds_")
        self.vector_memory, self.vector_alu, self.lanes = bool(vector), False, False
        if op == "s_waitcnt":
            n = [re.search(r"\b%s\((\d+)\)" % c, rest) for c in ("vmcnt", "lgkmcnt")]
            self.wait = [int(m.group(1)) if m else 1 << 30 for m in n]
            return
        if op == "s_nop":
            self.slots = int(rest, 0) + 1
            return
        to_lds = "_lds_" in op or re.search(r"\blds\b", rest)
        if vector:
            self.counter = "vm"
            self.load = "vm" if "_load" in op and not to_lds else None
        elif lds:
            self.counter = "lds"
            self.load = "lds" if re.match(r"ds_(read|bpermute|permute|swizzle)", op) else None
        elif re.match(r"s_(buffer_)?load", op):
            self.load = "scalar"
        out = []
        if not (NO_RESULT.match(op) or (self.counter and not self.load)):
            out = registers(operands[0]) + (registers(operands[1]) if CARRY_OUT.match(op) else [])
        into = registers(",".join(operands[1:] if out else operands))
        if "permlane" in op and "swap" in op:
            out = into = registers(rest)
        if op.startswith("v_writelane"):
            into = into + out
        if op.startswith("v_mfma"):
            self.passes = {"v_mfma_f32_16x16x32_bf16": 4, "v_mfma_f32_32x32x16_bf16": 8, "v_mfma_f32_32x32x2_f32": 16}[op]
            self.factors = registers(operands[1]) + registers(operands[2])
        self.out, self.into = out, into
        self.vector_alu = op.startswith("v_") and not self.passes
        self.lanes = "permlane" in op or re.search(r"quad_perm|row_|wave_", rest)


def findings(listing):
    """[(index, instruction, register, what)] of one kernel: lines "label:" and instructions."""
    labels, code = {}, []
    for line in listing:
        if line.endswith(":"):
            labels[line[:-1]] = len(code)
        else:
            code.append(Instruction(line))
    found = {}

    def step(state, i):
        x, (loads, products, recent) = code[i], state
        if x.wait:
            vm, lgkm = x.wait
            loads = {r: (k, n) for r, (k, n) in loads.items()
                     if not (n >= (vm if k == "vm" else lgkm) if k != "scalar" else lgkm == 0)}
        else:
            for r in x.into if loads else ():
                if r in loads:
                    found[i, r] = "read while a load into it is under way"
            for r in x.out if loads else ():
                if r in loads and not (loads[r][0] == x.load != "scalar"):      # (loads of one kind arrive in order)
                    found[i, r] = "written while a load into it is under way"
            if products and x.passes:
                for r in x.factors:
                    if r in products:
                        found[i, r] = "factor of a product too early"
            elif products and (x.counter or x.vector_alu):
                for r in x.into:
                    if r in products:
                        found[i, r] = "result of a product read %d slots early" % (products[r][2] - products[r][0])
                for r in x.out if x.vector_alu else ():
                    if r in products and products[r][2] - products[r][0] > 1:
                        found[i, r] = "result of a product overwritten %d slots early" % (products[r][2] - products[r][0] - 1)
            for r in x.into if recent else ():
                if r in recent and recent[r] < (5 if r[0] == "s" and x.vector_memory else 2 if r[0] == "v" and x.lanes else 0):
                    found[i, r] = "read by %s too early" % ("an address" if r[0] == "s" else "another lane")
            if x.counter:
                loads = {r: (k, n + (n < 64) if k == x.counter else n) for r, (k, n) in loads.items()}
            if x.load:
                loads = {**loads, **{r: (x.load, 0) for r in x.out}}
        aged = {r: (max(e + 1, p) if x.passes else e + x.slots, p, n) for r, (e, p, n) in products.items()}
        products = {r: v for r, v in aged.items() if v[0] < v[2]}
        recent = {r: e + x.slots for r, e in recent.items()
                   if e + x.slots < (5 if r[0] == "s" else 2) and not (x.op.startswith("s_") and r in x.out)}
        if x.passes:
            products.update({r: (0, x.passes, {4: 8, 8: 12, 16: 18}[x.passes]) for r in x.out})
        elif x.vector_alu:
            recent.update({r: 0 for r in x.out})
        return loads, products, recent

    def join(old, new):
        """`old` with what is nearer in `new`, or None if that adds nothing."""
        merged, changed = [dict(o) for o in old], False
        for m, n, nearer in zip(merged, new, (lambda a, b: a[1] < b[1], lambda a, b: a[2] - a[0] > b[2] - b[0], lambda a, b: a < b)):
            for r, v in n.items():
                if r not in m or nearer(v, m[r]):
                    m[r], changed = v, True
        return merged if changed else None

    states, work = {0: ({}, {}, {})}, [0]
    while work:
        i = work.pop()
        after, x = step(states[i], i), code[i]
        assert not re.match(r"s_(swappc|setpc|call|cbranch_[gijr])", x.op), x.text
        targets = [labels[x.text.split()[1]]] if re.match(r"s_c?branch", x.op) else []
        if x.op not in ("s_branch", "s_endpgm") and i + 1 < len(code):
            targets.append(i + 1)
        for j in targets:
            state = join(states[j], after) if j in states else after
            if state is not None:
                states[j] = state
                work.append(j)
    return [(i, code[i].text, "%s%d" % r, what) for (i, r), what in sorted(found.items())]


def with_far_jumps(lines):
    """A listing of (address or None, label or instruction) with s_getpc / s_add / s_addc / s_setpc made a branch to a label."""
    targets, out = {}, []
    for n, (_, text) in enumerate(lines):
        if text.startswith("s_setpc"):
            (_, pc), (base, low), (_, high) = lines[n - 3:n]
            assert pc.startswith("s_getpc") and low.startswith("s_add_u32") and high.startswith("s_addc_u32")
            low, high = (int(t.split(",")[2], 0) for t in (low, high))
            targets[n] = (base + low + (high << 32)) % (1 << 64)
    for n, (address, text) in enumerate(lines):
        if address in targets.values():
            out.append("at%d:" % address)
        out.append("s_branch at%d" % targets[n] if n in targets else text)
    return out


def kernels_of(path):
    """(name, listing) of every kernel of a gfx950 code object."""
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", "--symbolize-operands", path],
                          capture_output=True, text=True, check=True).stdout
    name, lines = None, []
    for line in text.splitlines():
        head = re.match(r"<(.*)>:$", line)
        if head and not re.match(r"L\d+$", head.group(1)):
            if name:
                yield name, with_far_jumps(lines)
            name, lines = head.group(1), []
        elif head:
            lines.append((None, head.group(1) + ":"))
        elif name and "//" in line:
            instruction, _, address = line.partition("//")
            lines.append((int(address.split(":")[0], 16), instruction.strip()))
    if name:
        yield name, with_far_jumps(lines)


def check_object(path):
    kernels = list(kernels_of(path))
    return len(kernels), [(name, f[:3]) for name, f in ((n, findings(c)) for n, c in kernels) if f]


def code_objects(folder):
    """The gfx950 code objects inside the library, one file each."""
    with open(LIB, "rb") as f:
        data = f.read()
    magic, at, paths = b"__CLANG_OFFLOAD_BUNDLE__", 0, []
    while (at := data.find(magic, at)) >= 0:
        pos, (count,) = at + 32, struct.unpack_from("<Q", data, at + 24)
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + length]:
                paths.append(os.path.join(folder, "%d.co" % len(paths)))
                with open(paths[-1], "wb") as out:
                    out.write(data[at + offset:at + offset + size])
            pos += 24 + length
        at += len(magic)
    return paths


@pytest.mark.skipif(not (os.path.exists(LIB) and shutil.which(OBJDUMP)), reason="needs the built library and ROCm's objdump")
def test_built_kernels_wait_for_what_they_use(tmp_path):
    paths = code_objects(str(tmp_path))
    with concurrent.futures.ProcessPoolExecutor(4) as pool:
        results = list(pool.map(check_object, paths))
    assert sum(n for n, _ in results) > 300
    bad = [b for _, found in results for b in found]
    assert not bad, "%d kernels, among them %s" % (len(bad), bad[:4])


def test_the_check_finds_what_is_missing():
    good = ["ds_read_b128 v[4:7], v0", "s_cbranch_scc0 L0", "s_nop 2", "L0:", "s_waitcnt lgkmcnt(0)",
            "v_mfma_f32_32x32x16_bf16 v[16:31], v[4:7], v[8:11], v[16:31]", "s_cbranch_vccz L1", "s_nop 9", "L1:", "s_nop 10",
            "v_mov_b32_e32 v2, v31", "global_load_dword v3, v[0:1], off", "global_load_dword v12, v[0:1], off", "s_waitcnt vmcnt(1)",
            "v_add_f32_e32 v3, v3, v3", "v_readfirstlane_b32 s4, v3", "s_nop 4", "global_load_dword v13, v2, s[4:5]",
            "v_add_f32_e32 v14, v3, v3", "s_nop 1", "v_permlane32_swap_b32_e32 v14, v15", "s_nop 1",
            "v_add_f32_dpp v15, v14, v14 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf", "s_endpgm"]
    assert findings(good) == []
    for i, worse in ((4, None), (9, "s_nop 9"), (13, "s_waitcnt vmcnt(2)"), (13, None), (16, "s_nop 3"), (19, "s_nop 0"), (21, "s_nop 0")):
        assert findings(good[:i] + ([worse] if worse else []) + good[i + 1:]), (good[i], worse)
    # the shorter product: 8 slots, and one behind another leaves after 4 passes, not after 8
    short = "v_mfma_f32_16x16x32_bf16 v[%d:%d], v[4:7], v[8:11], 0"
    for slots, lines in ((8, [short % (16, 19)]), (4, [short % (16, 19), short % (20, 23)]), (8, ["v_mfma_f32_32x32x16_bf16 v[32:47], v[4:7], v[8:11], 0", short % (16, 19)])):
        for missing in (0, 1):
            assert bool(findings(lines + ["s_nop %d" % (slots - 1 - missing), "v_mov_b32_e32 v2, v16", "s_endpgm"])) == bool(missing), (slots, lines, missing)
    # a copy of what is still on its way, in front of the wait
    assert findings(good[:4] + ["v_mov_b64_e32 v[20:21], v[4:5]"] + good[4:])
