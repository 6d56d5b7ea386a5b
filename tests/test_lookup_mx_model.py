"""The generated fill loop of lutgemm_mx_kernel (tf-approximate_amd/csrc/gen_lookup_mx.py) waits for LDS and memory
operations with derived counts.  This test runs the emitted text, three fills long, through a model of the hardware's
two in-order queues and follows the data of one wavefront: no instruction may touch a register that an operation in
flight has yet to write, at most 15 LDS operations may be outstanding, every sum must start from its start value and
receive exactly the 16 looked-up quadruples of its pixels per fill, made from the activations of its own unit and fill,
and every fill's rows must be loaded exactly once while the fill before is looked up.  Which buffer they go to and how
the wavefronts wait for each other is test_lookup_mx_workgroup.py's."""
import importlib.util
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("gen_lookup_mx", os.path.join(ROOT, "tf-approximate_amd", "csrc", "gen_lookup_mx.py"))
gen = importlib.util.module_from_spec(spec)
spec.loader.exec_module(gen)

FILLS = 3


def regs(tok):
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", tok)
    if m:
        return ["%s%d" % (m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)]
    return [tok] if re.fullmatch(r"[va]\d+", tok) else []


class Machine:
    def __init__(self):
        self.lds, self.vm, self.val, self.busy = [], [], {}, {}

    def touch(self, names, what):
        for r in names:
            assert r not in self.busy, "%s uses %s, still in flight" % (what, r)

    def land(self, queue, left):
        while len(queue) > left:
            for r, v in queue.pop(0):
                self.val[r] = v
                del self.busy[r]

    def start(self, queue, writes):
        for r, _ in writes:
            assert r not in self.busy
            self.busy[r] = True
        queue.append(writes)


@pytest.mark.parametrize("variant", gen.VARIANTS, ids=str)
def test_fill_loop(variant):
    text = gen.emit(*variant)
    units = variant[0]
    lines = [x for x in re.findall(r'"([^"]*)\\n\\t"', text)]
    m = Machine()
    m.val["v%d" % gen.V_POLL] = "cinit"    # what the caller hands over in this register
    starts = {}
    vector_sums = {r for u in range(units) for j in range(4) for r in regs(gen.acc_reg(units, u, j)) if r[0] == "v"}
    base_of = {"v%d" % (gen.V_BASE + u): u for u in range(units)}
    loop, end = lines.index("Lfill_%=:"), lines.index("Lend_%=:")
    pc, fill, sums, loads, flips, steps, last_loads = 0, 0, {}, [], 0, 0, 0
    prologue = True
    while True:
        line = lines[pc]
        pc += 1
        if line.startswith("Lfill"):
            prologue = False
        if line.endswith(":"):
            continue
        op, _, rest = line.partition(" ")
        args = [a.strip() for a in rest.split(",")]
        first = args[-1].split()[0] if args[-1] else ""
        args[-1] = first
        if op == "s_waitcnt":
            for name, n in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", rest):
                m.land(m.vm if name == "vmcnt" else m.lds, int(n))
        elif op == "ds_read_b128":
            dst = regs(args[0])
            m.touch(dst + regs(args[1]), line)
            m.start(m.lds, [(r, ("look",) + m.val[args[1]]) for r in dst])
        elif op in ("ds_read_b32", "ds_add_u32"):
            m.touch(regs(args[0]) + regs(args[1]), line)
            m.start(m.lds, [(args[0], ("event",))] if op == "ds_read_b32" else [])
        elif op == "v_perm_b32":
            m.touch([r for a in args for r in regs(a)], line)
            act = m.val[args[1]]
            assert act[0] == "act", line
            step = int(args[3][1:]) - gen.V_SEL
            assert (args[2] == "v%d" % gen.V_CH0) == (step < 3)
            m.val[args[0]] = (act[1], act[2], act[3], step, flips)
        elif op.startswith("v_smfmac"):
            acc, data = regs(args[0]), regs(args[2])
            m.touch(acc + data, line)
            assert len(data) == 8 and args[1] == "v[%d:%d]" % (gen.V_A, gen.V_A + 3) and args[3] == "v%d" % gen.V_IDX
            for half in (data[:4], data[4:]):
                seen = {m.val[r] for r in half}
                assert len(seen) == 1
                sums.setdefault(tuple(acc), []).append(seen.pop())
        elif op.startswith("buffer_load") and rest.endswith("lds"):
            offset = int(re.search(r"offset:(\d+)", rest).group(1))
            loads.append((flips, m.val["m0"] + offset))
            m.start(m.vm, [])
        elif op.startswith("buffer_load"):
            dst = regs(args[0])
            m.touch(dst + regs(args[1]), line)
            kind, unit, at_fill = m.val[args[1]]
            assert kind == "addr"
            pixel = 0 if args[3].startswith("0") else int(re.search(r"p(\d)", args[3]).group(1))
            m.start(m.vm, [(r, ("act", at_fill, unit, pixel + i)) for i, r in enumerate(dst)])
        elif op == "v_add_u32" and args[1] in base_of:
            m.touch(regs(args[0]), line)
            m.val[args[0]] = ("addr", base_of[args[1]], steps)
        elif op == "v_add_u32" and args[0] == "v%d" % gen.V_KOFF and args[1] == "%[doff]":
            steps += 1
        elif op == "v_xor_b32" and args[0] == "v%d" % gen.V_CH0:
            flips += 1
        elif op == "s_add_u32" and args[0] == "m0":
            m.val["m0"] = int(args[2])
        elif op == "s_branch" and args[0].startswith("Lslow"):
            pc = lines.index(args[0].replace("slow", "ok") + ":") if args[0].replace("slow", "ok") + ":" in lines else None
            if pc is None:   # the labels are numbered in pairs: ok n, slow n + 1
                n = int(re.search(r"\d+", args[0]).group())
                pc = lines.index("Lok%d_%%=:" % (n - 1))
        elif op == "s_cbranch_scc1" and args[0].startswith("Lend"):
            fill += 1
            if fill == FILLS:
                break
        elif op == "s_branch" and args[0].startswith("Lfill"):
            pc = loop
        elif (op == "v_accvgpr_write_b32" or (op == "v_mov_b32" and regs(args[0])[0] in vector_sums)) and prologue:
            m.touch([r for a in args for r in regs(a)], line)
            assert args[0] not in starts
            starts[args[0]] = m.val.get(args[1], args[1])
        else:
            m.touch([r for a in args for r in regs(a)], line)
            assert not set(regs(args[0])) & set(starts), line
            if regs(args[0]):
                m.val[regs(args[0])[0]] = None
        assert len(m.lds) <= 15 and len(m.vm) <= 63
    assert end > loop and steps == FILLS
    # every sum: per fill 16 quadruples of its own unit and pixel, each step once, out of the fill's own buffer
    # and started from the correction (low bytes) or zero (high bytes)
    assert len(sums) == 4 * units and len(starts) == 16 * units
    for u in range(units):
        for j in range(4):
            assert [starts[r] for r in regs(gen.acc_reg(units, u, j))] == ["cinit", "0"] * 2
            got = sums[tuple(regs(gen.acc_reg(units, u, j)))]
            assert sorted(got) == sorted(("look", f, u, j, c, f) for f in range(FILLS) for c in range(4)), (u, j)
    # the rows: 16 pieces of 1 KiB per fill, while the wavefront reads the other buffer (before the flip to it)
    for f in range(FILLS):
        assert sorted(at for flip, at in loads if flip == f) == [1024 * i for i in range(gen.LOADS)], f
