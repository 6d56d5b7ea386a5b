"""Four wavefronts of lutgemm_mx_kernel run the generated fill loop (tf-approximate_amd/csrc/gen_lookup_mx.py) side by side
under random schedules: scalar registers, the LDS counters and the loads of the rows are followed instruction by
instruction, from tile to tile as lutgemm_mx_kernel.hip sets a tile up.  Checked:
  * every load of rows stays inside them by its scalar offset alone (the part a descriptor's bounds check may leave out),
    or lies behind the descriptor's end by its vector offset, and then moves nothing."""
import importlib.util
import os
import random
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("gen_lookup_mx", os.path.join(ROOT, "tf-approximate_amd", "csrc", "gen_lookup_mx.py"))
gen = importlib.util.module_from_spec(spec)
spec.loader.exec_module(gen)

WAVES, FILL_BYTES, CB = 4, 65536, 2 * 65536
SHARE = FILL_BYTES // WAVES
M32 = 0xffffffff


class Violation(AssertionError):
    pass


def decode(line, at):
    """An instruction as a function of the wavefront, or None for one that the model does not follow (vector arithmetic,
    matrix instructions)."""
    op, _, rest = line.partition(" ")
    a = [x.strip() for x in rest.split(",")] if rest else []
    name = [x[2:-1] if x.startswith("%[") else x for x in a]

    def value(x):
        if re.fullmatch(r"-?(0x[0-9a-f]+|\d+)", x):
            n = int(x, 0)
            return lambda r: n
        return lambda r: r[x]
    if op == "s_waitcnt":
        counts = [(q == "vmcnt", int(n)) for q, n in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", rest)]
        return lambda w: [w.land(w.vm if vm else w.lds, n) for vm, n in counts]
    if op == "ds_read_b32":
        reg, counter = name[1].split()[0], 8 if "offset:8" in line else 0
        return lambda w: w.look(name[0], w.r[reg] + counter)
    if op == "ds_add_u32":
        return lambda w: w.count(w.r[name[0]], w.r[name[1]])
    if op == "ds_read_b128":
        return lambda w: w.lds.append(None)
    if op.startswith("buffer_load") and line.endswith(" lds"):
        offset, reg = int(re.search(r"offset:(\d+)", line).group(1)), name[2].split()[0].rstrip("]").replace("%[", "")
        return lambda w: w.load_rows(w.r[name[0]], w.r[reg], offset)
    if op.startswith("buffer_load"):
        return lambda w: w.vm.append(None)
    if op in ("s_mov_b64", "s_mov_b32", "v_readfirstlane_b32") or (op == "v_mov_b32" and name[0] in LOOKS):
        get = value(name[1])
        return lambda w: w.put(name[0], get(w.r))
    if op in ARITHMETIC:
        x, y, f = value(name[1]), value(name[2]), ARITHMETIC[op]
        return lambda w: w.put(name[0], f(x(w.r), y(w.r)))
    if op in COMPARE:
        x, y, f = value(name[0]), value(name[1]), COMPARE[op]
        return lambda w: w.put("scc", int(f(x(w.r), y(w.r))))
    if op == "s_cselect_b32":
        x, y = value(name[1]), value(name[2])
        return lambda w: w.put(name[0], x(w.r) if w.r["scc"] else y(w.r))
    if op == "s_branch":
        return lambda w: w.jump(at[a[0]])
    if op in ("s_cbranch_scc0", "s_cbranch_scc1"):
        taken = int(op[-1])
        return lambda w: w.jump(at[a[0]]) if w.r["scc"] == taken else None
    assert op in ("s_nop", "s_sleep") or op[0] == "v", line
    return None


LOOKS = ["v%d" % r for r in (gen.V_POLL, gen.V_TMP, gen.V_CB)]
ARITHMETIC = {"s_add_u32": lambda x, y: x + y, "s_sub_u32": lambda x, y: x - y, "s_lshr_b32": lambda x, y: x >> y,
              "s_lshl_b32": lambda x, y: x << y, "s_xor_b32": lambda x, y: x ^ y, "s_and_b32": lambda x, y: x & y,
              "v_or_b32": lambda x, y: x | y}
COMPARE = {"s_cmp_eq_u32": lambda x, y: x == y, "s_cmp_lg_u32": lambda x, y: x != y, "s_cmp_ge_u32": lambda x, y: x >= y}


def program(units, vec):
    """The instructions that the model follows, jump targets counted in them."""
    lines = re.findall(r'"([^"]*)\\n\\t"', gen.emit(units, vec))
    at, code = {}, []
    for line in lines:
        if line.endswith(":"):
            at[line[:-1]] = len(code)
        else:
            step = decode(line, at)
            if step:
                code.append(step)
    return code


class Wave:
    def __init__(self, group, index):
        self.group, self.index = group, index
        self.r = {}                          # registers and operands by name
        self.vm, self.lds = [], []           # what is in flight, in order: None, or what happens as it lands
        self.gf = self.tile = self.pc = 0
        self.done = False

    def begin_tile(self):
        """What lutgemm_mx_kernel.hip hands to the loop."""
        g, wofs = self.group, self.index * SHARE
        first, count = g.tiles[self.tile]
        if self.tile + 1 < len(g.tiles):
            enext = g.tiles[self.tile + 1][0] * FILL_BYTES + wofs
        else:
            enext = 0x80000000
        other = (self.gf & 1) ^ 1
        after = (first + 1) * FILL_BYTES + wofs if count > 1 else enext
        self.r = {"gf": self.gf, "cbcur": CB + 4 * (self.gf & 1), "cboth": CB + 4 * other,
                  "edst": wofs + other * FILL_BYTES, "left": count, "enext": enext,
                  "free": 0 if self.gf == 0 else 4 * (2 * ((self.gf - 1) >> 1) + 2),
                  "whole": 4 * (2 * ((self.gf + 1) >> 1) + 1) if count > 1 else 0,
                  "whole0": 4 * (2 * (self.gf >> 1) + 1), "eoff": after & 0x7fffffff, "cb0": CB, "spin": g.spin,
                  "v%d" % gen.V_L16: after & 0x80000000, "exec": -1}
        self.pc = 0

    def put(self, name, value):
        self.r[name] = value & M32

    def jump(self, pc):
        self.pc = pc

    def land(self, queue, left):
        while len(queue) > left:
            arrive = queue.pop(0)
            if arrive:
                arrive()

    def look(self, reg, address):
        value = self.group.counter[(address - CB) // 4]
        self.lds.append(lambda: self.put(reg, value))

    def count(self, address, value):
        assert self.r["exec"] == 1
        self.group.counter[(address - CB) // 4] += value
        self.lds.append(None)

    def step(self):
        instruction = self.group.code[self.pc]
        self.pc += 1
        instruction(self)
        if self.pc >= len(self.group.code):
            self.end_tile()

    def load_rows(self, voff, soff, offset):
        g = self.group
        if soff + 1024 + offset > g.rows_bytes:
            raise Violation("the scalar offset %#x leaves the rows" % soff)
        fill = self.r["gf"] + 1                              # of the workgroup: the one these rows are for
        if voff >= g.rows_bytes:                             # behind the descriptor's end: nothing moves
            if fill < g.total_fills:
                raise Violation("fill %d is not loaded" % fill)
            self.vm.append(None)
            return
        if fill >= g.total_fills:
            raise Violation("rows behind the last fill are loaded")
        if (soff + offset) // FILL_BYTES != g.row_fill[fill] or (soff + offset) % FILL_BYTES // SHARE != self.index:
            raise Violation("fill %d gets rows from %#x" % (fill, soff + offset))
        self.vm.append(None)

    def end_tile(self):
        assert not self.vm and not self.lds and self.r["fail"] == 0, self.r["fail"]
        self.gf = self.r["gf"]
        self.tile += 1
        if self.tile == len(self.group.tiles):
            self.done = True
        else:
            self.begin_tile()


class Workgroup:
    def __init__(self, code, tiles, rows_fills, spin=1 << 20):
        """tiles: (first fill of its rows, number of fills)"""
        self.code, self.tiles, self.spin = code, tiles, spin
        self.rows_bytes = rows_fills * FILL_BYTES
        self.row_fill = [first + k for first, count in tiles for k in range(count)]
        self.total_fills = len(self.row_fill)
        self.counter = [WAVES, 0, 0]          # the very first fill has arrived
        self.waves = [Wave(self, i) for i in range(WAVES)]
        for w in self.waves:
            w.begin_tile()

    def run(self, rng, limit):
        steps = 0
        while True:
            left = [w for w in self.waves if not w.done]
            if not left:
                return
            w = rng.choice(left)
            for _ in range(rng.choice((1, 7, 60, 400))):
                if w.done:
                    break
                w.step()
                steps += 1
            assert steps < limit, "the wavefronts do not finish"


TILES = {"one tile of one fill": [(2, 1)], "tiles of one fill": [(0, 1), (1, 1), (0, 1)],
         "two tiles": [(1, 3), (0, 2)]}


@pytest.mark.parametrize("tiles", TILES.values(), ids=TILES.keys())
@pytest.mark.parametrize("variant", [v for v in gen.VARIANTS if v[0] in (2, 3, 6, 13, 25)], ids=str)
def test_four_wavefronts(variant, tiles):
    code = program(*variant)
    group = Workgroup(code, tiles, 1 + max(first + count for first, count in tiles))
    group.run(random.Random(str(variant)), 400 * len(code))
    assert group.counter[0] + group.counter[1] >= WAVES * 2 * group.total_fills
