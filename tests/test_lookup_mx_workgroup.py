"""Four wavefronts of lutgemm_mx_kernel run the generated fill loop (tf-approximate_amd/csrc/gen_lookup_mx.py) side by side
under random schedules: scalar registers, the LDS counters, the loads of the rows and the lookups are followed instruction
by instruction, from tile to tile as lutgemm_mx_kernel.hip sets a tile up.  Operations in flight happen at any moment from
their issue to the wait that needs them, in order within a queue.  Checked:
  * every load of rows stays inside them by its scalar offset alone (the part a descriptor's bounds check may leave out),
    or lies behind the descriptor's end by its vector offset, and then moves nothing;
  * every fill's rows are loaded once, every wavefront its own share, into the fill's own buffer;
  * every lookup of a fill finds the whole fill in the buffer it reads: all rows landed, none being overwritten;
  * a fill's arrival is counted after its loads have landed, and a wavefront's reading of it after its last lookup.
The last test takes these parts out of the emitted text, one at a time, and expects the model to object."""
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


def check(ok, what):
    if not ok:
        raise Violation(what)


def decode(line, at):
    """An instruction as a function of the wavefront, or None for one that the model does not follow (other vector
    arithmetic, matrix instructions)."""
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
    if op == "v_perm_b32":
        return lambda w: w.put(name[0], w.r[name[2]] >> 24)             # of an address the buffer
    if op == "ds_read_b128":
        return lambda w: w.lookup(w.r[name[1]])
    if op.startswith("buffer_load") and line.endswith(" lds"):
        offset, reg = int(re.search(r"offset:(\d+)", line).group(1)), name[2].split()[0].rstrip("]").replace("%[", "")
        return lambda w: w.load_rows(w.r[name[0]], w.r[reg], offset)
    if op.startswith("buffer_load"):
        return lambda w: w.vm.append(None)
    if op in ("s_mov_b64", "s_mov_b32", "v_readfirstlane_b32") or (op == "v_mov_b32" and name[0] in LOOKS):
        get = value(name[1])
        return lambda w: w.put(name[0], get(w.r))
    if op in ARITHMETIC and (op != "v_xor_b32" or name[0] in CHUNKS):
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
              "v_or_b32": lambda x, y: x | y, "v_xor_b32": lambda x, y: x ^ y}
CHUNKS = ["v%d" % r for r in (gen.V_CH0, gen.V_CH1)]
COMPARE = {"s_cmp_eq_u32": lambda x, y: x == y, "s_cmp_lg_u32": lambda x, y: x != y, "s_cmp_ge_u32": lambda x, y: x >= y}


def program(units, vec, mutate=None):
    """The instructions that the model follows, jump targets counted in them."""
    lines = re.findall(r'"([^"]*)\\n\\t"', gen.emit(units, vec))
    if mutate:
        lines = mutate(lines)
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
        self.done = self.arrived = False

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
        for chunk in CHUNKS:
            self.r[chunk] = (self.gf & 1) << 24
        self.pc = 0
        self.tile_gf, self.lookups, self.loads, self.events = self.gf, 0, {}, []

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
        self.lds.append(lambda: self.put(reg, self.group.counter[(address - CB) // 4]))

    def count(self, address, value):
        check(self.r["exec"] == 1, "counted by more than one lane")
        event = "arrived" if address == self.r["cboth"] else "read"
        fill = self.r["gf"] + (event == "arrived")
        check((event, fill) not in self.events, "fill %d counted twice" % fill)
        self.events.append((event, fill))
        if event == "arrived":
            pieces = self.loads.get(fill, {})
            check(len(pieces) == gen.LOADS and all(pieces.values()), "fill %d counted before its rows have landed" % fill)
        else:                                                 # a wavefront's LDS operations happen in order
            check(self.lookups >= (fill - self.tile_gf + 1) * self.group.lookups, "fill %d counted as read too early" % fill)

        def happen():
            self.group.counter[(address - CB) // 4] += value
        self.lds.append(happen)

    def lookup(self, buffer):
        fill = self.tile_gf + self.lookups // self.group.lookups
        self.lookups += 1
        if fill >= self.tile_gf + self.group.tiles[self.tile][1]:   # ahead of the tile's end: of no account
            self.lds.append(None)
            return

        def happen():
            check(buffer == fill & 1, "fill %d looked up in the other buffer" % fill)
            check(self.group.whole(buffer) == fill, "fill %d looked up while it is not there" % fill)
        self.lds.append(happen)

    def step(self, rng):
        if not self.arrived:             # the kernel's own first fill: rows, a wait for all of them, one event
            self.arrived = True
            for i in range(gen.LOADS):
                self.group.set(0, self.index * gen.LOADS + i, 0)
            self.group.counter[0] += 1
            return
        for queue in (self.vm, self.lds):                     # what is in flight may happen now
            if queue and rng.random() < self.group.eagerness:
                self.land(queue, rng.randrange(len(queue)))
        instruction = self.group.code[self.pc]
        self.pc += 1
        instruction(self)
        if self.pc >= len(self.group.code):
            self.end_tile()

    def load_rows(self, voff, soff, offset):
        g = self.group
        check(soff + 1024 + offset <= g.rows_bytes, "the scalar offset %#x leaves the rows" % soff)
        fill, dest = self.r["gf"] + 1, self.r["m0"] + offset   # of the workgroup: the one these rows are for
        pieces, piece = self.loads.setdefault(fill, {}), dest // 1024 % 64
        check(dest // FILL_BYTES == fill & 1, "fill %d goes into the buffer being read" % fill)
        check(piece // gen.LOADS == self.index and piece not in pieces, "piece %d of fill %d loaded twice" % (piece, fill))
        if voff >= g.rows_bytes:                             # behind the descriptor's end: nothing moves
            check(fill >= g.total_fills, "fill %d is not loaded" % fill)
            pieces[piece] = True
            self.vm.append(None)
            return
        check(fill < g.total_fills, "rows behind the last fill are loaded")
        check((soff + offset) // FILL_BYTES == g.row_fill[fill] and (soff + offset) % FILL_BYTES == dest % FILL_BYTES,
              "fill %d gets rows from %#x" % (fill, soff + offset))
        pieces[piece] = False
        g.set(fill & 1, piece, None)                         # from here on neither the old rows nor the new

        def land():
            pieces[piece] = True
            g.set(fill & 1, piece, fill)
        self.vm.append(land)

    def end_tile(self):
        check(self.r["fail"] == 0, "a wait has run out")
        assert not self.vm and not self.lds
        fills = range(self.tile_gf, self.r["gf"])
        check(len(fills) == self.group.tiles[self.tile][1], "%d fills" % len(fills))
        check(sorted(self.events) == sorted([("arrived", f + 1) for f in fills] + [("read", f) for f in fills]), "events")
        self.gf = self.r["gf"]
        self.tile += 1
        if self.tile == len(self.group.tiles):
            self.done = True
        else:
            self.begin_tile()


class Workgroup:
    def __init__(self, code, units, tiles, rows_fills, spin=1 << 20):
        """tiles: (first fill of its rows, number of fills)"""
        self.code, self.tiles, self.spin, self.lookups = code, tiles, spin, 16 * units
        self.rows_bytes = rows_fills * FILL_BYTES
        self.row_fill = [first + k for first, count in tiles for k in range(count)]
        self.total_fills = len(self.row_fill)
        self.counter = [0, 0, 0]
        self.pieces, self.full = [[None] * 64, [None] * 64], [None, None]
        self.waves = [Wave(self, i) for i in range(WAVES)]
        for w in self.waves:
            w.begin_tile()

    def set(self, buffer, piece, fill):
        self.pieces[buffer][piece] = fill
        self.full[buffer] = fill if fill is not None and all(f == fill for f in self.pieces[buffer]) else None

    def whole(self, buffer):
        """The fill whose rows are all in the buffer, or None."""
        return self.full[buffer]

    def run(self, rng, limit):
        self.eagerness, steps = rng.choice((0.0, 0.003, 0.1)), 0
        while True:
            left = [w for w in self.waves if not w.done]
            if not left:
                return
            w = rng.choice(left)
            for _ in range(rng.choice((1, 7, 30, 100, 300))):
                if w.done:
                    break
                w.step(rng)
                steps += 1
            check(steps < limit, "the wavefronts do not finish")


TILES = {"one tile of one fill": [(2, 1)], "tiles of one fill": [(0, 1), (1, 1), (0, 1)],
         "two tiles": [(1, 3), (0, 2)]}


def run(code, units, tiles, seed, limit=4000):
    group = Workgroup(code, units, tiles, 1 + max(first + count for first, count in tiles))
    group.run(random.Random(seed), limit * len(code))
    return group


@pytest.mark.parametrize("tiles", TILES.values(), ids=TILES.keys())
@pytest.mark.parametrize("variant", [v for v in gen.VARIANTS if v[0] in (2, 3, 6, 13, 25)], ids=str)
def test_four_wavefronts(variant, tiles):
    code = program(*variant)
    for seed in range(6):
        group = run(code, variant[0], tiles, seed)
        # of every fill four arrivals and four readers, and four "arrivals" behind the last one
        assert sum(group.counter[:2]) == WAVES * 2 * group.total_fills + WAVES


def without(pattern, first=True):
    """The lines without the first (or every) one that matches."""
    def mutate(lines):
        hits = [i for i, line in enumerate(lines) if re.search(pattern, line)]
        assert hits, pattern
        drop = set(hits[:1] if first else hits)
        return [line for i, line in enumerate(lines) if i not in drop]
    return mutate


def without_check_of(target):
    """No branch to the loop of further looks behind the comparison with this target."""
    def mutate(lines):
        at = lines.index("s_cmp_ge_u32 %%[ev], %%[%s]" % target)
        assert lines[at + 1].startswith("s_cbranch_scc0 Lslow")
        return lines[:at + 1] + lines[at + 2:]
    return mutate


def event_lines(lines, counter):
    """Where the five lines that count an event of this counter begin."""
    at = [i for i, line in enumerate(lines) if line.startswith("ds_add_u32")]
    return [i - 3 for i in at if lines[i - 3].endswith("%%[%s]" % counter)][0]


def arrival_before_its_wait(lines):
    at = event_lines(lines, "cboth")
    assert lines[at - 1].startswith("s_waitcnt vmcnt")
    return lines[:at - 1] + lines[at:]


def reader_event_early(lines):
    """Counted where the next fill's first lookups begin, with the last lookups of this one still to come."""
    at = event_lines(lines, "cbcur")
    to = event_lines(lines, "cboth")
    return lines[:to] + lines[at:at + 5] + lines[to:at] + lines[at + 5:]


def no_reader_event(lines):
    at = event_lines(lines, "cbcur")
    return lines[:at] + lines[at + 5:]


MUTATIONS = {   # and what the model has to say
    "buffer refilled without looking whether it is free": (without_check_of("free"), "looked up while it is not there"),
    "buffer read without looking whether it is whole": (without_check_of("whole"), "looked up while it is not there"),
    "rows always into the same buffer": (without(r"s_xor_b32 %\[edst\]"), "goes into the buffer being read"),
    "lookups always in the same buffer": (without(r"v_xor_b32 v(%d|%d)," % (gen.V_CH0, gen.V_CH1), first=False),
                                          "looked up in the other buffer"),
    "arrival counted before the loads have landed": (arrival_before_its_wait, "before its rows have landed"),
    "reading counted too early": (reader_event_early, "read too early"),
    "reading never counted": (no_reader_event, "do not finish"),
    "counters not exchanged": (without(r"s_xor_b32 %\[cboth\]"), "counted|do not finish"),
    "a piece of a fill never loaded": (without(r"buffer_load_dwordx4 .* lds$"), "before its rows have landed"),
    "no mark behind the last fill": (without(r"^v_or_b32"), "behind the last fill"),
}


@pytest.mark.parametrize("mutate,says", MUTATIONS.values(), ids=MUTATIONS.keys())
@pytest.mark.parametrize("variant", [(3, True), (10, False)], ids=str)
def test_the_model_objects_to_a_loop_without(variant, mutate, says):
    code = program(*variant, mutate)
    said = []
    for seed in range(300):
        try:
            run(code, variant[0], [(1, 3), (0, 2)], seed, limit=300)
        except Violation as e:
            said.append(str(e))
            if re.search(says, said[-1]):
                return
    raise AssertionError(set(said))
