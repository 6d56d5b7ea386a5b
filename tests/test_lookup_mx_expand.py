"""The expanding form of lutgemm_mx_kernel's fill loop (tf-approximate_amd/csrc/gen_lookup_mx.py, emit(..., expand=True)) run
on the CPU: four wavefronts of 64 lanes execute the emitted text side by side under random schedules, on real bytes of LDS,
filter codes, truth table and activation codes, from tile to tile as lutgemm_mx_kernel.h sets a tile up.  A load's data
land, and an LDS operation happens, at any moment between its issue and the wait that needs it, in order within a queue;
until then nobody may touch its registers.  At the end of a tile every sum must be the one the truth table gives.
The last test takes parts out of the emitted text, one at a time, and expects a wrong sum or an objection."""
import importlib.util
import os
import random
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
spec = importlib.util.spec_from_file_location("gen_lookup_mx", os.path.join(ROOT, "tf-approximate_amd", "csrc", "gen_lookup_mx.py"))
gen = importlib.util.module_from_spec(spec)
spec.loader.exec_module(gen)

LANE = np.arange(64)
Q, I = LANE >> 4, LANE & 15
S, C = (LANE >> 1) & 15, (LANE & 1) | ((LANE >> 5) << 1)       # mx_x_element, mx_x_codes
CB, FILL = 131072, 65536
M32 = 0xffffffff


class Violation(AssertionError):
    pass


def check(ok, what):
    if not ok:
        raise Violation(what)


def regs(tok):
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", tok)
    if m:
        return ["%s%d" % (m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)]
    return [tok] if re.fullmatch(r"[va]\d+", tok) else []


def phys_row(a):
    return (a >> 2) | ((a & 3) << 6)


class Problem:
    """A layer's data: K order of quads (tap row, tap column, channel quad), one column tile per entry of `cols`."""

    def __init__(self, rng, units, vec, fills, n_col):
        self.units, self.vec, self.fills, self.n_col = units, vec, fills, n_col
        self.c4, self.kw, self.quad, self.kwstep, self.khstep = 3, 3, 4 * rng.randrange(1, 9), 64, 256
        self.pitch = 4 if vec else 8
        self.table = rng_array(rng, (257, 256), 65536).astype(np.uint16)     # [filter code][activation code]
        self.table[256] = 0
        self.flipped = self.table ^ 0x8080
        self.wq = rng_array(rng, (n_col, fills, 16, 8), 257).astype(np.uint16)
        self.base = [rng_array(rng, 16, 64) * 4 for _ in range(units * 4)]   # [wavefront * units + u][i]
        kh = fills * 4 // (self.c4 * self.kw) + 2
        self.xq = rng_array(rng, 256 + 64 + kh * self.khstep + self.kw * 64 + 3 * 40, 256).astype(np.uint8)

    def koff(self, quad):
        tap, q = quad // self.c4, quad % self.c4
        return tap // self.kw * self.khstep + tap % self.kw * self.kwstep + q * self.quad

    def sums(self, wave, u, ct, f0, count):
        """[pixel 4 i + j][column]: (sum of low bytes, of high bytes), both of the flipped, signed bytes, plus the start."""
        lo, hi = np.zeros((16, 4, 8), np.int64), np.zeros((16, 4, 8), np.int64)
        back = np.zeros(256, np.int64)
        back[phys_row(np.arange(256))] = np.arange(256)
        for f in range(f0, f0 + count):
            for e in range(16):
                at = self.base[wave * self.units + u][:, None] + self.koff(4 * f + e // 4) + np.arange(4)[None] * self.pitch + e % 4
                t = self.table[self.wq[ct, f, e]][:, back[self.xq[at]]].transpose(1, 2, 0).astype(np.int64)   # [i][j][column]
                lo += t & 255
                hi += t >> 8
        return lo - 128 * 16 * count, hi - 128 * 16 * count


def rng_array(rng, shape, below):
    return np.random.RandomState(rng.randrange(1 << 30)).randint(0, below, shape)


class Wave:
    def __init__(self, group, index):
        self.g, self.index = group, index
        self.v, self.s, self.busy = {}, {}, {}
        self.vm, self.lds = [], []
        self.gf = self.tile = 0
        self.done = False
        p = group.p
        first = group.first(0)
        self.toff = (64 * index + 8 * C) * 2
        self.ldst = (16 * index + 2 * C) * 256 + 16 * S
        for b in range(2):                       # the kernel's own first fill
            for e in range(8):
                codes = p.wq.reshape(-1, 16, 8)[first][S]                         # [lane][column]
                chunk = p.flipped[codes, (64 * index + 8 * C + 32 * b + e)[:, None]]
                group.store(self.ldst + (e >> 2) * 256 + (e & 3) * 16384 + b * 2048, chunk.view(np.uint32).reshape(64, 4))
        wq = p.wq.reshape(-1, 16, 8)
        self.codes = wq[first + 2][S].copy().view(np.uint32).reshape(64, 4)
        self.entries = np.zeros((64, 16, 4), np.uint32)
        for i in range(16):                      # the second fill's entries: [lane][8 block + column]
            at = 64 * index + 8 * C + 32 * (i // 8)
            self.entries[:, i] = p.flipped[wq[first + 1][S, i % 8][:, None], at[:, None] + np.arange(8)].view(np.uint32)
        group.counter[0] += 1
        self.begin()

    def begin(self):
        g, p, gf = self.g, self.g.p, self.gf
        ct, f0, count = g.tiles[self.tile]
        first = g.first(self.tile)
        more = self.tile + 1 < len(g.tiles)
        enext = g.first(self.tile + 1) * 256 if more else 0x80000000
        after = (first + 3) * 256 if count > 3 else enext
        other = (gf & 1) ^ 1
        plane = (I >> 2) ^ np.array([0, 3, 1, 2])[Q]
        ilo = I & 3
        quad = f0 * 4 + plane
        tap, ql = quad // p.c4, quad % p.c4
        v = self.v = {}
        one = lambda value: np.broadcast_to(np.asarray(value, np.uint32), (64,)).copy()
        sel = [0x0c030000 | ((4 + (ilo ^ c)) << 8) | (c if c < 3 else 0) for c in range(4)]
        chunk = [(plane * 4 + (ilo ^ c)) << 4 for c in range(4)]
        buf = (gf & 1) << 24
        v[gen.V_CH0] = one(chunk[0] | chunk[1] << 8 | chunk[2] << 16 | buf)
        v[gen.V_CH1] = one(chunk[3] | buf)
        for c in range(4):
            v[gen.V_SEL + c] = one(sel[c])
        v[gen.V_Q], v[gen.V_KW] = one(ql), one(tap % p.kw)
        v[gen.V_KOFF] = one(p.koff(quad))
        v[gen.V_POLL] = one(0)                   # the sums' start: left out
        v[gen.V_L16] = one(S * 16 | (after & 0x80000000))
        for u in range(p.units):
            v[gen.V_BASE + u] = one(p.base[self.index * p.units + u][I])
        codes, _, land, _, toff, ldst = gen.expand_layout(p.units)
        for k in range(4):
            v[codes + k] = one(self.codes[:, k])
        for i in range(64):
            v[land + i] = one(self.entries[:, i // 4, i % 4])
        v[toff], v[ldst] = one(self.toff), one(self.ldst + other * FILL)
        self.v = {"v%d" % r: x for r, x in v.items()}
        whole = lambda f: 4 * (2 * (f >> 1) + 1)
        self.s = {"gf": gf, "cbcur": CB + 4 * (gf & 1), "cboth": CB + 4 * other, "left": count, "enext": enext,
                  "free": 0 if gf == 0 else 4 * (2 * ((gf - 1) >> 1) + 2), "whole": whole(gf + 1) if count > 1 else 0,
                  "whole0": whole(gf), "eoff": after & 0x7fffffff, "cb0": CB, "spin": g.spin, "rowb": 512,
                  "lo": 0x05040100, "hi": 0x07060302, "c4": p.c4, "kwn": p.kw, "p1": p.pitch, "p2": 2 * p.pitch, "p3": 3 * p.pitch}
        taps = 4 // p.c4
        dq, dkw = 4 % p.c4, taps % p.kw
        self.s.update({"dq": dq, "dkw": dkw, "doff": dq * p.quad + dkw * p.kwstep + taps // p.kw * p.khstep,
                       "qoff": (p.kwstep - p.c4 * p.quad) & M32, "kwoff": (p.khstep - p.kw * p.kwstep) & M32})
        self.exec = np.ones(64, bool)
        self.pc = 0

    # operands
    def get(self, tok):
        if tok in self.v:
            return self.v[tok]
        if tok.startswith("%["):
            return self.s[tok[2:-1]]
        return int(tok, 0) & M32

    def put(self, tok, value):
        if tok.startswith("%["):
            self.s[tok[2:-1]] = int(value) & M32
            return
        old = self.v.get(tok, np.zeros(64, np.uint32))
        self.v[tok] = np.where(self.exec, np.asarray(value).astype(np.uint64) & M32, old).astype(np.uint32)

    def land(self, queue, left):
        while len(queue) > left:
            names, act = queue.pop(0)
            for r in names:
                del self.busy[r]
            act()

    def issue(self, queue, names, act):
        for r in names:
            check(r not in self.busy, "%s loaded twice" % r)
            self.busy[r] = True
        queue.append((names, act))
        check(len(self.lds) <= 15 and len(self.vm) <= 63, "more in flight than the counters hold")

    def step(self, rng):
        for queue in (self.vm, self.lds):
            if queue and rng.random() < self.g.eager:
                self.land(queue, rng.randrange(len(queue)))
        line = self.g.lines[self.pc]
        self.pc += 1
        if not line.endswith(":"):
            self.run(line)
        if self.pc >= len(self.g.lines):
            self.end_tile()

    def run(self, line):
        op, _, rest = line.partition(" ")
        a = [x.strip() for x in rest.split(",")] if rest else []
        words = [x.split()[0] if x else x for x in a]
        if op != "s_waitcnt":
            for x in words:
                for r in regs(x):
                    check(r not in self.busy, "%s uses %s, still in flight" % (line, r))
        mem, g = self.g, self.g
        offset = int(re.search(r"offset:(\d+)", rest).group(1)) if "offset:" in rest else 0
        if op == "s_waitcnt":
            for name, n in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", rest):
                self.land(self.vm if name == "vmcnt" else self.lds, int(n))
        elif op == "ds_read_b128":
            names, addr = regs(words[0]), self.get(words[1]).astype(np.int64)

            def act():
                for k, r in enumerate(names):
                    self.v[r] = mem.lds32[addr // 4 + k].copy()
            self.issue(self.lds, names, act)
        elif op == "ds_write_b128":
            addr = self.get(words[0]).astype(np.int64) + offset
            data = np.stack([self.v[r] for r in regs(words[1])], 1)
            self.issue(self.lds, [], lambda: mem.store(addr, data))
        elif op == "ds_read_b32":
            r, at = words[0], (int(self.get(words[1])[0]) - CB + offset) // 4
            self.issue(self.lds, [r], lambda: self.v.__setitem__(r, np.full(64, mem.counter[at], np.uint32)))
        elif op == "ds_add_u32":
            check(int(self.exec.sum()) == 1, "counted by more than one lane")
            at, n = (int(self.get(words[0])[0]) - CB) // 4, int(self.get(words[1])[0])

            def act():
                mem.counter[at] += n
            self.issue(self.lds, [], act)
        elif op.startswith("buffer_load"):
            names, voff, p = regs(words[0]), self.get(words[1]).astype(np.int64) + offset, g.p
            soff = self.get(words[3])
            data = {"%[xq]": p.xq, "%[wrc]": p.wq.reshape(-1).view(np.uint8), "%[erc]": p.flipped.reshape(-1).view(np.uint8)}[words[2]]
            check(soff + 16 <= len(data), "the scalar offset leaves the buffer: " + line)
            ok = voff + 4 * len(names) <= len(data)
            at = np.where(ok, voff + soff, 0)
            check(bool((at + 4 * len(names) <= len(data)).all()), "beyond the buffer: " + line)

            def act():
                for k, r in enumerate(names):
                    b = data[at[:, None] + 4 * k + np.arange(4)].astype(np.uint32)
                    self.v[r] = np.where(ok, b[:, 0] | b[:, 1] << 8 | b[:, 2] << 16 | b[:, 3] << 24, 0).astype(np.uint32)
            self.issue(self.vm, names, act)
        elif op == "v_perm_b32":
            hi, lo, sel = (np.broadcast_to(np.asarray(self.get(x), np.uint64), (64,)) for x in words[1:])
            both, out = (hi << np.uint64(32)) | lo, np.zeros(64, np.uint64)
            for k in range(4):
                s = (sel >> np.uint64(8 * k)) & np.uint64(255)
                byte = np.where(s < 8, (both >> (8 * np.minimum(s, 7)).astype(np.uint64)) & np.uint64(255), 0)   # 12: zero
                check(bool(((s < 8) | (s == 12)).all()), line)
                out |= byte << np.uint64(8 * k)
            self.put(words[0], out)
        elif op == "v_mad_u32_u16":
            x = self.get(words[1])
            x = x >> 16 if "op_sel:[1,0,0,0]" in rest else x & 0xffff
            self.put(words[0], x.astype(np.uint64) * self.get(words[2]) + self.get(words[3]))
        elif op.startswith("v_smfmac"):
            data = np.stack([self.v[r] for r in regs(words[2])], 1)
            b = data.copy().view(np.int8).reshape(4, 16, 2, 16).astype(np.int64).sum((0, 2))      # [i][byte]
            for k, r in enumerate(regs(words[0])):
                self.v[r] = (self.v[r].astype(np.int64) + b[I, 4 * Q + k]).astype(np.uint64).astype(np.uint32)
        elif op == "v_accvgpr_write_b32" or op == "v_mov_b32":
            self.put(words[0], np.broadcast_to(np.asarray(self.get(words[1]), np.uint32), (64,)))
        elif op == "v_readfirstlane_b32":
            self.put(words[0], self.get(words[1])[0])
        elif op in ("v_add_u32", "v_subrev_u32", "v_xor_b32", "v_or_b32"):
            x, y = (np.asarray(self.get(t)).astype(np.int64) for t in words[1:])
            self.put(words[0], {"v_add_u32": x + y, "v_subrev_u32": y - x, "v_xor_b32": x ^ y, "v_or_b32": x | y}[op] & M32)
        elif op == "v_cmpx_le_u32":
            self.exec = self.exec & (np.asarray(self.get(words[1])) <= self.get(words[2]))
        elif op == "s_mov_b64":
            self.exec = np.ones(64, bool) if words[1] == "-1" else LANE == 0
        elif op in ("s_add_u32", "s_sub_u32", "s_lshr_b32", "s_lshl_b32", "s_xor_b32", "s_and_b32"):
            x, y = self.get(words[1]), self.get(words[2])
            self.put(words[0], {"s_add_u32": x + y, "s_sub_u32": x - y, "s_lshr_b32": x >> y, "s_lshl_b32": x << y,
                                "s_xor_b32": x ^ y, "s_and_b32": x & y}[op])
        elif op == "s_mov_b32":
            self.put(words[0], self.get(words[1]))
        elif op.startswith("s_cmp_"):
            x, y = self.get(words[0]), self.get(words[1])
            self.scc = {"eq": x == y, "lg": x != y, "ge": x >= y}[op[6:8]]
        elif op == "s_cselect_b32":
            self.put(words[0], self.get(words[1] if self.scc else words[2]))
        elif op == "s_branch" or (op == "s_cbranch_scc0" and not self.scc) or (op == "s_cbranch_scc1" and self.scc):
            self.pc = g.at[words[0]]
        else:
            check(op in ("s_nop", "s_sleep") or op.startswith("s_cbranch"), line)

    def end_tile(self):
        g, p = self.g, self.g.p
        check(not self.vm and not self.lds, "operations in flight at the end")
        if self.s["fail"] and g.spin == 0:       # as the kernel does: tell the others, and leave
            g.counter[2] = 1
            g.gave_up += 1
            self.done = True
            return
        check(self.s["fail"] == 0, "a wait has run out")
        ct, f0, count = g.tiles[self.tile]
        for u in range(p.units):
            lo, hi = p.sums(self.index, u, ct, f0, count)
            want = np.stack([lo, hi], -1).reshape(16, 4, 16)                     # [i][j][byte]
            for j in range(4):
                got = np.stack([self.v[r].astype(np.int32) for r in regs(gen.acc_reg(p.units, u, j))], 1)
                check(np.array_equal(got, np.stack([want[I, j, 4 * Q + k] for k in range(4)], 1)), "a wrong sum")
        codes, _, land = gen.expand_layout(p.units)[:3]
        self.codes = np.stack([self.v["v%d" % (codes + k)] for k in range(4)], 1)
        self.entries = np.stack([self.v["v%d" % (land + i)] for i in range(64)], 1).reshape(64, 16, 4)
        self.gf = self.s["gf"]
        self.tile += 1
        if self.tile == len(g.tiles):
            self.done = True
        else:
            self.begin()


class Group:
    def __init__(self, problem, tiles, rng, mutate=None, spin=1 << 20):
        self.p, self.tiles, self.spin, self.gave_up = problem, tiles, spin, 0
        lines = re.findall(r'"([^"]*)\\n\\t"', gen.emit(problem.units, problem.vec, expand=True))
        self.lines = mutate(lines) if mutate else lines
        self.at = {x[:-1]: i for i, x in enumerate(self.lines) if x.endswith(":")}
        self.lds32 = rng_array(rng, 2 * FILL // 4, 1 << 31).astype(np.uint32)
        self.counter = [0, 0, 0]
        self.eager = rng.choice((0.0, 0.01, 0.2))
        self.waves = [Wave(self, i) for i in range(4)]

    def first(self, tile):
        ct, f0, _ = self.tiles[tile]
        return ct * self.p.fills + f0

    def store(self, addr, data):
        check(bool((addr + 16 <= 2 * FILL).all()), "a store outside the buffers")
        for k in range(4):
            self.lds32[addr // 4 + k] = data[:, k]

    def run(self, rng, limit=300000):
        steps = 0
        while True:
            left = [w for w in self.waves if not w.done]
            if not left:
                return
            w = rng.choice(left)
            for _ in range(rng.choice((1, 10, 100, 400, 1000))):
                if w.done:
                    break
                w.step(rng)
                steps += 1
            check(steps < limit, "the wavefronts do not finish")


def run(variant, tiles, seed, fills=5, mutate=None, limit=300000):
    rng = random.Random(seed)
    problem = Problem(rng, variant[0], variant[1], fills, 1 + max(t[0] for t in tiles))
    with np.errstate(over="ignore"):
        group = Group(problem, tiles, rng, mutate)
        group.run(rng, limit)
    # of every fill four arrivals and four readers, and four arrivals behind the last one
    assert sum(group.counter[:2]) == 8 * sum(t[2] for t in tiles) + 4


# (column tile, first fill, fills): whole K, parts of K, the shortest a tile may be
TILES = {"one tile of three fills": [(0, 1, 3)], "three, four and three": [(1, 0, 3), (0, 1, 4), (1, 2, 3)], "five": [(0, 0, 5)],
         "two tiles": [(1, 0, 3), (0, 0, 3)]}


@pytest.mark.parametrize("tiles", TILES.values(), ids=TILES.keys())
@pytest.mark.parametrize("variant", [(2, True), (3, False), (6, True)], ids=str)
def test_sums_of_four_wavefronts(variant, tiles):
    run(variant, tiles, seed=variant[0] + len(tiles))


@pytest.mark.parametrize("variant", [v for v in gen.XVARIANTS if v[1] == (v[0] % 4 == 0) or v[0] in (2, 3)], ids=str)
def test_sums_of_four_wavefronts_in_every_height(variant):
    run(variant, TILES["two tiles"], seed=variant[0], fills=3)


@pytest.mark.parametrize("variant", [(2, True), (3, False), (6, True)], ids=str)
def test_waits_of_no_further_polls_end_in_every_wavefront(variant):
    """With a limit of zero polls a wavefront that looks too early gives up, and whoever waits for it does too: all of them
    leave, with nothing in flight."""
    gave_up = 0
    for seed in range(6):
        rng = random.Random(seed)
        with np.errstate(over="ignore"):
            group = Group(Problem(rng, variant[0], variant[1], 4, 2), [(1, 0, 4), (0, 0, 3)], rng, spin=0)
            group.run(rng)
        assert all(w.done for w in group.waves)
        gave_up += group.gave_up
    assert gave_up > 0


def without(pattern):
    def mutate(lines):
        hit = [i for i, line in enumerate(lines) if re.search(pattern, line)][0]
        return lines[:hit] + lines[hit + 1:]
    return mutate


def without_check_of(target):
    def mutate(lines):
        at = lines.index("s_cmp_ge_u32 %%[ev], %%[%s]" % target)
        return lines[:at + 1] + lines[at + 2:]
    return mutate


def no_wait_for_the_entries(lines):
    first = [i for i, line in enumerate(lines) if line.startswith("ds_write_b128")][0]
    wait = max(i for i in range(first) if lines[i].startswith("s_waitcnt vmcnt"))
    return lines[:wait] + lines[wait + 1:]


MUTATIONS = {"a chunk never stored": without(r"^ds_write_b128"), "the buffer not looked at before it is overwritten": without_check_of("free"),
             "the buffer not looked at before it is read": without_check_of("whole"), "chunks always into one buffer": without(r"^v_xor_b32 v\d+, 0x10000,"),
             "entries turned before they have landed": no_wait_for_the_entries, "filter codes of the same fill for ever": without(r"s_add_u32 %\[eoff\]")}


@pytest.mark.parametrize("mutate", MUTATIONS.values(), ids=MUTATIONS.keys())
@pytest.mark.parametrize("variant", [(2, True)], ids=str)
def test_the_model_objects_to_a_loop_without(variant, mutate):
    for seed in range(40):
        try:
            run(variant, [(1, 0, 4), (0, 0, 3)], seed, fills=4, mutate=mutate, limit=20000 * variant[0])
        except Violation:
            return
    raise AssertionError("no objection")
