#!/usr/bin/env python3
"""Writes lookup_mx.inc: the fill loop of lutgemm_mx_kernel.hip as inline assembly, one macro per tile height.

A wavefront owns U units of 64 output pixels and 8 columns, and runs alone on its SIMD (four wavefronts per workgroup,
512 registers each), so that nothing but the order of its own instructions hides latency.  Per fill - 16 filter
elements x 8 columns = 128 slots, 256 bytes per activation code - and unit it makes 16 lookups, each

    v_perm_b32      address = buffer << 16 | activation row << 8 | chunk << 4
    ds_read_b128    eight table entries of one filter element

and for every two of them one v_smfmac_i32_16x16x128_i8 that adds the 32 bytes a lane has fetched into int32 sums.
The matrix instruction multiplies nothing: its other operand holds a one where a byte belongs to a sum and zeros
elsewhere.  The bytes are signed there, so entries are stored with both bytes' top bits flipped (entry ^ 0x8080) and
128 x 257 per slot is added back (CINIT, the value the sums of the low bytes start from).

Which lane looks up what: lane (q, i), i = lane & 15, works for pixels 4 i .. 4 i + 3 of the unit; the four lanes of
the same i share a pixel's 16 filter elements.  In step c (0..3) of pixel j lane (q, i) reads chunk
    (plane << 2) | ((i & 3) ^ c),    plane = (i >> 2) ^ (0, 3, 1, 2)[q],
so that over the steps the four lanes cover all 16 chunks and in every step the 16 lanes that the LDS serves
together - {0-3, 12-15, 20-23, 24-27} and {4-7, 8-11, 16-19, 28-31} of each half - read 16 different chunks: no bank
conflict whatever the codes are.  A lane therefore only ever needs the codes of one plane (four consecutive filter
elements, one dword) per pixel and fill: a 16-byte load brings those of its four pixels.

The stream of instructions (modelled here, so that every s_waitcnt is derived and not guessed):
  * reads run W ahead of the sums through a ring of W register quadruples, across the end of a fill;
  * the activations of unit u + D are loaded while unit u is looked up, across the end of a fill;
  * a fill's rows are 64 loads of 1 KiB, memory straight into the other LDS buffer, 16 per wavefront, spread over the
    first three quarters of the fill.

The wavefronts are held together by one LDS counter per buffer that only grows (EVENTS in the kernel): each adds 1
when its share of a fill has arrived and 1 when it has finished reading it.  A fill may be read once all four shares
are there (whole), and its buffer refilled once all four have read it (free).  Both are looked at ahead of the point
that needs them; a look that finds too small a count goes into a bounded loop of further looks (SPIN of them) out of
line, and a loop that runs out leaves the assembly with FAIL set.

The expanding form (emit(..., expand=True), macros MX_XFILLS_*) makes a fill's rows itself, out of the truth table:
nothing is written to memory and read back.  A wavefront makes the rows of 64 activation codes, in two blocks of 32.
Lane (s, c), s = bits 1-4 of the lane and c = bits 5 and 0, has the fill's filter element s: per block it loads 16
bytes - the entries of eight activation codes - of the table rows of the element's eight filter codes, turns that
8 x 8 square of 16-bit entries with 32 v_perm_b32 and stores eight 16-byte chunks, one per activation code.  Two
neighbouring lanes read 32 consecutive bytes, and 16 lanes that the LDS serves together store into 16 or 8 different
chunks.  (Lane order measured on the load, turn and store alone, 256 workgroups, us a fill: s in the low bits 1.76, its
loads alone 1.76; c in the low bits 0.90, its stores alone 0.85; this one 0.92, stores 0.51, which leaves the LDS to the
lookups.)  While fill f is looked up the entries of fill f + 1 are turned and stored, those of fill f + 2 loaded into the
registers that this leaves free, and the filter codes of fill f + 3 loaded; both stay loaded from tile to tile, which makes
three fills the shortest tile.  (With entries loaded and stored within one fill, us a fill for U = 2, 4, 8, 14: 1.43, 1.59,
2.03, 2.69; like this 1.10, 1.28, 1.78, 2.65 on 1x1 layers of 18 and 72 fills, 0.95 for U = 2 and
2.55 for U = 14 on 3x3 layers.)
"""
import sys

UNITS = (2, 3, 4, 6, 8, 10, 13, 16, 20, 25)   # tile heights: units of 64 pixels per wavefront
VARIANTS = [(u, vec) for u in UNITS for vec in (True, False)]
W = 8                                         # lookups in flight (a unit is a whole number of rings)
LOADS = 16                                    # 1 KiB loads per wavefront and fill
XUNITS = (2, 3, 4, 6, 8, 10, 12, 13, 14, 16, 18)   # tile heights of the expanding form (20 and 25 leave it too few registers)
XVARIANTS = [(u, vec) for u in XUNITS for vec in (True, False)]
CODE_BYTES = 256                              # packed filter codes of a fill: 128 x uint16

# registers the assembly uses by number
V_A, V_IDX, V_SEL, V_CH0, V_CH1, V_L16 = 0, 4, 5, 9, 10, 11
V_ADDR = 12                                   # four address temporaries
V_KOFF, V_Q, V_KW, V_TMP, V_POLL, V_CB = 16, 17, 18, 19, 20, 21
V_BASE = 22
AGPR_UNITS = 16                               # units whose sums live in AGPRs (16 registers each)


def ring_plan(units):
    """(D, slot of each unit): activations are loaded D units ahead.  Any D units that follow each other, across the end
    of a fill too, need different slots: runs of D or D + 1 slots, repeated."""
    if units <= 6:
        return units, list(range(units))
    for d in (5, 6, 4):
        for b in range(units // (d + 1) + 1):
            if (units - b * (d + 1)) % d == 0:
                runs = [d] * ((units - b * (d + 1)) // d) + [d + 1] * b
                return d, [s for run in runs for s in range(run)]
    raise ValueError(units)


class Stream:
    """Instruction text plus the two in-order queues a wavefront waits on."""

    def __init__(self):
        self.lines, self.slow, self.lds_q, self.vm_q, self.count = [], [], [], [], 0
        self.tags = {}                     # vector-memory operations that a loop carries: what they are

    def ins(self, text):
        self.lines.append(text)

    def lds(self, text):
        if len(self.lds_q) == 15:          # all that the counter holds (the expanding form's bursts of stores)
            self.wait_lds(self.lds_q[0])
        self.ins(text)
        self.count += 1
        self.lds_q.append(self.count)
        return self.count

    def vm(self, text, tag=None):
        self.ins(text)
        self.count += 1
        self.vm_q.append(self.count)
        self.tags[self.count] = tag
        assert len(self.vm_q) <= 63
        return self.count

    def carry(self, tags):                 # the operations in flight where a loop begins, as its end leaves them
        self.vm_q = []
        for tag in tags:
            self.count += 1
            self.vm_q.append(self.count)
            self.tags[self.count] = tag
        return {self.tags[op]: op for op in self.vm_q}

    def wait_lds(self, *ops):
        ops = [op for op in ops if op in self.lds_q]
        if ops:
            i = max(self.lds_q.index(op) for op in ops)
            self.ins("s_waitcnt lgkmcnt(%d)" % (len(self.lds_q) - 1 - i))
            del self.lds_q[:i + 1]

    def wait_vm(self, *ops):
        ops = [op for op in ops if op in self.vm_q]
        if ops:
            i = max(self.vm_q.index(op) for op in ops)
            self.ins("s_waitcnt vmcnt(%d)" % (len(self.vm_q) - 1 - i))
            del self.vm_q[:i + 1]


def layout(units):
    d, slots = ring_plan(units)
    ring = V_BASE + units
    ring += ring & 1
    win = ring + 4 * (max(slots) + 1)
    end = win + 4 * W
    vacc = 256 - 16 * max(0, units - AGPR_UNITS)
    assert end <= vacc and 16 % W == 0, (units, end, vacc)
    return d, slots, ring, win, end, vacc


def expand_layout(units):
    """Registers of the expanding form behind those of layout(): a fill's filter codes, the addresses of their table rows,
    the entries on their way in (two blocks of eight quadruples), the turned chunks on their way out, and the lane's
    offsets into a table row and into the LDS buffer."""
    end, vacc = layout(units)[4:]
    codes = end + (end & 1)
    row, land = codes + 4, codes + 12
    out = land + 64
    toff, ldst = out + 8, out + 9
    assert ldst < vacc, (units, ldst, vacc)
    return codes, row, land, out, toff, ldst


def acc_reg(units, u, j):
    if u < AGPR_UNITS:
        r = 16 * u + 4 * j
        return "a[%d:%d]" % (r, r + 3)
    r = layout(units)[5] + 16 * (u - AGPR_UNITS) + 4 * j
    return "v[%d:%d]" % (r, r + 3)


def emit(units, vec, expand=False):
    if not expand:
        return emit_form(units, vec, expand)[0]
    tags = []
    for _ in range(4):                     # until the loop's end leaves in flight what its beginning assumed
        text, end = emit_form(units, vec, expand, tags)
        if end == tags:
            return text
        tags = end
    raise ValueError(units)


def emit_form(units, vec, expand, carried=None):
    d, slots, ring, win, end, vacc = layout(units)
    n_look, n_pair = 16 * units, 8 * units
    st = Stream()
    labels = [0]

    def fresh(prefix):
        labels[0] += 1
        return "L%s%d_%%=" % (prefix, labels[0])

    def order(k):            # k-th lookup of a unit -> (pixel j, step c): two steps of one pixel, then the next pixel
        return (k // 2) % 4, (k // 8) * 2 + k % 2

    def quad(base, i):
        return "v[%d:%d]" % (base + 4 * i, base + 4 * i + 3)

    def act_load(u):
        st.ins("v_add_u32 v%d, v%d, v%d" % (V_TMP, V_BASE + u, V_KOFF))
        r = ring + 4 * slots[u]
        if vec:
            return [st.vm("buffer_load_dwordx4 v[%d:%d], v%d, %%[xq], 0 offen" % (r, r + 3, V_TMP), ("act", u, 0))]
        return [st.vm("buffer_load_dword v%d, v%d, %%[xq], %s offen" % (r + j, V_TMP, "0" if j == 0 else "%%[p%d]" % j),
                      ("act", u, j)) for j in range(4)]

    def koff_step():         # every lane's filter position moves on by four quads: (tap column, quad) with carries
        st.ins("v_add_u32 v%d, %%[dq], v%d" % (V_Q, V_Q))
        st.ins("v_add_u32 v%d, %%[dkw], v%d" % (V_KW, V_KW))
        st.ins("v_add_u32 v%d, %%[doff], v%d" % (V_KOFF, V_KOFF))
        st.ins("v_cmpx_le_u32 vcc, %%[c4], v%d" % V_Q)
        st.ins("v_subrev_u32 v%d, %%[c4], v%d" % (V_Q, V_Q))
        st.ins("v_add_u32 v%d, 1, v%d" % (V_KW, V_KW))
        st.ins("v_add_u32 v%d, %%[qoff], v%d" % (V_KOFF, V_KOFF))
        st.ins("s_mov_b64 exec, -1")
        st.ins("v_cmpx_le_u32 vcc, %%[kwn], v%d" % V_KW)
        st.ins("v_subrev_u32 v%d, %%[kwn], v%d" % (V_KW, V_KW))
        st.ins("v_add_u32 v%d, %%[kwoff], v%d" % (V_KOFF, V_KOFF))
        st.ins("s_mov_b64 exec, -1")

    def addresses(n):
        u, k = divmod(n % n_look, 16)
        j, c = order(k)
        st.ins("v_perm_b32 v%d, v%d, v%d, v%d" % (V_ADDR + n % 4, ring + 4 * slots[u] + j, V_CH0 if c < 3 else V_CH1, V_SEL + c))

    def read(n):
        return st.lds("ds_read_b128 %s, v%d" % (quad(win, n % W), V_ADDR + n % 4))

    def look(counter):       # one look at EVENTS[counter] (an SGPR operand with its LDS address)
        st.ins("v_mov_b32 v%d, %%[%s]" % (V_CB, counter))
        return st.lds("ds_read_b32 v%d, v%d" % (V_POLL, V_CB))

    def need(op, counter, target, code):
        """Goes on once the look `op` has found EVENTS at the target; otherwise looks again, out of line."""
        ok, slow = fresh("ok"), fresh("slow")
        if op is not None:
            st.wait_lds(op)
            st.ins("v_readfirstlane_b32 %%[ev], v%d" % V_POLL)
            st.ins("s_cmp_ge_u32 %%[ev], %s" % target)
            st.ins("s_cbranch_scc0 %s" % slow)
        else:
            st.ins("s_branch %s" % slow)
        st.ins("%s:" % ok)
        s = st.slow
        s.append("%s:" % slow)
        s.append("s_mov_b32 %[tmp], %[spin]")
        again = fresh("again")
        s.append("%s:" % again)
        s.append("v_mov_b32 v%d, %%[%s]" % (V_CB, counter))
        s.append("ds_read_b32 v%d, v%d" % (V_POLL, V_CB))
        s.append("v_mov_b32 v%d, %%[cb0]" % V_CB)
        s.append("ds_read_b32 v%d, v%d offset:8" % (V_TMP, V_CB))       # ABORT
        s.append("s_waitcnt lgkmcnt(0)")
        s.append("v_readfirstlane_b32 %%[ev], v%d" % V_POLL)
        s.append("s_cmp_ge_u32 %%[ev], %s" % target)
        s.append("s_cbranch_scc1 %s" % ok)
        s.append("v_readfirstlane_b32 %%[ev], v%d" % V_TMP)
        s.append("s_mov_b32 %%[fail], %d" % code)
        s.append("s_cmp_lg_u32 %[ev], 0")
        s.append("s_cbranch_scc1 Lend_%=")
        s.append("s_cmp_eq_u32 %[tmp], 0")
        s.append("s_cbranch_scc1 Lend_%=")
        s.append("s_mov_b32 %[fail], 0")
        s.append("s_sub_u32 %[tmp], %[tmp], 1")
        s.append("s_sleep 1")
        s.append("s_branch %s" % again)

    def count(counter):      # EVENTS[counter] += 1, by one lane
        st.ins("v_mov_b32 v%d, %%[%s]" % (V_CB, counter))
        st.ins("v_mov_b32 v%d, 1" % V_POLL)
        st.ins("s_mov_b64 exec, 1")
        op = st.lds("ds_add_u32 v%d, v%d" % (V_CB, V_POLL))
        st.ins("s_mov_b64 exec, -1")
        return op

    if expand:
        codes, row, land, out, toff, ldst = expand_layout(units)

    def row_addresses():     # of the table rows that the fill's eight filter codes of this lane name
        for i in range(8):
            st.ins("v_mad_u32_u16 v%d, v%d, %%[rowb], v%d%s"
                   % (row + i, codes + i // 2, toff, " op_sel:[1,0,0,0]" if i & 1 else ""))

    def row_load(i):         # entries of eight activation codes (block i / 8) of column i % 8
        b, j = divmod(i, 8)
        return st.vm("buffer_load_dwordx4 %s, v%d, %%[erc], 0 offen offset:%d" % (quad(land, i), row + j, 64 * b), ("row", i))

    def chunk_store(i):      # activation code i % 8 of block i / 8: the square's column, as a row's 16 bytes
        b, e = divmod(i, 8)
        for k in range(4):
            st.ins("v_perm_b32 v%d, v%d, v%d, %%[%s]" % (out + 4 * (i & 1) + k, land + 4 * (8 * b + 2 * k + 1) + e // 2,
                                                        land + 4 * (8 * b + 2 * k) + e // 2, "hi" if e & 1 else "lo"))
        st.lds("ds_write_b128 v%d, %s offset:%d" % (ldst, quad(out, i & 1), (e >> 2) * 256 + (e & 3) * 16384 + b * 2048))

    # ---- prologue: the sums' start values, the first activations, the first reads ----
    st.ins("s_nop 7")   # the caller's last vector instructions may have written the scalar operands of the loads below
    acts = {}
    for u in range(d):
        acts[u] = act_load(u)
    for u in range(units):
        for j in range(4):
            for r in range(4):
                name = acc_reg(units, u, j)
                base = int(name[2:name.index(":")]) + r
                if name[0] == "a":
                    st.ins("v_accvgpr_write_b32 a%d, %s" % (base, "0" if r & 1 else "v%d" % V_POLL))
                else:
                    st.ins("v_mov_b32 v%d, %s" % (base, "0" if r & 1 else "v%d" % V_POLL))
    st.ins("s_mov_b32 %[fail], 0")
    need(None, "cbcur", "%[whole0]", 1)
    if expand:               # nothing is in flight but what the loop counts itself
        st.wait_vm(*st.vm_q)
    st.wait_vm(*acts[0])
    pending = {}
    for n in range(W):
        addresses(n)
        pending[n] = read(n)
    st.ins("Lfill_%=:")
    # ---- one fill ----
    # cbcur / cboth: LDS addresses of the counters of this fill's buffer and of the other one; whole: what the other
    # counter must reach for the next fill to be readable (0 behind the tile's last fill); free: ... for the other
    # buffer to be refilled
    entering = {}
    if expand:
        entering = st.carry(carried)
        acts = {u: [op for tag, op in entering.items() if tag[:2] == ("act", u)] for u in range(d)}
    entry_vm, entry_lds = list(st.vm_q), list(st.lds_q)
    first_load = 4 if units > 2 else 2                      # pair in which the first load is issued
    last_load = n_pair * 3 // 4 if units > 3 else n_pair // 2
    load_at = [first_load + (last_load - first_load) * i // (LOADS - 1) for i in range(LOADS)]
    cross = n_pair - W // 2                                 # pair whose reads are the next fill's first
    arrive_at = cross - 3 if units > 3 else cross - 1
    look_whole_at = cross - 2 if units > 3 else cross
    look_free_at = 0
    if expand:               # stores from when the buffer may be free to the arrival, a block's loads behind its stores
        first_store = 1 if units == 2 else 2
        store_at = [first_store + (arrive_at - 1 - first_store) * i // 15 for i in range(LOADS)]
        per_pair = 2 if units <= 3 else 1
        load_at = [store_at[i // 8 * 8 + 7] + i % 8 // per_pair for i in range(LOADS)]
        assert load_at[-1] < n_pair and load_at[7] <= store_at[15]
    loaded = stored = 0
    load_ops = []
    ops = {}
    stepped = False
    for p in range(n_pair):
        n = 2 * p
        u, k = divmod(n, 16)
        j, _ = order(k)
        if p == look_free_at:
            ops["free"] = look("cboth")
        st.wait_lds(pending[n], pending[n + 1])
        m = n + W
        if p == arrive_at:   # (a wavefront's LDS operations happen in order: its stores before this)
            assert stored == LOADS if expand else loaded == LOADS
            if not expand:
                st.wait_vm(*load_ops)
            ops["arrive"] = count("cboth")
        if p == look_whole_at:
            ops["whole"] = look("cboth")
        if p == cross:
            need(ops["whole"], "cboth", "%[whole]", 2)
            st.ins("v_xor_b32 v%d, 0x01000000, v%d" % (V_CH0, V_CH0))
            st.ins("v_xor_b32 v%d, 0x01000000, v%d" % (V_CH1, V_CH1))
        mu, mk = divmod(m % n_look, 16)
        if mk == 0:
            st.wait_vm(*acts[mu])
        addresses(m)
        addresses(m + 1)
        st.ins("v_smfmac_i32_16x16x128_i8 %s, v[%d:%d], v[%d:%d], v%d"
               % (acc_reg(units, u, j), V_A, V_A + 3, win + 4 * (n % W), win + 4 * (n % W) + 7, V_IDX))
        pending[m] = read(m)
        pending[m + 1] = read(m + 1)
        if mk == 14:         # the unit's last addresses are made: its slot takes the activations D units on
            nu = mu + d
            if nu >= units and not stepped:
                koff_step()
                stepped = True
            acts[nu % units] = act_load(nu % units)
        if expand:
            if p == 0:
                row_addresses()
                ops["codes"] = st.vm("buffer_load_dwordx4 %s, v%d, %%[wrc], %%[eoff] offen" % (quad(codes, 0), V_L16))
            if p == store_at[0]:
                need(ops["free"], "cboth", "%[free]", 3)
            while stored < LOADS and store_at[stored] == p:
                if stored % 8 == 0:
                    st.wait_vm(*[entering.get(("row", i)) for i in range(stored, stored + 8)])
                chunk_store(stored)
                stored += 1
            while loaded < LOADS and load_at[loaded] == p:
                load_ops.append(row_load(loaded))
                loaded += 1
            continue
        if p == first_load:
            need(ops["free"], "cboth", "%[free]", 3)
        while loaded < LOADS and load_at[loaded] == p:
            if loaded % 4 == 0:
                st.ins("s_add_u32 m0, %%[edst], %d" % (loaded * 1024))
                st.ins("s_add_u32 %%[tmp], %%[eoff], %d" % (loaded * 1024))
            load_ops.append(st.vm("buffer_load_dwordx4 v%d, %%[erc], %%[tmp] offen offset:%d lds" % (V_L16, loaded % 4 * 1024)))
            loaded += 1
    assert stepped and loaded == LOADS
    # this wavefront is done with the fill; on to the next one
    count("cbcur")
    st.ins("s_xor_b32 %[cbcur], %[cbcur], 4")
    st.ins("s_xor_b32 %[cboth], %[cboth], 4")
    if expand:
        st.wait_vm(ops["codes"])
        st.ins("v_xor_b32 v%d, 0x10000, v%d" % (ldst, ldst))
    else:
        st.ins("s_xor_b32 %[edst], %[edst], 0x10000")
    # counts: the buffer's next fill is two on (8 more events); whole and free alternate between the buffers
    st.ins("s_add_u32 %[gf], %[gf], 1")
    st.ins("s_sub_u32 %[left], %[left], 1")
    st.ins("s_cmp_eq_u32 %[left], 0")
    st.ins("s_cbranch_scc1 Lend_%=")
    # fill gf + 1 goes into the other buffer, free once fill gf - 1 is read: 4 (2 ((gf - 1) / 2) + 2)
    st.ins("s_sub_u32 %[tmp], %[gf], 1")
    st.ins("s_lshr_b32 %[tmp], %[tmp], 1")
    st.ins("s_lshl_b32 %[tmp], %[tmp], 3")
    st.ins("s_add_u32 %[free], %[tmp], 8")
    # ... and whole at 4 (2 ((gf + 1) / 2) + 1); nobody reads behind the tile's last fill
    st.ins("s_add_u32 %[tmp], %[gf], 1")
    st.ins("s_lshr_b32 %[tmp], %[tmp], 1")
    st.ins("s_lshl_b32 %[tmp], %[tmp], 3")
    st.ins("s_add_u32 %[whole], %[tmp], 4")
    st.ins("s_cmp_eq_u32 %[left], 1")
    st.ins("s_cselect_b32 %[whole], 0, %[whole]")
    # the rows that follow: the tile's next fill, or the first one of the workgroup's next tile, or none: then ENEXT has bit
    # 31 set, which moves into the vector offset.  That one is what a descriptor's bounds check covers; the scalar offset
    # must stay inside the rows by itself.
    # (expanding: the same for the filter codes, which are loaded two fills further ahead)
    st.ins("s_add_u32 %%[eoff], %%[eoff], %d" % (CODE_BYTES if expand else 0x10000))
    st.ins("s_cmp_eq_u32 %%[left], %d" % (3 if expand else 1))
    st.ins("s_cselect_b32 %[eoff], %[enext], %[eoff]")
    st.ins("s_and_b32 %[tmp], %[eoff], 0x80000000")
    st.ins("s_xor_b32 %[eoff], %[eoff], %[tmp]")
    st.ins("v_or_b32 v%d, %%[tmp], v%d" % (V_L16, V_L16))
    # the state the loop was entered with: W reads and D units of activations in flight, nothing else that counts
    # (operations older than those only make a wait stricter)
    if not expand:
        assert st.vm_q == [op for x in range(1, d) for op in acts[x]][-len(st.vm_q):] or not st.vm_q
        assert len(st.vm_q) <= len(entry_vm)
    leaving = [st.tags[op] for op in st.vm_q]
    assert None not in leaving
    assert [op for op in st.lds_q if op in pending.values()] == [pending[n_look + i] for i in range(W)]
    assert len(entry_lds) == W
    st.ins("s_branch Lfill_%=")
    st.lines += st.slow
    st.ins("Lend_%=:")
    st.ins("s_waitcnt vmcnt(0) lgkmcnt(0)")
    st.ins("s_nop 15")
    st.ins("s_nop 15")

    outs = []
    for u in range(units):
        lo = acc_reg(units, u, 0)
        b = int(lo[2:lo.index(":")])
        outs.append('"={%s[%d:%d]}"(ACC[%d])' % (lo[0], b, b + 15, u))
    inouts = [("CH0", V_CH0), ("CH1", V_CH1), ("KOFF", V_KOFF), ("QL", V_Q), ("KWL", V_KW), ("CINIT", V_POLL), ("L16", V_L16)]
    outs += ['"+{v%d}"(%s)' % (r, name) for name, r in inouts]
    if expand:
        outs += ['"+{v[%d:%d]}"(CODES)' % (codes, codes + 3), '"+{v%d}"(LDST)' % ldst]
    if expand:
        outs += ['"+{v[%d:%d]}"(LAND[%d])' % (land + 16 * i, land + 16 * i + 15, i) for i in range(4)]
    scalars = [("cbcur", "CBCUR"), ("cboth", "CBOTH")] + ([] if expand else [("edst", "EDST")]) + [("gf", "GF"), ("left", "LEFT"), ("free", "FREE"),
               ("whole", "WHOLE"), ("eoff", "EOFF")]
    outs += ['[%s] "+&s"(%s)' % s for s in scalars]
    outs += ['[fail] "=&s"(FAIL)', '[tmp] "=&s"(TMP)', '[ev] "=&s"(EV)']
    ins = ['"{v[%d:%d]}"(AOP)' % (V_A, V_A + 3), '"{v%d}"(IDX)' % V_IDX]
    ins += ['"{v%d}"(SEL[%d])' % (V_SEL + c, c) for c in range(4)]
    ins += ['"{v%d}"(BASE[%d])' % (V_BASE + u, u) for u in range(units)]
    ins += ['[%s] "s"(%s)' % x for x in [("xq", "XQ"), ("erc", "ERC"), ("enext", "ENEXT"), ("cb0", "CB0"), ("spin", "SPIN"), ("whole0", "WHOLE0"),
                                          ("dq", "KS.dq"), ("dkw", "KS.dkw"), ("doff", "KS.doff"), ("c4", "KS.c4"),
                                          ("qoff", "KS.qoff"), ("kwn", "KS.kwn"), ("kwoff", "KS.kwoff")]]
    if not vec:
        ins += ['[p%d] "s"(KS.pitch[%d])' % (j, j - 1) for j in (1, 2, 3)]
    clob = ['"v%d"' % r for r in list(range(V_ADDR, V_ADDR + 4)) + [V_TMP, V_CB] + list(range(ring, end))]
    if expand:
        ins += ['"{v%d}"(TOFF)' % toff] + ['[%s] "s"(%s)' % x for x in [("wrc", "WRC"), ("rowb", "512u"), ("lo", "0x05040100u"),
                                                                      ("hi", "0x07060302u")]]
        clob += ['"v%d"' % r for r in range(row, toff) if not land <= r < land + 64]
    clob += ['"m0"', '"scc"', '"vcc"', '"memory"']
    args = ("ACC, CH0, CH1, KOFF, QL, KWL, CINIT, L16, CBCUR, CBOTH, EDST, GF, LEFT, FREE, WHOLE, EOFF, FAIL, TMP, EV, AOP, "
            "IDX, SEL, BASE, XQ, ERC, ENEXT, CB0, SPIN, WHOLE0, KS")
    if expand:
        args = args.replace("EDST, ", "") + ", WRC, CODES, LDST, TOFF, LAND"
    text = " \\\n        ".join('"%s\\n\\t"' % line for line in st.lines)
    text = ("#define MX_%sFILLS_U%d_%s(%s) \\\n    asm volatile( \\\n        %s \\\n        : %s \\\n        : %s \\\n        : %s)\n"
            % ("X" if expand else "", units, "V" if vec else "S", args, text, ", ".join(outs), ", ".join(ins), ", ".join(clob)))
    return text, leaving


if __name__ == "__main__":
    print("// Generated by gen_lookup_mx.py -- do not edit.")
    for variant in VARIANTS:
        print(emit(*variant))
    for variant in XVARIANTS:
        print(emit(*variant, expand=True))
    sys.exit(0)
