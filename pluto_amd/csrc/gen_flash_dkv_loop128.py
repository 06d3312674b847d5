#!/usr/bin/env python3
"""Writes flash_dkv_loop128.inc: the hand-scheduled gfx950 instruction stream of
the key-owned attention backward kernel for heads of 128 channels
(flash_dkv_wide.hip), the body of one `asm volatile` statement with a fixed
register allocation.

As for 64 channels (gen_flash_dkv_loop.py) a wave owns 64 keys, two halves of 32,
so that every A operand read from LDS feeds two matrix instructions.  A wave of 32
keys reads 32 KiB for 32 matrix instructions of 32 cycles, which for four waves
is all that LDS can deliver.  Here the accumulators fill the 256 AGPRs and K and
V half of the VGPRs, so there is one S and one dP a half and the vector work of a
block runs beside that block's own later products.  Per block of 32 queries, 64
matrix instructions, each followed by what one of them (32 cycles) hides:

  instructions   matrix                      vector
  0 .. 15        S, both halves
  16 .. 31       dP, both halves             P of rows 0-7, 16-23 (accumulator registers 0-7)
  32 .. 39       dV, first 16 rows           their dS; P of the other rows
  40 .. 47       dK, first 16 rows           P of the other rows
  48 .. 55       dV, second 16 rows          their dS
  56 .. 63       dK, second 16 rows

The 32 A operands of a block pass through a ring of eight register groups, each
refilled from LDS as soon as its second product is on its way (seven pairs, 448
cycles, before its next use).  Row statistics are read into the accumulators of half 0
and serve as the C operand of the first product of both halves.  dS is packed over
dP; P is packed beside S (dS needs it unrounded).

Query blocks travel global -> LDS through a ring of four stages; the barrier of
step b stands before instruction 48 of block b - 1, where the last of that block's
operands have been requested, and block b + 2 is requested behind it.  The second
wave's keys start 64 rows later: it idles for the first two blocks.

A wave's first two blocks (the causal diagonal crosses them) and its last one (the
sequence may end inside it) run a variant that compares every element's query row
with two per-lane bounds.

Usage: python gen_flash_dkv_loop128.py [output]   (default: flash_dkv_loop128.inc
beside this file)
"""
import os
import sys

from gen_flash_dkv_loop import MFMA, at_, c_string, vt

D = 128
KS = D // 16
DB = D // 32
RING = 4                # LDS stages
POOL = 8                # register groups the A operands pass through
TILE_BYTES = 32 * D * 2
STAT_BYTES = 256
STAGE_BYTES = 2 * TILE_BYTES + 2 * STAT_BYTES
ROW_BYTES = D * 2
FILL_OPS = 9            # vector-memory operations a wave and stage: 4 Q, 4 dO, 1 statistics
GAP = 28                # issue cycles beside one matrix instruction


class Registers:
    def __init__(self):
        at = 4          # v0 .. v3 stay with the compiler

        def take(n=1):
            nonlocal at
            first = at
            at += n
            return first
        self.QFILL = [take(), take()]
        self.GFILL = [take(), take()]
        self.SFILL = take()
        self.N4 = take()
        self.TL4 = take()
        self.inputs_end = at
        self.ROWADDR = [take() for _ in range(4)]       # moved from stage to stage
        self.TRADDR = [take() for _ in range(2)]
        self.STATADDR = take()
        self.moved_end = at
        self.FTMP = [take(), take()]
        self.F = [take(), take()]
        self.LIM = take()
        self.NEG = take()
        assert at == 24
        self.PB = [take(4), take(4)]                    # [c]
        self.OPS = [take(4) for _ in range(POOL)]
        self.temps_end = at
        assert at == 64
        self.KF = [[64 + 4 * (KS * c + ks) for ks in range(KS)] for c in range(2)]
        self.VF = [[128 + 4 * (KS * c + ks) for ks in range(KS)] for c in range(2)]
        self.S = [192, 208]
        self.DP = [224, 240]
        self.DK = [[16 * (DB * c + db) for db in range(DB)] for c in range(2)]
        self.DV = [[128 + 16 * (DB * c + db) for db in range(DB)] for c in range(2)]


def weight(text):
    if text.startswith("v_exp"):
        return 16
    return 4


class Emitter:
    def __init__(self):
        self.r = Registers()
        self.lines = []
        self.lds_queue = []

    def emit(self, text):
        self.lines.append(text)

    # ---- LDS reads with lgkmcnt bookkeeping (reads return in order, the counter holds 15) ----
    def lds_read(self, text, dest):
        if len(self.lds_queue) >= 15:
            self.emit("s_waitcnt lgkmcnt(14)")
            self.lds_queue = self.lds_queue[len(self.lds_queue) - 14:]
        self.emit(text)
        self.lds_queue.append(dest)

    def wait_for(self, dest):
        last = -1
        for i, d in enumerate(self.lds_queue):
            if d == dest:
                last = i
        if last < 0:
            return
        self.emit("s_waitcnt lgkmcnt(%d)" % (len(self.lds_queue) - 1 - last))
        self.lds_queue = self.lds_queue[last + 1:]

    # ---- the 32 A operands of a block, by the pair of products they feed ----------------------
    def operand_reads(self, pair):
        """Rows of Q, rows of dO, then dO^T and Q^T of rows 0-15, of rows 16-31."""
        r = self.r
        reg = r.OPS[pair % POOL]
        if pair < 16:
            tensor, ks = divmod(pair, 8)
            return [("ds_read_b128 %s, v%d offset:%d" %
                     (vt(reg, 4), r.ROWADDR[ks % 4], tensor * TILE_BYTES + ks // 4 * 128), ("op", pair))]
        s2, rest = divmod(pair - 16, 8)
        tile = TILE_BYTES if rest < 4 else 0
        db = rest % 4
        return [("ds_read_b64_tr_b16 %s, v%d offset:%d" %
                 (vt(reg + 2 * part, 2), r.TRADDR[db % 2],
                  tile + (16 * s2 + 8 * part) * ROW_BYTES + db // 2 * 128), ("op", pair))
                for part in range(2)]

    def stat_reads(self, name):
        """Register i <- statistic of query 8 (i / 4) + 4 h + i % 4."""
        r = self.r
        base, offset = (r.S[0], 0) if name == "lse" else (r.DP[0], STAT_BYTES)
        return [("ds_read_b128 %s, v%d offset:%d" % (vt(base + 4 * j, 4), r.STATADDR, offset + 32 * j), name)
                for j in range(4)]

    # ---- matrix side: (what it waits for, instruction) -----------------------------------------
    def products(self):
        r = self.r
        out = []
        for tensor, (acc, frags, stat) in enumerate(((r.S, r.KF, "lse"), (r.DP, r.VF, "del"))):
            for ks in range(KS):
                pair = 8 * tensor + ks
                for c in (1, 0):
                    start = vt(acc[0], 16) if ks == 0 else vt(acc[c], 16)
                    needs = [("op", pair)] + ([stat] if ks == 0 else []) if c == 1 else []
                    out.append((needs, "%s %s, %s, %s, %s" %
                                (MFMA, vt(acc[c], 16), vt(r.OPS[pair % POOL], 4), vt(frags[c][ks], 4), start)))
        for s2 in range(2):
            for tensor in range(2):
                for db in range(DB):
                    pair = 16 + 8 * s2 + 4 * tensor + db
                    for c in (0, 1):
                        acc = at_((r.DV if tensor == 0 else r.DK)[c][db], 16)
                        b = r.PB[c] if tensor == 0 else r.DP[c] + 8 * s2
                        out.append(([("op", pair)] if c == 0 else [], "%s %s, %s, %s, %s" %
                                    (MFMA, acc, vt(r.OPS[pair % POOL], 4), vt(b, 4), acc)))
        assert len(out) == 64
        return out

    # ---- vector side ------------------------------------------------------------------------------
    def probabilities(self, s2, masked):
        """P of both halves, accumulator registers 8 s2 .. 8 s2 + 7, four at a time."""
        r = self.r
        exps, packs = [], []
        for c in range(2):
            S = r.S[c]
            for first in range(8 * s2, 8 * s2 + 8, 4):
                group = range(first, first + 4)
                if masked:
                    for i in group:
                        ci = 8 * (i // 4) + i % 4
                        exps.append("v_cmp_ge_i32 vcc, %d, v%d" % (ci, r.F[c]))
                        exps.append("v_cmp_le_i32_e64 %%[mpair], %d, v%d" % (ci, r.LIM))
                        exps.append("s_and_b64 vcc, vcc, %[mpair]")
                        exps.append("v_cndmask_b32 v%d, v%d, v%d, vcc" % (S + i, r.NEG, S + i))
                exps += ["v_mul_f32 v%d, %%[scale2], v%d" % (S + i, S + i) for i in group]
                exps += ["v_exp_f32 v%d, v%d" % (S + i, S + i) for i in group]
            for w in range(4):
                packs.append("v_cvt_pk_bf16_f32 v%d, v%d, v%d" %
                             (r.PB[c] + w, S + 8 * s2 + 2 * w, S + 8 * s2 + 2 * w + 1))
        return exps, packs

    def score_gradients(self, s2):
        r = self.r
        items = []
        for c in range(2):
            S, DP = r.S[c] + 8 * s2, r.DP[c] + 8 * s2
            items += ["v_mul_f32 v%d, v%d, v%d" % (DP + i, S + i, DP + i) for i in range(8)]
            items += ["v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (DP + w, DP + 2 * w, DP + 2 * w + 1)
                      for w in range(4)]
        return items

    @staticmethod
    def spread(gaps, items, first, last):
        """Deals items evenly over gaps first .. last."""
        items = list(items)
        for g in range(first, last + 1):
            left = sum(weight(t) for t in items)
            share, taken = -(-left // (last - g + 1)), 0
            while items and taken < share:
                taken += weight(items[0])
                gaps[g].append(items.pop(0))
        assert not items

    @staticmethod
    def fill_up(gaps, items, which):
        """Fills gaps up to GAP cycles beside what they hold; returns what is left."""
        items = list(items)
        for g in which:
            used = sum(weight(t) for t in gaps[g])
            while items and used + weight(items[0]) <= GAP + 8:
                used += weight(items[0])
                gaps[g].append(items.pop(0))
        return items

    def vector_gaps(self, masked):
        """The instruction after which each vector item stands.  Results of matrix
        instruction i are read from gap i + 2 on, operands written before gap i - 1;
        P of the second rows is packed once instruction 39 has read the first's."""
        gaps = [[] for _ in range(64)]
        exps, packs = self.probabilities(0, masked)
        self.spread(gaps, exps + packs, 17, 30)
        self.spread(gaps, self.score_gradients(0), 33, 38)
        exps, packs = self.probabilities(1, masked)
        exps = self.fill_up(gaps, exps, [31] + list(range(33, 39)))
        self.spread(gaps, exps + packs, 39, 46)
        self.spread(gaps, self.score_gradients(1), 47, 54)
        return gaps

    # ---- stages ---------------------------------------------------------------------------------
    def barrier(self):
        """Step s = tcount: block s has landed for every wave, everyone is done with
        block s - 2, whose stage takes block s + 2."""
        e = self.emit
        e("s_waitcnt vmcnt(%d)" % (FILL_OPS * (RING - 3)))
        e("s_barrier")

    def advance(self):
        """Moves the read addresses to the stage of step tcount and counts it."""
        r = self.r
        out = ["s_and_b32 %%[t0], %%[tcount], %d" % (RING - 1),
               "s_cmp_eq_u32 %[t0], 0",
               "s_mov_b32 %%[t0], %d" % STAGE_BYTES,
               "s_cselect_b32 %%[t0], %d, %%[t0]" % (-(RING - 1) * STAGE_BYTES)]
        out += ["v_add_u32 v%d, %%[t0], v%d" % (v, v) for v in r.ROWADDR + [r.STATADDR] + r.TRADDR]
        return out

    def fill_groups(self, stage=None):
        """The requests of block tcount + 2 (or of `stage`, at the start), one list a
        vector-memory instruction.  The running offsets are added into the lanes' (a
        descriptor's range check sees the vector offset only); an instruction's offset
        moves its LDS and its global address.  One other instruction stands
        between a write of M0 and the request that reads it."""
        r = self.r
        groups = []
        if stage is None:
            head = ["s_add_u32 %%[t1], %%[tcount], %d" % (RING - 2),
                    "s_and_b32 %%[t1], %%[t1], %d" % (RING - 1),
                    "s_mul_i32 %%[t1], %%[t1], %d" % STAGE_BYTES]
        else:
            head = ["s_mov_b32 %%[t1], %d" % (stage * STAGE_BYTES)]
        for tensor, (fill, name) in enumerate(((r.QFILL, "q"), (r.GFILL, "g"))):
            for pair in range(2):
                setup = []
                if pair == 0:
                    setup += head if tensor == 0 else []
                    setup.append("s_add_u32 m0, %[ldsq], %[t1]" if tensor == 0 else
                                 "s_add_u32 m0, m0, %d" % TILE_BYTES)
                    source = "%%[%soff]" % name
                else:
                    setup.append("s_add_u32 %%[t0], %%[%soff], %%[%seight]" % (name, name))
                    source = "%[t0]"
                setup += ["v_add_u32 v%d, %s, v%d" % (r.FTMP[i], source, fill[i]) for i in range(2)]
                for i in range(2):
                    groups.append((setup if i == 0 else []) +
                                  ["buffer_load_dwordx4 v%d, %%[%srsrc], 0 offen offset:%d lds" %
                                   (r.FTMP[i], name, 1024 * (2 * pair + i))])
            groups[-1].append("s_add_u32 %%[%soff], %%[%soff], %%[%sstep]" % (name, name, name))
        groups.append(["s_add_u32 m0, %[ldss], %[t1]",
                       "v_add_u32 v%d, %%[soff], v%d" % (r.FTMP[0], r.SFILL),
                       "buffer_load_dword v%d, %%[srsrc], 0 offen lds" % r.FTMP[0],
                       "s_add_u32 %[soff], %[soff], 128"])
        assert len(groups) == FILL_OPS
        return groups

    def whole_step(self):
        self.barrier()
        for text in self.advance():
            self.emit(text)
        for group in self.fill_groups():
            for text in group:
                self.emit(text)
        self.emit("s_add_u32 %[tcount], %[tcount], 1")

    # ---- one block ---------------------------------------------------------------------------------
    def rows_of_next(self):
        """Reads that a block finds on their way: (gap of the block before, reads)."""
        lse = self.stat_reads("lse")
        out = []
        for k in range(8):
            out.append((49 + 2 * k, self.operand_reads(k)))
        out.append((56, lse[:2]))
        out.append((58, lse[2:]))
        return sorted(out, key=lambda x: x[0])

    def block(self, masked):
        r = self.r
        e = self.emit
        if masked:
            e("s_lshl_b32 %[t0], %[bcount], 5")
            e("v_subrev_u32 v%d, %%[t0], v%d" % (r.F[0], r.N4))
            e("v_subrev_u32 v%d, %%[t0], v%d" % (r.LIM, r.TL4))
            e("v_add_u32 v%d, 32, v%d" % (r.F[1], r.F[0]))
        reads = [[] for _ in range(64)]
        for j, read in enumerate(self.stat_reads("del")):
            reads[1 + j].append(read)
        for pair in range(8, 32):
            reads[2 * (pair - 8) + 1] += self.operand_reads(pair)
        for gap, items in self.rows_of_next():
            reads[gap] += items
        other = [[] for _ in range(64)]
        for i, text in enumerate(self.advance()):
            other[48].append(text)
        for i, group in enumerate(self.fill_groups()):
            other[51 + i] += group
        other[61].append("s_add_u32 %[tcount], %[tcount], 1")
        vector = self.vector_gaps(masked)
        for g, (needs, text) in enumerate(self.products()):
            if g == 48:
                self.barrier()
            for need in needs:
                self.wait_for(need)
            e(text)
            for item in other[g]:
                e(item)
            for item, dest in reads[g]:
                self.lds_read(item, dest)
            for item in vector[g]:
                e(item)

    def outputs(self):
        """(name of the descriptor, accumulators, whether they take the scale)."""
        return (("dk", self.r.DK, True), ("dv", self.r.DV, False))

    def store(self):
        """The accumulators leave through the wave's 8 KiB of LDS, 32 keys x 64 channels at
        a time, so that every store instruction writes whole rows (16 lanes x 16
        bytes); a descriptor ends at the sequence's last row.  Here and not behind the
        statement because the compiler has no registers to take 256 accumulators in."""
        r = self.r
        e = self.emit
        lane, n, write, read, out = 64, 65, 66, 67, 68
        slot, wait = [70, 71, 72, 73], 74
        values, rows = 80, [112, 144]
        e("v_mbcnt_lo_u32_b32 v%d, -1, 0" % lane)
        e("v_mbcnt_hi_u32_b32 v%d, -1, v%d" % (lane, lane))
        # write: row n = lane % 32, 16-byte piece (8 d2 + 2 j + h) ^ n % 16
        e("v_and_b32 v%d, 31, v%d" % (n, lane))
        e("v_lshrrev_b32 v%d, 5, v%d" % (write, lane))
        e("v_and_b32 v%d, 15, v%d" % (wait, lane))
        e("v_xor_b32 v%d, v%d, v%d" % (write, write, wait))
        e("v_lshlrev_b32 v%d, 4, v%d" % (write, write))
        e("v_lshl_add_u32 v%d, v%d, 8, v%d" % (write, n, write))
        e("v_add_u32 v%d, %%[area], v%d" % (write, write))
        # read: row 4 i + lane / 16, piece lane % 16 ^ row % 16
        e("v_lshrrev_b32 v%d, 4, v%d" % (n, lane))
        e("v_xor_b32 v%d, v%d, v%d" % (read, n, wait))
        e("v_lshlrev_b32 v%d, 4, v%d" % (read, read))
        e("v_lshl_add_u32 v%d, v%d, 8, v%d" % (read, n, read))
        e("v_add_u32 v%d, %%[area], v%d" % (read, read))
        for i in range(4):
            e("v_xor_b32 v%d, %d, v%d" % (slot[i], 64 * i, read))
        e("v_mul_lo_u32 v%d, %%[rowbytes], v%d" % (out, n))
        e("v_lshl_add_u32 v%d, v%d, 4, v%d" % (out, wait, out))
        e("s_lshl_b32 %[t0], %[rowbytes], 2")
        step = 0
        for c in range(2):
            for tensor, regs, scaled in self.outputs():
                for part in range(2):
                    for d2 in range(2):
                        for j in range(4):
                            value = values + 4 * (4 * d2 + j)
                            for i in range(4):
                                e("v_accvgpr_read_b32 v%d, a%d" %
                                  (value + i, regs[c][2 * part + d2] + 4 * j + i))
                            if scaled:
                                for i in range(4):
                                    e("v_mul_f32 v%d, %%[scale], v%d" % (value + i, value + i))
                            e("v_xor_b32 v%d, %d, v%d" % (wait, 16 * (8 * d2 + 2 * j), write))
                            e("ds_write_b128 v%d, %s" % (wait, vt(value, 4)))
                    row = rows[step % 2]
                    e("s_waitcnt lgkmcnt(0)")
                    for i in range(8):
                        e("ds_read_b128 %s, v%d offset:%d" % (vt(row + 4 * i, 4), slot[i % 4], 1024 * i))
                    e("s_waitcnt lgkmcnt(0)")
                    e("v_mov_b32 v%d, v%d" % (wait, out))
                    for i in range(8):
                        e("buffer_store_dwordx4 %s, v%d, %%[%srsrc], 0 offen offset:%d" %
                          (vt(row + 4 * i, 4), wait, tensor, 256 * part))
                        if i < 7:
                            e("v_add_u32 v%d, %%[t0], v%d" % (wait, wait))
                    step += 1
            e("s_lshl_b32 %[t1], %[rowbytes], 5")
            e("v_add_u32 v%d, %%[t1], v%d" % (out, out))
        e("s_waitcnt vmcnt(0)")

    def build(self):
        r = self.r
        e = self.emit
        e("s_mov_b32 %[m0save], m0")
        e("s_waitcnt lgkmcnt(0)")
        for stage in range(RING - 2):
            for group in self.fill_groups(stage):
                for text in group:
                    e(text)
        for i in range(256):
            e("v_accvgpr_write_b32 a%d, 0" % i)
        e("v_mov_b32 v%d, 0xf149f2ca" % r.NEG)      # -1e30: 2^(that * scale) is zero
        e("s_waitcnt vmcnt(%d)" % (FILL_OPS * (RING - 2)))  # K and V
        idle, start, top, masked, after, finish = ("Lidle_%=", "Lstart_%=", "Ltop_%=", "Lmasked_%=",
                                                   "Lafter_%=", "Lfinish_%=")
        e("%s:" % idle)
        e("s_cmp_eq_u32 %[idle], 0")
        e("s_cbranch_scc1 %s" % start)
        self.whole_step()
        e("s_sub_u32 %[idle], %[idle], 1")
        e("s_branch %s" % idle)
        e("%s:" % start)
        e("s_cmp_eq_u32 %[nblk], 0")
        e("s_cbranch_scc1 %s" % finish)
        e("s_mov_b32 %[bcount], 0")
        self.whole_step()
        for _, items in self.rows_of_next():
            for text, dest in items:
                self.lds_read(text, dest)
        at_top = list(self.lds_queue)
        e("%s:" % top)
        e("s_cmp_le_u32 %[bcount], 1")
        e("s_cbranch_scc1 %s" % masked)
        e("s_add_u32 %[t0], %[bcount], 1")
        e("s_cmp_eq_u32 %[t0], %[nblk]")
        e("s_cbranch_scc1 %s" % masked)
        self.block(False)
        assert self.lds_queue == at_top, (self.lds_queue, at_top)
        e("s_branch %s" % after)
        e("%s:" % masked)
        self.lds_queue = list(at_top)
        self.block(True)
        assert self.lds_queue == at_top
        e("%s:" % after)
        e("s_add_u32 %[bcount], %[bcount], 1")
        e("s_cmp_lt_u32 %[bcount], %[nblk]")
        e("s_cbranch_scc1 %s" % top)
        e("%s:" % finish)
        # requests beyond the last block are still on their way into LDS
        e("s_waitcnt vmcnt(0) lgkmcnt(0)")
        e("s_nop 15")
        e("s_nop 15")
        e("s_barrier")
        self.store()
        e("s_mov_b32 m0, %[m0save]")


def render():
    g = Emitter()
    g.build()
    r = g.r
    name = "FLASH_DKV_D128"
    out = ["// heads of 128 channels, two waves a workgroup: %d instructions and labels" % len(g.lines)]
    out.append("#define %s_ASM \\" % name)
    out.append(" \\\n".join(c_string(g.lines).split("\n")))
    out.append("")

    def define(tag, value):
        out.append("#define %s_%s %s" % (name, tag, value))

    define("KEYS_VALUES(kf, vf)", ", ".join(
        '"+{%s}"(%s[%d][%d])' % (vt(regs[c][ks], 4), tensor, c, ks)
        for tensor, regs in (("kf", r.KF), ("vf", r.VF)) for c in range(2) for ks in range(KS)))
    define("ADDRESSES(row_read, tr_read, stat_read)", ", ".join(
        ['"+{v%d}"(row_read[%d])' % (v, i) for i, v in enumerate(r.ROWADDR)] +
        ['"+{v%d}"(tr_read[%d])' % (v, i) for i, v in enumerate(r.TRADDR)] +
        ['"+{v%d}"(stat_read)' % r.STATADDR]))
    define("FILLS(q_fill, g_fill, s_fill)", ", ".join(
        ['"{v%d}"(q_fill[%d])' % (v, i) for i, v in enumerate(r.QFILL)] +
        ['"{v%d}"(g_fill[%d])' % (v, i) for i, v in enumerate(r.GFILL)] +
        ['"{v%d}"(s_fill)' % r.SFILL]))
    define("BOUNDS(first, last)", '"{v%d}"(first), "{v%d}"(last)' % (r.N4, r.TL4))
    clobbers = ['"v%d"' % v for v in range(r.moved_end, r.temps_end)]
    clobbers += ['"v%d"' % v for v in range(192, 256)]
    clobbers += ['"a%d"' % a for a in range(256)]
    define("CLOBBERS", ", ".join(clobbers) + ', "vcc", "scc", "memory"')
    define("RING", str(RING))
    define("STAGE_BYTES", str(STAGE_BYTES))
    define("TILE_BYTES", str(TILE_BYTES))
    return "\n".join(out) + "\n"


def main():
    here = os.path.dirname(os.path.abspath(__file__))
    target = sys.argv[1] if len(sys.argv) > 1 else os.path.join(here, "flash_dkv_loop128.inc")
    text = ("// Generated by gen_flash_dkv_loop128.py; do not edit.  The instruction stream of the\n"
            "// main loop of flash_dkv_wide128_kernel, see the generator for the schedule.\n\n")
    text += render()
    with open(target, "w") as f:
        f.write(text)


if __name__ == "__main__":
    main()
