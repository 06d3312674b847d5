#!/usr/bin/env python3
"""Writes flash_dq_loop128.inc: the hand-scheduled gfx950 instruction stream of
the query-owned attention backward kernel for heads of 128 channels
(flash_dq_wide.hip), the body of one `asm volatile` statement with a fixed register
allocation.

A wave owns 64 queries (two halves of 32, lane = query) and walks the key blocks of
32 rows that they see in ascending order, so that every A operand read from LDS
feeds two matrix instructions.  Q, dO and the accumulators fill the AGPRs.  Per block b,
48 matrix instructions, each followed by what one of them (32 cycles) hides:

  instructions   matrix                  vector
  0 .. 15        S^T(b) = K Q^T          packing of dS(b - 1)
  16 .. 31       dP^T(b) = V dO^T        P(b) = 2^(S scale log2 e - lse)
  32 .. 47       dQ^T += K^T dS^T(b - 1) the rest of P(b), dS(b) = P dP

dP starts from -delta, which stands in registers for the first product's C operand.
The 24 A operands of a block pass through a ring of eight register groups, each
refilled from LDS as soon as its second product is on its way (seven pairs, 448
cycles, before its next use).

Key blocks travel global -> LDS through a ring of five stages (their keys are read
again a block later, transposed); the barrier of step b stands before instruction 32
of block b - 1, and block b + 2 is requested behind it, into the stage of block b - 3.

The last two blocks of a wave (the causal diagonal crosses them) and its first run a
variant that compares every element's key with a per-lane bound.

Usage: python gen_flash_dq_loop128.py [output]   (default: flash_dq_loop128.inc
beside this file)
"""
import os
import sys

import gen_flash_dkv_loop128 as dkv
from gen_flash_dkv_loop import MFMA, at_, c_string, vt

D, KS, DB = dkv.D, dkv.KS, dkv.DB
RING = 5
POOL = 8
TILE_BYTES = dkv.TILE_BYTES
STAGE_BYTES = 2 * TILE_BYTES
ROW_BYTES = dkv.ROW_BYTES
FILL_OPS = 8            # vector-memory operations a wave and stage: 4 K, 4 V
AHEAD = 2               # a block is requested this many steps before its rows are read
weight = dkv.weight


class Registers:
    def __init__(self):
        at = 4          # v0 .. v3 stay with the compiler

        def take(n=1):
            nonlocal at
            first = at
            at += n
            return first
        self.FILL = [take(), take()]                    # K and V rows share their stride
        self.LSE = [take(), take()]                     # minus the scaled log2-sum-exp
        self.DELTA = [take(), take()]                   # minus delta
        self.BOUND = take()
        self.inputs_end = at
        self.ROWADDR = [take() for _ in range(4)]
        self.TRADDR = [take() for _ in range(2)]
        self.moved_end = at
        self.FTMP = [take(), take()]
        self.LIM = [take(), take()]
        self.NEG = take()
        at = 24
        self.DS = [[take(4) for _ in range(2)] for _ in range(2)]   # [c][s2], packed
        self.OPS = [take(4) for _ in range(POOL)]
        self.DELTAS = [take(16), take(16)]
        self.temps_end = at
        assert at <= 128
        # v128 .. v255 bring Q and dO in
        self.QIN = [[128 + 4 * (KS * c + ks) for ks in range(KS)] for c in range(2)]
        self.GIN = [[192 + 4 * (KS * c + ks) for ks in range(KS)] for c in range(2)]
        self.S = [128, 144]
        self.DP = [160, 176]
        # AGPRs
        self.DQ = [[16 * (DB * c + db) for db in range(DB)] for c in range(2)]
        self.QF = [[128 + 4 * (KS * c + ks) for ks in range(KS)] for c in range(2)]
        self.GF = [[192 + 4 * (KS * c + ks) for ks in range(KS)] for c in range(2)]


class Emitter(dkv.Emitter):
    def __init__(self):
        self.r = Registers()
        self.lines = []
        self.lds_queue = []

    def outputs(self):
        return (("dq", self.r.DQ, True),)

    def operand_reads(self, pair):
        """Rows of K, rows of V, then K^T of the block before."""
        r = self.r
        reg = r.OPS[pair % POOL]
        if pair < 16:
            tensor, ks = divmod(pair, 8)
            return [("ds_read_b128 %s, v%d offset:%d" %
                     (vt(reg, 4), r.ROWADDR[ks % 4], tensor * TILE_BYTES + ks // 4 * 128), ("op", pair))]
        s2, db = divmod(pair - 16, DB)
        return [("ds_read_b64_tr_b16 %s, v%d offset:%d" %
                 (vt(reg + 2 * part, 2), r.TRADDR[db % 2],
                  (16 * s2 + 8 * part) * ROW_BYTES + db // 2 * 128), ("op", pair))
                for part in range(2)]

    def products(self):
        r = self.r
        out = []
        for tensor, (acc, frags) in enumerate(((r.S, r.QF), (r.DP, r.GF))):
            for ks in range(KS):
                pair = 8 * tensor + ks
                for c in range(2):
                    own = vt(acc[c], 16)
                    start = own if ks else ("0" if tensor == 0 else vt(r.DELTAS[c], 16))
                    out.append(([("op", pair)], "%s %s, %s, %s, %s" %
                                (MFMA, own, vt(r.OPS[pair % POOL], 4), at_(frags[c][ks], 4), start)))
        for s2 in range(2):
            for db in range(DB):
                pair = 16 + DB * s2 + db
                for c in range(2):
                    acc = at_(r.DQ[c][db], 16)
                    out.append(([("op", pair)], "%s %s, %s, %s, %s" %
                                (MFMA, acc, vt(r.OPS[pair % POOL], 4), vt(r.DS[c][s2], 4), acc)))
        assert len(out) == 48
        return out

    # ---- vector side: four elements at a time, accumulator registers 0-7 of both halves first ----
    def groups(self):
        return [(c, first) for s2 in range(2) for c in range(2) for first in (8 * s2, 8 * s2 + 4)]

    def probabilities(self, masked):
        r = self.r
        out = []
        for c, first in self.groups():
            S = r.S[c]
            group = range(first, first + 4)
            if masked:
                for i in group:
                    out.append("v_cmp_le_i32 vcc, %d, v%d" % (8 * (i // 4) + i % 4, r.LIM[c]))
                    out.append("v_cndmask_b32 v%d, v%d, v%d, vcc" % (S + i, r.NEG, S + i))
            out += ["v_fma_f32 v%d, v%d, %%[scale2], v%d" % (S + i, S + i, r.LSE[c]) for i in group]
            out += ["v_exp_f32 v%d, v%d" % (S + i, S + i) for i in group]
        return out

    def score_gradients(self):
        r = self.r
        return ["v_mul_f32 v%d, v%d, v%d" % (r.DP[c] + i, r.S[c] + i, r.DP[c] + i)
                for c, first in self.groups() for i in range(first, first + 4)]

    def packs(self):
        r = self.r
        return ["v_cvt_pk_bf16_f32 v%d, v%d, v%d" %
                (r.DS[c][s2] + w, r.DP[c] + 8 * s2 + 2 * w, r.DP[c] + 8 * s2 + 2 * w + 1)
                for s2 in range(2) for c in range(2) for w in range(4)]

    def vector_gaps(self, masked, owed):
        """The instruction after which each vector item stands.  Results of matrix
        instruction i are read from gap i + 2 on, operands written before gap i - 1."""
        gaps = [[] for _ in range(48)]
        if owed:
            self.spread(gaps, self.packs(), 1, 8)
        exps, muls = self.probabilities(masked), self.score_gradients()
        share = -(-sum(weight(t) for t in exps + muls) // 30)   # of gaps 17 .. 46
        finished = set()    # registers that hold P

        def take_exp():
            text = exps.pop(0)
            if text.startswith("v_exp"):
                finished.add(text.split()[1])
            return text

        for g in range(17, 33):
            taken = 0
            while exps and taken < share:
                taken += weight(exps[0])
                gaps[g].append(take_exp())
        rest, credit, ratio = [], 0.0, len(muls) / len(exps)
        while exps:         # the muls among the remaining exps, never ahead of their P
            rest.append(take_exp())
            credit += ratio
            while credit >= 1 and muls[0].split()[2] in finished and not rest[-1].startswith("v_exp"):
                rest.append(muls.pop(0))
                credit -= 1
        self.spread(gaps, rest + muls, 33, 46)
        return gaps

    # ---- stages -------------------------------------------------------------------------------------
    def barrier(self):
        """Step s: block s has landed for every wave, everyone is done with block s - 3,
        whose stage takes block s + 2."""
        self.emit("s_waitcnt vmcnt(%d)" % (FILL_OPS * (AHEAD - 1)))
        self.emit("s_barrier")

    def move(self, stage, registers):
        return ["s_add_u32 %%[%s], %%[%s], %d" % (stage, stage, STAGE_BYTES),
                "s_mov_b32 %%[t0], %d" % STAGE_BYTES,
                "s_cmp_eq_u32 %%[%s], %d" % (stage, RING * STAGE_BYTES),
                "s_cselect_b32 %%[t0], %d, %%[t0]" % (-(RING - 1) * STAGE_BYTES),
                "s_cselect_b32 %%[%s], 0, %%[%s]" % (stage, stage)] + \
               ["v_add_u32 v%d, %%[t0], v%d" % (v, v) for v in registers]

    def advance(self):
        return self.move("rstage", self.r.ROWADDR)

    def fill_groups(self, stage=None):
        """The requests of the next block into the fill stage, one list a vector-memory
        instruction (see gen_flash_dkv_loop128.py)."""
        r = self.r
        groups = []
        for tensor, name in enumerate("kv"):
            for pair in range(2):
                setup = []
                if pair == 0:
                    setup.append("s_add_u32 m0, %[ldsq], %[fstage]" if tensor == 0 else
                                 "s_add_u32 m0, m0, %d" % TILE_BYTES)
                    source = "%[koff]"
                else:
                    setup.append("s_add_u32 %[t0], %[koff], %[keight]")
                    source = "%[t0]"
                setup += ["v_add_u32 v%d, %s, v%d" % (r.FTMP[i], source, r.FILL[i]) for i in range(2)]
                for i in range(2):
                    groups.append((setup if i == 0 else []) +
                                  ["buffer_load_dwordx4 v%d, %%[%srsrc], 0 offen offset:%d lds" %
                                   (r.FTMP[i], name, 1024 * (2 * pair + i))])
        groups[-1] += ["s_add_u32 %[koff], %[koff], %[kstep]",
                       "s_add_u32 %%[fstage], %%[fstage], %d" % STAGE_BYTES,
                       "s_cmp_eq_u32 %%[fstage], %d" % (RING * STAGE_BYTES),
                       "s_cselect_b32 %[fstage], 0, %[fstage]"]
        assert len(groups) == FILL_OPS
        return groups

    def whole_step(self):
        self.barrier()
        for text in self.advance():
            self.emit(text)
        for group in self.fill_groups():
            for text in group:
                self.emit(text)

    # ---- one block ---------------------------------------------------------------------------------
    def rows_of_next(self):
        return [(33 + 2 * k, self.operand_reads(k)) for k in range(8)]

    def bounds(self):
        """Hidden where the key's place in the block exceeds LIM."""
        r = self.r
        self.emit("s_lshl_b32 %[t0], %[bcount], 5")
        self.emit("v_subrev_u32 v%d, %%[t0], v%d" % (r.LIM[0], r.BOUND))
        self.emit("v_add_u32 v%d, 32, v%d" % (r.LIM[1], r.LIM[0]))

    def block(self, masked, owed=True):
        """owed: the block before still owes its dQ."""
        if masked:
            self.bounds()
        reads = [[] for _ in range(48)]
        for pair in range(8, 24 if owed else 16):
            reads[2 * (pair - 8) + 1] += self.operand_reads(pair)
        for gap, items in self.rows_of_next():
            reads[gap] += items
        other = [[] for _ in range(48)]
        other[32] += self.advance()
        if owed:        # the transposed reads of the block before are out
            other[32] += self.move("tstage", self.r.TRADDR)
        for i, group in enumerate(self.fill_groups()):
            other[34 + i] += group
        vector = self.vector_gaps(masked, owed)
        for g, (needs, text) in enumerate(self.products()):
            if g == 32:
                self.barrier()
            if g < 32 or owed:
                for need in needs:
                    self.wait_for(need)
                self.emit(text)
            elif g == 32:
                self.emit("s_nop 15")       # dP, with no product in between
                self.emit("s_nop 15")
            for item in other[g]:
                self.emit(item)
            for item, dest in reads[g]:
                self.lds_read(item, dest)
            for item in vector[g]:
                self.emit(item)

    def drain(self):
        """dQ of the last block; the row reads of the block after it are dropped."""
        e = self.emit
        self.lds_queue = []
        e("s_waitcnt lgkmcnt(0)")
        for pair in range(16, 24):
            for text, dest in self.operand_reads(pair):
                self.lds_read(text, dest)
        for text in self.packs():
            e(text)
        e("s_nop 7")
        for needs, text in self.products()[32:]:
            for need in needs:
                self.wait_for(need)
            e(text)

    def build(self):
        r = self.r
        e = self.emit
        e("s_mov_b32 %[m0save], m0")
        e("s_waitcnt vmcnt(0) lgkmcnt(0)")
        for _ in range(AHEAD):
            for group in self.fill_groups():
                for text in group:
                    e(text)
        for regs, agprs in ((r.QIN, r.QF), (r.GIN, r.GF)):
            for c in range(2):
                for ks in range(KS):
                    for i in range(4):
                        e("v_accvgpr_write_b32 a%d, v%d" % (agprs[c][ks] + i, regs[c][ks] + i))
        for i in range(128):
            e("v_accvgpr_write_b32 a%d, 0" % i)
        for c in range(2):
            for i in range(16):
                e("v_mov_b32 v%d, v%d" % (r.DELTAS[c] + i, r.DELTA[c]))
        e("v_mov_b32 v%d, 0xf149f2ca" % r.NEG)      # -1e30: 2^(that * scale) is zero
        top, masked, after, drain, idle, finish = ("Ltop_%=", "Lmasked_%=", "Lafter_%=", "Ldrain_%=",
                                                   "Lidle_%=", "Lfinish_%=")
        e("s_cmp_eq_u32 %[nblk], 0")
        e("s_cbranch_scc1 %s" % idle)
        e("s_mov_b32 %[bcount], 0")
        self.whole_step()
        for _, items in self.rows_of_next():
            for text, dest in items:
                self.lds_read(text, dest)
        at_top = list(self.lds_queue)
        self.block(True, owed=False)
        assert self.lds_queue == at_top
        e("s_mov_b32 %[bcount], 1")
        e("%s:" % top)
        e("s_cmp_eq_u32 %[bcount], %[nblk]")
        e("s_cbranch_scc1 %s" % drain)
        e("s_cmp_ge_u32 %[bcount], %[diagonal]")
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
        e("s_branch %s" % top)
        e("%s:" % drain)
        self.drain()
        # the steps that the workgroup's other wave still has
        e("%s:" % idle)
        e("s_cmp_eq_u32 %[idle], 0")
        e("s_cbranch_scc1 %s" % finish)
        self.whole_step()
        e("s_sub_u32 %[idle], %[idle], 1")
        e("s_branch %s" % idle)
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
    name = "FLASH_DQ_D128"
    out = ["// heads of 128 channels, two waves a workgroup: %d instructions and labels" % len(g.lines)]
    out.append("#define %s_ASM \\" % name)
    out.append(" \\\n".join(c_string(g.lines).split("\n")))
    out.append("")

    def define(tag, value):
        out.append("#define %s_%s %s" % (name, tag, value))

    define("ROWS(qf, gf)", ", ".join(
        '"+{%s}"(%s[%d][%d])' % (vt(regs[c][ks], 4), tensor, c, ks)
        for tensor, regs in (("qf", r.QIN), ("gf", r.GIN)) for c in range(2) for ks in range(KS)))
    define("ADDRESSES(row_read, tr_read)", ", ".join(
        ['"+{v%d}"(row_read[%d])' % (v, i) for i, v in enumerate(r.ROWADDR)] +
        ['"+{v%d}"(tr_read[%d])' % (v, i) for i, v in enumerate(r.TRADDR)]))
    define("LANES(fill, lse, delta, bound)", ", ".join(
        '"{v%d}"(%s[%d])' % (regs[i], tensor, i)
        for tensor, regs in (("fill", r.FILL), ("lse", r.LSE), ("delta", r.DELTA)) for i in range(2)) +
        ', "{v%d}"(bound)' % r.BOUND)
    clobbers = ['"v%d"' % v for v in range(r.moved_end, 128)]
    clobbers += ['"a%d"' % a for a in range(256)]
    define("CLOBBERS", ", ".join(clobbers) + ', "vcc", "scc", "memory"')
    define("RING", str(RING))
    define("STAGE_BYTES", str(STAGE_BYTES))
    define("TILE_BYTES", str(TILE_BYTES))
    return "\n".join(out) + "\n"


def main():
    here = os.path.dirname(os.path.abspath(__file__))
    target = sys.argv[1] if len(sys.argv) > 1 else os.path.join(here, "flash_dq_loop128.inc")
    text = ("// Generated by gen_flash_dq_loop128.py; do not edit.  The instruction stream of the\n"
            "// main loop of flash_dq_wide_kernel, see the generator for the schedule.\n\n")
    text += render()
    with open(target, "w") as f:
        f.write(text)


if __name__ == "__main__":
    main()
