"""Writes the main loops of the one-wavefront-per-SIMD attention kernels as assembly (``attn_loops.inc``).

The kernels around them (``attn_bwd_dkv128.h``) are HIP; only the loop is laid down instruction by instruction, because with
one wavefront on a SIMD the order of its instructions IS the schedule: a ``16x16x32`` MFMA occupies the matrix pipe for 16 cycles,
a wavefront issues one instruction in about 5, so two or three others fit beneath each MFMA for free and anything that stands
in the wrong place is paid in full.  (Written as single asm statements the compiler puts an ``s_nop`` between any two of which one
reads what the other wrote, 74 in a tile of 128 MFMAs: 10 % of the loop.)

``Stream`` keeps the account of the loops' LDS reads, MFMAs and vector instructions (``lds``, ``mfma``, ``valu``): it counts reads in
flight (they complete in order) and places the waits, and it refuses
  * an MFMA or vector instruction that reads a register whose LDS read nothing has waited for,
  * a vector instruction on the result of an MFMA with fewer than two MFMAs between them,
  * an MFMA on a register that a vector instruction wrote fewer than two instructions ago,
  * the result of a transcendental in the very next instruction,
  * an LDS read into a register that an earlier read has not filled yet,
  * an MFMA on a fragment that a later read has replaced.
What goes out through ``put`` (masks, the moving reference, the code in front of and behind the loops) is not looked at and waits by
``s_nop``.  Which stage of LDS a copy may fill is no matter of registers: ``tests/test_build_checks.py`` runs the finished text and
checks that no copy goes to a stage that is still read, and no read to one that has not landed.
"""
import re
import sys


def regs(text, kind="v"):
    """The registers of one kind that an operand list names by number, as a set."""
    out = set()
    for lo, hi in re.findall(r"(?<![\w\]])%s\[(\d+):(\d+)\]" % kind, text):
        out |= set(range(int(lo), int(hi) + 1))
    out |= {int(n) for n in re.findall(r"(?<![\w\[%%])%s(\d+)\b" % kind, text)}
    return out


def v(n, count=1):
    return "v%d" % n if count == 1 else "v[%d:%d]" % (n, n + count - 1)


def s(n, count=1):
    return "s%d" % n if count == 1 else "s[%d:%d]" % (n, n + count - 1)


class Stream:
    """A straight piece of code with its account of what is in flight."""

    def __init__(self, dtype):
        self.mfma_name = "v_mfma_f32_16x16x32_" + {"bf16": "bf16", "f16": "f16"}[dtype]
        self.pack_name = "v_cvt_pk_%s_f32" % dtype
        self.lines = []
        self.reads = []                # LDS reads that may be in flight, oldest first: sets of registers
        self.mfma_at, self.mfmas = {}, 0
        self.valu_at, self.count = {}, 0
        self.holds = {}                # what the last LDS read into a register brought
        self.trans = set()
        self.pad = False               # out of line: waits where it would refuse (MFMAs are left out there)

    def state(self):
        """The account at this point, for a piece of code that is entered from here (``resume``)."""
        return [set(r) for r in self.reads], dict(self.mfma_at), self.mfmas, dict(self.valu_at), self.count, dict(self.holds)

    def resume(self, state):
        reads, mfma_at, self.mfmas, valu_at, self.count, holds = state
        self.reads, self.mfma_at, self.valu_at, self.holds, self.trans = [set(r) for r in reads], dict(mfma_at), dict(valu_at), dict(holds), set()

    def put(self, text):
        self.lines.append(text)
        self.count += 1
        self.trans = set()

    def fresh(self, used):
        for r in self.reads:
            assert not (r & used), ("read in flight", used, self.lines[-3:])

    # -- LDS --
    def lds(self, text, dst, width, what=None):
        d = set(range(dst, dst + width))
        self.holds.update((r, what) for r in d)
        for r in self.reads:
            assert not (r & d), ("two reads in flight into", d)
        self.reads.append(d)
        self.put(text)

    def wait(self, used):
        """Waits for the reads into `used`, if they may be in flight."""
        last = max((i for i, r in enumerate(self.reads) if r & used), default=-1)
        if last >= 0:
            left = len(self.reads) - 1 - last
            self.reads = self.reads[last + 1:]
            self.put("s_waitcnt lgkmcnt(%d)" % min(left, 15))

    # -- matrix and vector --
    def mfma(self, d, x, y, c, holds=()):
        used = regs(x, "v") | regs(y, "v") | regs(c, "v")
        for operand, what in holds:
            for r in regs(operand, "v"):
                assert self.holds.get(r) == what, ("another read came in between", r, what, self.holds.get(r))
        self.fresh(used | regs(d, "v"))
        while self.pad and any(self.count - self.valu_at.get(r, -99) < 3 for r in used):
            self.put("s_nop 0")
        for r in used:
            assert self.count - self.valu_at.get(r, -99) >= 3, ("MFMA too soon behind", r, self.lines[-3:])
        self.put("%s %s, %s, %s, %s" % (self.mfma_name, d, x, y, c))
        self.mfmas += 1
        for r in regs(d, "v"):
            self.mfma_at[r] = self.mfmas

    def valu(self, op, d, *src, trans=False):
        used = set().union(*[regs(x, "v") for x in src])
        self.fresh(used | regs(d, "v"))
        if self.pad and self.trans & used:
            self.put("s_nop 0")
        assert not (self.trans & used), ("behind a transcendental", op, d, src)
        if self.pad and any(self.mfmas - self.mfma_at.get(r, -99) < 2 for r in used | regs(d, "v")):
            self.settle()
        for r in used | regs(d, "v"):
            assert self.mfmas - self.mfma_at.get(r, -99) >= 2, ("too soon behind the MFMA of", r, self.lines[-3:])
        self.put("%s %s" % (op, ", ".join((d,) + src)))
        for r in regs(d, "v"):
            self.valu_at[r] = self.count
        self.trans = regs(d, "v") if trans else set()

    def settle(self):
        """Waits for every MFMA."""
        self.put("s_nop 15")
        self.mfma_at = {}


class DKV:
    """dK/dV: the loop over a wavefront's tiles of 32 query rows, two stages unrolled.

    Steps of four MFMAs (one per block of 16 keys): 0..7 S (k step, row block), 8..15 dP, 16..23 dV (d block), 24..31 dK.
    """
    KEEP = 100                                     # VGPRs below this are the compiler's (operands)
    S, DP, PP, DSP, RING, L4, D4, E = 100, 132, 164, 180, 196, 228, 236, 244
    NEG = 248
    RSQ, RSD, RSL, QSTEP, DSTEP, QWRAP, DWRAP, LWRAP, DSC, DSS, DSTEP_DS, WRAP_DS, T, CTC, PADS = 40, 44, 48, 52, 54, 56, 58, 60, 62, 64, 66, 68, 70, 76, 78
    LOOK = 15                                      # MFMAs between an LDS read and its use
    ROWB, QTB, SLOTB = 256, 8192, 16640

    def __init__(self, dtype, store_ds):
        self.store_ds = store_ds
        self.x = Stream(dtype)
        # K fragments of three k steps lie where dP and P's pairs come to be
        self.fk = [[self.DP + 4 * kb for kb in range(4)], [self.DP + 16 + 4 * kb for kb in range(4)], [self.PP + 4 * kb for kb in range(4)]]
        self.ops = self.tile_reads()

    def ring(self, step):
        return self.RING + 4 * (step % 8)

    def tile_reads(self):
        """LDS reads of a tile in order: (first MFMA that uses it, destination, width, function of the stage's offset)."""
        ops = []
        for step in range(32):
            u, r = 4 * step, self.ring(step)
            if step < 8:
                ks, qb = step // 2, step % 2
                if qb == 0:
                    for kb in range(4):
                        ops.append((u + kb, self.fk[ks % 3][kb], 4, lambda st, d, ks=ks, kb=kb: "ds_read_b128 %s, %%[rk%d] offset:%d" % (v(d, 4), ks, 16 * self.ROWB * kb)))
                        if kb == 0:
                            ops.append((u, r, 4, lambda st, d, ks=ks: "ds_read_b128 %s, %%[rq%d] offset:%d" % (v(d, 4), ks, st)))
                else:
                    ops.append((u, r, 4, lambda st, d, ks=ks: "ds_read_b128 %s, %%[rq%d] offset:%d" % (v(d, 4), ks, st + 16 * self.ROWB)))
            elif step < 16:
                ks, qb = (step - 8) // 2, step % 2
                ops.append((u, r, 4, lambda st, d, ks=ks, qb=qb: "ds_read_b128 %s, %%[rq%d] offset:%d" % (v(d, 4), ks, st + self.QTB + 16 * self.ROWB * qb)))
                if step in (8, 9):
                    ops.append((u, self.D4 + 4 * qb, 4, lambda st, d, qb=qb: "ds_read_b128 %s, %%[ldr] offset:%d" % (v(d, 4), st + 128 + 64 * qb)))
                    ops.append((u, self.L4 + 4 * qb, 4, lambda st, d, qb=qb: "ds_read_b128 %s, %%[ldr] offset:%d" % (v(d, 4), st + 64 * qb)))
            else:
                t, off = step % 8, self.QTB if step < 24 else 0
                for h in range(2):
                    ops.append((u, r + 2 * h, 2, lambda st, d, t=t, off=off, h=h: "ds_read_b64_tr_b16 %s, %%[ta%d] offset:%d" % (v(d, 2), t, st + off + 16 * self.ROWB * h)))
        # the slot behind which each is issued: LOOK MFMAs ahead, one a slot (negative: during the tile before)
        slot, out = -10 ** 9, []
        for use, d, n, f in ops:
            slot = max(slot + 1, use - self.LOOK)
            assert slot < use
            out.append((slot, use, d, n, f))
        return out

    def vector_work(self):
        """Vector instructions behind each MFMA: {slot: [function, ..]}.

        Pair j of P and of dS: rows 2 (j % 2) .. of row block (j / 2) % 2, key block j / 4."""
        x, work = self.x, {}

        def at(j):
            kb, qb, e = j >> 2, (j >> 1) & 1, 2 * (j & 1)
            return kb, qb, e, self.S + 4 * (4 * qb + kb) + e, self.DP + 4 * (4 * qb + kb) + e

        def p_fma(j):
            kb, qb, e, p, _ = at(j)
            for i in range(2):
                x.valu("v_fma_f32", v(p + i), v(p + i), "%[scale]", "-" + v(self.L4 + 4 * qb + e + i))

        def p_exp(j):
            p = at(j)[3]
            for i in range(2):
                x.valu("v_exp_f32", v(p + i), v(p + i), trans=True)

        def p_pack(j):
            p = at(j)[3]
            x.valu(x.pack_name, v(self.PP + 4 * (j >> 2) + (j & 3)), v(p), v(p + 1))

        def ds_mul(j):
            _, _, _, p, d = at(j)
            for i in range(2):
                x.valu("v_mul_f32", v(p + i), v(p + i), v(d + i))

        def ds_pack(j):
            p = at(j)[3]
            x.valu(x.pack_name, v(self.DSP + 4 * (j >> 2) + (j & 3)), v(p), v(p + 1))

        def put(slot, f, j):
            work.setdefault(slot, []).append(lambda: f(j))
        # P beneath dP (MFMAs 32..63) and the first of dV, dS beneath the rest of dV
        for j in range(16):
            base = 33 + 29 * j // 15
            put(base, p_fma, j)
            put(base + 1, p_exp, j)
            put(base + 2, p_pack, j)
            base = 68 + 26 * j // 16
            put(base, ds_mul, j)
            put(base + 1, ds_pack, j)
        return work

    def advance(self):
        """To the tile that is copied next, as pieces of scalar code: its rows (a descriptor of no bytes behind the last tile)."""
        R = self
        out = [["s_mov_b32 s%d, %%[ct]" % R.CTC, "s_add_u32 %[ct], %[ct], 4"]]
        if self.store_ds:
            out += [["s_mov_b64 %s, %s" % (s(R.DSS, 2), s(R.DSC, 2))], ["s_add_u32 %s, %s, %s" % (s(R.DSC), s(R.DSC), s(R.DSTEP_DS)), "s_addc_u32 %s, %s, %s" % (s(R.DSC + 1), s(R.DSC + 1), s(R.DSTEP_DS + 1))]]
        for p, st in ((R.RSQ, R.QSTEP), (R.RSD, R.DSTEP)):
            out.append(["s_add_u32 %s, %s, %s" % (s(p), s(p), s(st)), "s_addc_u32 %s, %s, %s" % (s(p + 1), s(p + 1), s(st + 1))])
        out.append(["s_add_u32 %s, %s, 0x200" % (s(R.RSL), s(R.RSL)), "s_addc_u32 %s, %s, 0" % (s(R.RSL + 1), s(R.RSL + 1))])
        out.append(["s_cmp_ge_i32 %[ct], %[ntq]", "s_cbranch_scc1 WRAP{0}", "BACK{0}:"])
        t = s(R.T)
        out.append(["s_lshl_b32 %s, %%[ct], 5" % t, "s_sub_i32 %s, %%[rows], %s" % (t, t)])
        out.append(["s_min_i32 %s, %s, 32" % (t, t), "s_sub_i32 %s, %s, 1" % (t, t)])
        out.append(["s_mul_i32 %s, %s, %%[qrowb]" % (s(R.RSQ + 2), t), "s_mul_i32 %s, %s, %%[drowb]" % (s(R.RSD + 2), t)])
        out.append(["s_add_u32 %s, %s, 0x100" % (s(R.RSQ + 2), s(R.RSQ + 2)), "s_add_u32 %s, %s, 0x100" % (s(R.RSD + 2), s(R.RSD + 2))])
        out.append(["s_cmp_gt_i32 %[rem], 1"] + ["s_cselect_b32 %s, %s, 0" % (s(r + 2), s(r + 2)) for r in (R.RSQ, R.RSD)] +
                   ["s_cselect_b32 %s, %%[ldbytes], 0" % s(R.RSL + 2)])
        return out

    def wrap(self, i):
        """Out of line: the copied tile is past the head's last one; the same tile of the next head."""
        R = self
        self.label("WRAP%d" % i)
        pairs = [(R.RSQ, R.QWRAP), (R.RSD, R.DWRAP), (R.RSL, R.LWRAP)] + ([(R.DSC, R.WRAP_DS)] if self.store_ds else [])
        for p, w in pairs:
            self.x.put("s_add_u32 %s, %s, %s" % (s(p), s(p), s(w)))
            self.x.put("s_addc_u32 %s, %s, %s" % (s(p + 1), s(p + 1), s(w + 1)))
        self.x.put("s_sub_u32 %[ct], %[ct], %[ntq]")
        self.x.put("s_cmp_ge_i32 %[ct], %[ntq]")
        self.x.put("s_cbranch_scc1 %s" % self.ref("WRAP%d" % i))
        self.x.put("s_branch %s" % self.ref("BACK%d" % i))

    def ref(self, name):
        return "L%s_%%=" % name

    def label(self, name):
        self.x.lines.append(self.ref(name) + ":")

    def scalar(self, piece, i):
        for line in piece:
            if line == "BACK{0}:":
                self.label("BACK%d" % i)
            elif "WRAP{0}" in line:
                self.x.put("s_cbranch_scc1 %s" % self.ref("WRAP%d" % i))
            else:
                self.x.put(line)

    def mask(self, i):
        """Out of line: scores past the diagonal and, where dS is kept, of keys past the end become -inf.  So do those of rows past the
        end: their Q is 0, but a key that no row sees may hold what 0 times it is none (keys that some row sees lie in other tiles too, and
        made dQ of that row none there).  The first tile of a causal one has 32 keys that no row of it sees: no products of theirs."""
        x = self.x
        self.label("MASK%d" % i)
        x.put("s_nop 15")
        x.put("s_nop 7")
        diag, rows = v(self.E), v(self.E + 1)
        x.put("v_mov_b32 %s, 0xff800000" % v(self.NEG))
        if self.store_ds:
            x.put("s_cmp_eq_u32 %[dsmask], 0")
            x.put("s_cbranch_scc1 %s" % self.ref("KEYS%d" % i))
            for kb in range(4):
                x.put("v_cmp_le_i32 vcc, %d, %%[vy]" % (-16 * kb))
                x.put("s_nop 1")
                for qb in range(2):
                    for e in range(4):
                        r = v(self.S + 4 * (4 * qb + kb) + e)
                        x.put("v_cndmask_b32 %s, %s, %s, vcc" % (r, r, v(self.NEG)))
            self.label("KEYS%d" % i)
            x.put("s_cmp_ge_i32 %s, %%[mct]" % s(self.CTC))
            x.put("s_cbranch_scc1 %s" % self.ref("MASKED%d" % i))
        x.put("s_lshl_b32 %s, %s, 5" % (s(self.T), s(self.CTC)))
        x.put("v_subrev_u32 %s, %s, %%[vx]" % (diag, s(self.T)))
        for qb in range(2):
            for kb in range(4):
                for e in range(4):
                    r = v(self.S + 4 * (4 * qb + kb) + e)
                    x.put("v_cmp_lt_i32 vcc, %d, %s" % (16 * qb + e - 16 * kb, diag))
                    x.put("s_nop 1")
                    x.put("v_cndmask_b32 %s, %s, %s, vcc" % (r, r, v(self.NEG)))
        x.put("s_cmp_lg_u32 %s, %%[pct]" % s(self.CTC))
        x.put("s_cbranch_scc1 %s" % self.ref("WHOLE%d" % i))
        x.put("v_add_u32 %s, %s, %%[vz]" % (rows, s(self.T)))
        for qb in range(2):
            if qb:
                x.put("v_add_u32 %s, 16, %s" % (rows, rows))
            for e in range(4):
                x.put("v_cmp_le_i32 %s, %d, %s" % (s(self.PADS + 2 * e, 2), -e, rows))
            x.put("s_nop 1")
            for kb in range(4):
                for e in range(4):
                    r = v(self.S + 4 * (4 * qb + kb) + e)
                    x.put("v_cndmask_b32 %s, %s, %s, %s" % (r, r, v(self.NEG), s(self.PADS + 2 * e, 2)))
        self.label("WHOLE%d" % i)
        x.put("s_cmp_lg_u32 %s, 0" % s(self.CTC))
        x.put("s_cbranch_scc1 %s" % self.ref("MASKED%d" % i))
        x.pad = True
        x.resume(self.masked_from[i])
        self.piece(i, 32, 128, (2, 3))
        x.pad = False
        x.put("s_branch %s" % self.ref("DONE%d" % i))

    def tile(self, stage):
        x = self.x
        self.piece(stage, 0, 32)
        x.put("s_cbranch_vccnz %s" % self.ref("MASK%d" % stage))      # scores to mask
        self.label("MASKED%d" % stage)
        self.masked_from[stage] = x.state()
        self.piece(stage, 32, 128)
        self.label("DONE%d" % stage)

    def piece(self, stage, first, end, without=()):
        """MFMAs `first` to `end` of a tile and what goes with them; dV and dK of the key blocks `without` get nothing."""
        x, st, nx = self.x, self.SLOTB * stage, self.SLOTB * (1 - stage)
        issue = {}
        for slot, use, d, n, f in self.ops:
            if slot >= 0:
                issue.setdefault(slot, []).append((f(st, d), d, n, use // 4))
        for slot, use, d, n, f in self.ops:          # the next tile's first ones
            if slot < 0:
                issue.setdefault(128 + slot, []).append((f(nx, d), d, n, use // 4))
        first_ahead = 128 + min(o[0] for o in self.ops)
        work = self.vector_work()
        copies = [("q", i) for i in range(8)] + [("d", i) for i in range(8)] + [("l", 0)]
        adv = self.advance()
        adv_at = {97 + i: p for i, p in enumerate(adv)}
        assert 97 + len(adv) <= first_ahead + 16
        nstores = 8 if self.store_ds else 0
        for m in range(first, end):
            step, kb = m // 4, m % 4
            r = self.ring(step)
            copy = copies[m // 2 + (m == 31)] if m < 32 and (m % 2 == 0 or m == 31) and m // 2 + (m == 31) < 17 else None
            if copy:
                c, i = copy
                x.put("s_add_u32 m0, %%[wbase], %d" % (nx + {"q": 1024 * i, "d": self.QTB + 1024 * i, "l": 2 * self.QTB}[c]))
            if m == first_ahead:
                x.put("s_waitcnt vmcnt(%d)" % nstores)         # the next tile has landed
            frag = v(r, 4)
            if step < 8:
                ks, qb = step // 2, step % 2
                d, y = self.S + 4 * (4 * qb + kb), v(self.fk[ks % 3][kb], 4)
                need = set(range(r, r + 4)) | regs(y, "v")
                c = "0" if ks == 0 else v(d, 4)
                out = v(d, 4)
            elif step < 16:
                ks, qb = (step - 8) // 2, step % 2
                d, y = self.DP + 4 * (4 * qb + kb), "%%[V%d%d]" % (kb, ks)
                need = set(range(r, r + 4)) | (set(range(self.D4 + 4 * qb, self.D4 + 4 * qb + 4)) if ks == 0 else set())
                c = v(self.D4 + 4 * qb, 4) if ks == 0 else v(d, 4)
                out = v(d, 4)
            else:
                t = step % 8
                out = c = "%%[%s%d%d]" % ("dv" if step < 24 else "dk", kb, t)
                y = v((self.PP if step < 24 else self.DSP) + 4 * kb, 4)
                need = set(range(r, r + 4))
            if kb == 0 and step % 2 == 0:                      # one wait for two steps where the later reads are old enough
                later = self.ring(step + 1) if step < 31 else None
                if later is not None:
                    need |= set(range(later, later + 4))
                if step < 8:
                    need |= set(range(self.fk[(step // 2) % 3][0], self.fk[(step // 2) % 3][0] + 16))
                if step == 8:
                    need |= set(range(self.L4, self.L4 + 8)) | set(range(self.D4, self.D4 + 8))
            x.wait(need)
            if step < 16 or kb not in without:
                x.mfma(out, frag, y, c, [(frag, step)] + ([(y, step & ~1)] if step < 8 else []) + ([(c, step)] if step in (8, 9) else []))
            if copy:
                c, i = copy
                if c == "l":
                    x.put("buffer_load_dword %%[cld], %s, 0 offen lds" % s(self.RSL, 4))
                else:
                    x.put("buffer_load_dwordx4 %%[c%s%d], %s, %s offen lds" % (c, i & 3, s(self.RSQ if c == "q" else self.RSD, 4), "0" if i < 4 else "%%[%s16]" % c))
            for text, d, n, what in issue.get(m, []):
                x.lds(text, d, n, what)
            for f in work.get(m, []):
                f()
            if m == 20:                                        # whether this tile has scores to mask: vcc for the branch at 32
                x.put("s_cmp_lt_i32 %s, %%[mct]" % s(self.CTC))
                x.put("s_cselect_b64 vcc, -1, 0")
                if self.store_ds:
                    x.put("s_cmp_lg_u32 %[dsmask], 0")
                    x.put("s_cselect_b64 vcc, -1, vcc")
            if self.store_ds and 98 <= m < 98 + 8:
                i = m - 98
                kb_, qb_ = i >> 1, i & 1
                x.put("global_store_dwordx2 %%[dso], %s, %s offset:%d" % (v(self.DSP + 4 * kb_ + 2 * qb_, 2), s(self.DSS, 2), (kb_ >> 1) * 2048 + qb_ * 1024 + (kb_ & 1) * 256))
            if m == 96:
                x.put("s_sub_u32 %[rem], %[rem], 1")
            shift = 10 if self.store_ds else 0                 # behind the stores, which need the tile's own address
            if m - shift in adv_at:
                self.scalar(adv_at[m - shift], stage + (3 if without else 0))

    def text(self):
        x, R = self.x, self
        for dst, name in ((R.RSQ, "qp"), (R.RSD, "dp"), (R.RSL, "lp"), (R.QSTEP, "qstep"), (R.DSTEP, "dstep"), (R.QWRAP, "qwrap"),
                          (R.DWRAP, "dwrap"), (R.LWRAP, "lwrap")) + (((R.DSC, "dsp"), (R.DSTEP_DS, "dsstep"), (R.WRAP_DS, "dswrap")) if self.store_ds else ()):
            x.put("s_mov_b64 %s, %%[%s]" % (s(dst, 2), name))
        for r in (R.RSQ, R.RSD, R.RSL):
            x.put("s_mov_b32 %s, 0x20000" % s(r + 3))
        for i in range(4):
            x.put("v_mov_b32 %s, 0" % v(R.RING + i))
        x.put("s_nop 3")
        for i in range(64):                        # dV = dK = 0
            x.put("%s %%[d%s%d%d], %s, %s, 0" % (x.mfma_name, "vk"[i // 32], i // 8 % 4, i % 8, v(R.RING, 4), v(R.RING, 4)))
        x.put("s_waitcnt vmcnt(0)")
        x.put("s_barrier")                         # the K tile and the first tile are there
        x.put("s_cmp_eq_u32 %[rem], 0")
        x.put("s_cbranch_scc1 %s" % self.ref("END"))
        for piece in self.advance():
            self.scalar(piece, 2)
        for slot, use, d, n, f in self.ops:
            if slot < 0:
                x.lds(f(0, d), d, n, use // 4)
        start = [set(r) for r in x.reads]
        self.masked_from = {}
        self.label("LOOP")
        for stage in range(2):
            self.tile(stage)
            assert len(x.reads) <= len(start) and x.reads == start[-len(x.reads):], "the two ends of the loop differ"
            x.reads = [set(r) for r in start]
            x.put("s_cmp_eq_u32 %[rem], 0")
            x.put("s_cbranch_scc%d %s" % ((1, self.ref("END")) if stage == 0 else (0, self.ref("LOOP"))))
        x.put("s_branch %s" % self.ref("END"))
        end = [set(r) for r in x.reads]
        for i in range(2):
            self.mask(i)
            assert x.reads == end, "the tile ends otherwise"
        for i in range(5):
            self.wrap(i)
        self.label("END")
        x.put("s_waitcnt vmcnt(0) lgkmcnt(0)")
        x.put("s_nop 15")
        x.put("s_nop 7")
        return x.lines


class Keys:
    """What the loops over key tiles have in common: a wavefront holds 64 query rows (four blocks of 16) and walks tiles of 32 keys of
    its stream; the wavefronts of a stream, two or four, copy a tile together (`copies` of its 16 KB each: K or V, or half of
    one), three tiles ahead into four stages, and meet at one barrier a tile, placed where the tile's last LDS read has been waited for.

    The query index is on lanes: block (kb, qb) of S^T is key rows 16 kb + 4 g + v and query 16 qb + r of lane 16 g + r.
    """
    STAGES, TILEB, STAGEB = 4, 8192, 16384         # bytes of a K (or V) tile and of a stage of a stream
    ROWB = 256

    def __init__(self, dtype, copies):
        self.x = Stream(dtype)
        self.copies = copies

    def ref(self, name):
        return "L%s_%%=" % name

    def label(self, name):
        self.x.lines.append(self.ref(name) + ":")

    # scalar registers: the descriptor of the rows that are copied next and how many are left of them; the tile's first key
    RSC, CSTEP, CLEFT, KEY, T = 40, 44, 46, 47, 48

    def enter(self):
        x = self.x
        for dst, name in ((self.RSC, "cp"), (self.CSTEP, "cstep")):
            x.put("s_mov_b64 %s, %%[%s]" % (s(dst, 2), name))
        x.put("s_mov_b32 %s, 0x20000" % s(self.RSC + 3))
        x.put("s_mov_b32 %s, %%[left]" % s(self.CLEFT))
        x.put("s_mov_b32 %s, %%[key]" % s(self.KEY))

    def rows_left(self):
        """Pieces of scalar code: the descriptor's length for the rows that are left."""
        r, t = self, s(self.T)
        return [["s_min_i32 %s, %s, %d" % (t, s(r.CLEFT), 4 * r.copies), "s_mul_i32 %s, %s, %%[crowb]" % (t, t)],
                ["s_sub_u32 %s, %s, %%[crowb]" % (t, t), "s_add_u32 %s, %s, 0x100" % (t, t)],
                ["s_cmp_gt_i32 %s, 0" % s(r.CLEFT), "s_cselect_b32 %s, %s, 0" % (s(r.RSC + 2), t)]]

    def to_next_rows(self):
        r = self
        return [["s_add_u32 %s, %s, %s" % (s(r.RSC), s(r.RSC), s(r.CSTEP)), "s_addc_u32 %s, %s, %s" % (s(r.RSC + 1), s(r.RSC + 1), s(r.CSTEP + 1))],
                ["s_sub_i32 %s, %s, %%[keystep]" % (s(r.CLEFT), s(r.CLEFT))]] + self.rows_left()

    def copy(self, i, stage, before):
        """Copy i of a tile, on both sides of an MFMA."""
        if before:
            self.x.put("s_add_u32 m0, %%[cdst], %d" % (stage * self.STAGEB + 1024 * i))
        else:
            self.x.put("buffer_load_dwordx4 %%[cl%d], %s, %s offen lds" % (i & 3, s(self.RSC, 4), "0" if i < 4 else "%[c16]"))

    def loop(self, tile, first_reads):
        """The unrolled stages of the loop between its labels; `first_reads(stage)` are those in front of the first tile."""
        x = self.x
        x.put("s_cmp_eq_u32 %[rem], 0")
        x.put("s_cbranch_scc1 %s" % self.ref("END"))
        first_reads()
        start = [set(r) for r in x.reads]
        self.label("LOOP")
        for stage in range(self.STAGES):
            tile(stage)
            assert x.reads == start[len(start) - len(x.reads):], "the two ends of the loop differ"
            x.reads = [set(r) for r in start]
            x.put("s_sub_u32 %[rem], %[rem], 1")
            x.put("s_cmp_eq_u32 %[rem], 0")
            last = stage == self.STAGES - 1
            x.put("s_cbranch_scc%d %s" % (0 if last else 1, self.ref("LOOP" if last else "END")))
        x.put("s_branch %s" % self.ref("END"))

    def leave(self):
        self.label("END")
        self.x.put("s_waitcnt vmcnt(0) lgkmcnt(0)")
        self.x.put("s_nop 15")
        self.x.put("s_nop 7")

    def mask_lanes(self, cx, cy):
        """cx = key - row and cy = key - keys of the tile's element (0, 0) of a lane."""
        self.x.put("v_add_u32 %s, %s, %%[vx]" % (v(cx), s(self.KEY)))
        self.x.put("v_add_u32 %s, %s, %%[vy]" % (v(cy), s(self.KEY)))

    def mask(self, first, value, cx, cy, blocks=(0, 1, 2, 3)):
        """The values of a tile (registers from `first`, [qb][kb][v]) past the diagonal or the last key become `value`."""
        x = self.x
        for qb in blocks:
            for kb in range(2):
                for e in range(4):
                    r = v(first + 4 * (2 * qb + kb) + e)
                    for c, op, bound in ((cx, "lt", 16 * qb - 16 * kb - e), (cy, "le", -16 * kb - e)):
                        x.put("v_cmp_%s_i32 vcc, %d, %s" % (op, bound, v(c)))
                        x.put("s_nop 1")
                        x.put("v_cndmask_b32 %s, %s, %s, vcc" % (r, r, value))


class DQ(Keys):
    """dQ: S^T = K Q^T, dP^T = V dO^T - delta, dQ^T += K^T dS^T; 96 MFMAs a tile, a query block after the other in each phase, so that
    P and dS of a block are formed beneath the next blocks' MFMAs."""
    KEEP = 72
    S, DP, DSP, KF, VF, KT, CX, CY, ZERO = 72, 104, 136, 152, 184, 216, 248, 249, 250

    def reads(self, stage):
        """(first MFMA that uses it, MFMA behind which it is issued, destination, width, text) in the order of issue."""
        st, nx, out = stage * self.STAGEB, (stage + 1) % self.STAGES * self.STAGEB, []
        for i in range(8):
            ks, kb = i // 2, i % 2
            out.append((32 + i, 8 + 2 * i, self.VF + 4 * i, 4, "ds_read_b128 %s, %%[rk%d] offset:%d" % (v(self.VF + 4 * i, 4), ks, st + self.TILEB + 16 * self.ROWB * kb)))
        for i in range(16):
            t, h = i // 2, i % 2
            d = self.KT + 4 * t + 2 * h
            out.append((64 + t, 26 + 3 * i // 2, d, 2, "ds_read_b64_tr_b16 %s, %%[ta%d] offset:%d" % (v(d, 2), t, st + 16 * self.ROWB * h)))
        for i in range(8):
            out.append((96 + i, self.AT_BARRIER + 2 * i, self.KF + 4 * i, 4, self.k_read(i, nx)))
        return out

    AT_BARRIER = 74

    def k_read(self, i, st):
        return "ds_read_b128 %s, %%[rk%d] offset:%d" % (v(self.KF + 4 * i, 4), i // 2, st + 16 * self.ROWB * (i % 2))

    def first_reads(self):
        for i in range(8):
            self.x.lds(self.k_read(i, 0), self.KF + 4 * i, 4, 96 + i)

    def vector_work(self):
        x, work = self.x, {}

        def put(slot, f, *args, **kw):
            work.setdefault(slot, []).append(lambda: f(*args, **kw))
        for j in range(16):                        # pairs: query block j / 4, key block (j / 2) % 2, rows 2 (j % 2) ..
            qb, kb, e = j >> 2, (j >> 1) & 1, 2 * (j & 1)
            p, d = self.S + 4 * (2 * qb + kb) + e, self.DP + 4 * (2 * qb + kb) + e
            at = 9 + 43 * j // 15
            for i in range(2):
                put(at, x.valu, "v_fma_f32", v(p + i), v(p + i), "%[scale]", "-%%[lse%d]" % qb)
            for i in range(2):
                put(at + 1, x.valu, "v_exp_f32", v(p + i), v(p + i), trans=True)
            at = self.AT_MASK + 15 * j // 8
            for i in range(2):
                put(at, x.valu, "v_mul_f32", v(p + i), v(p + i), v(d + i))
            put(at + 1, x.valu, x.pack_name, v(self.DSP + 4 * qb + 2 * kb + e // 2), v(p), v(p + 1))
        return work

    AT_MASK = 55

    def tile(self, stage):
        x = self.x
        self.piece(stage, 0, self.AT_MASK)
        x.put("s_cmp_gt_i32 %s, %%[mlim]" % s(self.KEY))
        x.put("s_cbranch_scc1 %s" % self.ref("MASK%d" % stage))
        self.label("MASKED%d" % stage)
        self.masked_from[stage] = x.state()
        self.piece(stage, self.AT_MASK, 96)
        self.label("DONE%d" % stage)

    def piece(self, stage, first, end, without=()):
        """MFMAs `first` to `end` of a tile and what goes with them; the products of the query blocks `without` are left out."""
        x, work, issue = self.x, self.vector_work(), {}
        for use, at, d, n, text in self.reads(stage):
            issue.setdefault(at, []).append((text, d, n, use))
        next_rows = dict(zip(range(40, 56, 3), self.to_next_rows()))
        for m in range(first, end):
            phase, qb, i = m // 32, m // 8 % 4, m % 8
            copies = (m - 1) // 3 if m % 3 == 1 and m < 3 * self.copies else None
            if copies is not None:
                self.copy(copies, (stage + 3) % self.STAGES, True)
            if m == 64 and without:
                x.settle()
                x.wait(set(range(self.KT, self.KT + 32)))
            if m == self.AT_BARRIER:
                x.put("s_waitcnt vmcnt(%d)" % (2 * self.copies))       # the next tile has landed ..
                x.put("s_barrier")                 # .. both its halves, and nobody reads this one any more
            if phase < 2:
                ks, kb = i // 2, i % 2
                d, frag = (self.S, self.DP)[phase] + 4 * (2 * qb + kb), (self.KF, self.VF)[phase] + 4 * i
                args = (v(d, 4), v(frag, 4), "%%[%s%d%d]" % ("qd"[phase], qb, ks), v(d, 4) if ks else ("0", "%%[nd%d]" % qb)[phase])
                holds = [(v(frag, 4), (96 if phase == 0 else 32) + i)]
            else:
                frag = self.KT + 4 * i
                acc = "%%[o%d%d]" % (qb, i)
                args = (acc, v(frag, 4), v(self.DSP + 4 * qb, 4), acc)
                holds = [(v(frag, 4), 64 + i)]
            if phase < 2 or qb not in without:
                need = set(range(frag, frag + 4))
                if qb == 0 and i % 2 == 0:         # one wait for two fragments
                    need |= set(range(frag, frag + 8))
                x.wait(need)
                x.mfma(*args, holds)
            if copies is not None:
                self.copy(copies, 0, False)
            for text, d, n, use in issue.get(m, []):
                x.lds(text, d, n, use)
            for f in work.get(m, []):
                f()
            for line in next_rows.get(m, []):
                x.put(line)
            if m == 80:
                x.put("s_add_u32 %s, %s, %%[keystep]" % (s(self.KEY), s(self.KEY)))

    def text(self):
        x = self.x
        self.enter()
        for line in sum(self.rows_left(), []):
            x.put(line)
        x.put("v_mov_b32 %s, 0" % v(self.ZERO))
        for i in range(4):
            x.put("v_mov_b32 %s, 0" % v(self.KT + i))
        x.put("s_nop 3")
        for i in range(32):
            x.put("%s %%[o%d%d], %s, %s, 0" % (x.mfma_name, i // 8, i % 8, v(self.KT, 4), v(self.KT, 4)))
        x.put("s_waitcnt vmcnt(%d)" % (2 * self.copies))
        x.put("s_barrier")
        self.masked_from = {}
        self.loop(self.tile, self.first_reads)
        end = [set(r) for r in x.reads]
        for stage in range(self.STAGES):
            self.label("MASK%d" % stage)
            self.mask_lanes(self.CX, self.CY)
            self.mask(self.S, v(self.ZERO), self.CX, self.CY)
            x.put("s_cmp_gt_i32 %s, %%[alim]" % s(self.KEY))
            x.put("s_cbranch_scc0 %s" % self.ref("MASKED%d" % stage))
            # keys behind the first 32 rows, or behind all 64: their blocks get no product
            x.put("s_add_u32 %s, %%[alim], 32" % s(self.T))
            x.put("s_cmp_gt_i32 %s, %s" % (s(self.KEY), s(self.T)))
            x.put("s_cbranch_scc1 %s" % self.ref("IDLE%d" % stage))
            x.pad = True
            for without in ((0, 1), (0, 1, 2, 3)):
                if len(without) == 4:
                    self.label("IDLE%d" % stage)
                x.resume(self.masked_from[stage])
                self.piece(stage, self.AT_MASK, 96, without)
                assert x.reads == end[len(end) - len(x.reads):], "the tile ends otherwise"
                x.put("s_branch %s" % self.ref("DONE%d" % stage))
            x.pad = False
        self.leave()
        return x.lines


class FWD(Keys):
    """Forward: S^T = K Q^T, P = 2^(S c - m), O^T += V^T P^T; 64 MFMAs a tile.  The query blocks go in two groups, A (0, 1) and B (2, 3), and
    the tile in quarters of 16 MFMAs,
        S of A | O of B, of the tile before | S of B | O of A,
    so that the softmax of either group has two quarters of MFMAs above it before its product is due.

    m is only a reference for the exponentials: the first 64 keys set it ahead of the loop (``reference``), so that the largest of few scores is 1
    exactly, and it moves (``move``, out of line) when the eight values of some lane sum to more than 2^8.  One branch asks that of a group, some instructions behind the comparisons (the
    branch directly behind each block's comparison cost 70 cycles apiece).  Tiles with scores to mask run a copy of the tile's code that
    masks a group's scores in front of its softmax.  O is divided by the sums of P as it was rounded, which one MFMA with ones a block
    brings, in a[128:143]: where a few scores dominate a row their rounding then cancels.  O is a[0:127] (query block, d block); at the end it goes to LDS as 64 rows of
    fp32, 16-byte chunks XORed with the row.
    """
    KEEP = 48
    S, KF, VT, P, PP, TS, MT, MX, TY, CX, CY, NEG = 48, 80, 112, 144, 160, 176, 180, 188, 189, 190, 191, 192
    ONES, SUMS = 194, 128
    RET, OVER, BOUND, BACK = 50, 52, 54, 56
    AT_BARRIER = 46

    def __init__(self, dtype, copies):
        super().__init__(dtype, copies)
        self.ones = {"bf16": "0x3f803f80", "f16": "0x3c003c00"}[dtype]

    def k_read(self, i, st):
        return "ds_read_b128 %s, %%[rk%d] offset:%d" % (v(self.KF + 4 * i, 4), i // 2, st + 16 * self.ROWB * (i % 2))

    def first_reads(self):
        for i in range(8):
            self.x.lds(self.k_read(i, 0), self.KF + 4 * i, 4, "k")

    def reads(self, stage):
        """(MFMA behind which it is issued, destination, width, text, what)."""
        st, nx, out = stage * self.STAGEB + self.TILEB, (stage + 1) % self.STAGES * self.STAGEB, []
        for i in range(16):
            t, h = i // 2, i % 2
            d = self.VT + 4 * t + 2 * h
            out.append((31 + i, d, 2, "ds_read_b64_tr_b16 %s, %%[ta%d] offset:%d" % (v(d, 2), t, st + 16 * self.ROWB * h), "v"))
        for i in range(8):
            out.append((self.AT_BARRIER + 1 + 2 * i, self.KF + 4 * i, 4, self.k_read(i, nx), "k"))
        return out

    def probs(self, qb):
        return [self.P + 8 * (qb & 1) + i for i in range(8)]

    def softmax(self, qb):
        """P of a block, packed, the sum of a lane's eight values and whether it is too large, as a list of instructions."""
        x, p, sc, ts, out = self.x, self.probs(qb), [self.S + 8 * qb + i for i in range(8)], v(self.TS + qb), []
        for i in range(0, 8, 2):
            out += [lambda i=i, k=k: x.valu("v_fma_f32", v(p[i + k]), v(sc[i + k]), "%[scale]", "-%%[m%d]" % qb) for k in range(2)]
            if i:                                  # of the two values before
                out.append(lambda i=i: x.valu(x.pack_name, v(self.PP + 4 * qb + i // 2 - 1), v(p[i - 2]), v(p[i - 1])))
            out += [lambda i=i, k=k: x.valu("v_exp_f32", v(p[i + k]), v(p[i + k]), trans=True) for k in range(2)]
            if i == 2:
                out.append(lambda: x.valu("v_add_f32", ts, v(p[0]), v(p[1])))
            elif i:
                out += [lambda i=i, k=k: x.valu("v_add_f32", ts, ts, v(p[i - 2 + k])) for k in range(2)]
        out += [lambda: x.valu("v_add_f32", ts, ts, v(p[6])),
                lambda: x.valu(x.pack_name, v(self.PP + 4 * qb + 3), v(p[6]), v(p[7])),
                lambda: x.valu("v_add_f32", ts, ts, v(p[7])),
                lambda: x.put("v_cmp_lt_f32 %s, %s, %s" % ("vcc" if qb & 1 else s(self.OVER, 2), s(self.BOUND), ts))]
        return out

    def check(self, group, name):
        x = self.x
        x.put("s_or_b64 vcc, vcc, %s" % s(self.OVER, 2))
        x.put("s_cbranch_vccnz %s" % self.ref("GROW%d%s" % (group, name)))
        self.label("GROWN%d%s" % (group, name))
        self.stubs.append((group, name))
        for qb in (2 * group, 2 * group + 1):
            x.valu("v_add_f32", "%%[l%d]" % qb, "%%[l%d]" % qb, v(self.TS + qb))

    def move(self, qb):
        """Out of line, called: the reference moves to the largest score of the row so far; O, l and P follow."""
        x, sc, mx, ty = self.x, [self.S + 8 * qb + i for i in range(8)], v(self.MX), v(self.TY)
        p = [self.MT + i for i in range(8)]
        self.label("MOVE%d" % qb)
        x.put("s_nop 15")
        for i in range(8):
            x.put("v_mul_f32 %s, %%[scale], %s" % (v(p[i]), v(sc[i])))
        x.put("v_max3_f32 %s, %s, %s, %s" % (mx, v(p[0]), v(p[1]), v(p[2])))
        x.put("v_max3_f32 %s, %s, %s, %s" % (mx, mx, v(p[3]), v(p[4])))
        x.put("v_max3_f32 %s, %s, %s, %s" % (mx, mx, v(p[5]), v(p[6])))
        x.put("v_max_f32 %s, %s, %s" % (mx, mx, v(p[7])))
        self.row_max(mx, ty)
        x.put("v_max_f32 %s, %s, %%[m%d]" % (mx, mx, qb))
        x.put("v_sub_f32 %s, %%[m%d], %s" % (ty, qb, mx))
        x.put("v_exp_f32 %s, %s" % (ty, ty))
        x.put("v_mov_b32 %%[m%d], %s" % (qb, mx))
        x.put("s_nop 0")
        x.put("v_mul_f32 %%[l%d], %%[l%d], %s" % (qb, qb, ty))
        acc = [32 * qb + i for i in range(32)] + [self.SUMS + 4 * qb + i for i in range(4)]
        for i in range(0, 36, 8):                  # eight of the block's registers at a time
            for f in ("v_accvgpr_read_b32 {p}, a{a}", "v_mul_f32 {p}, {p}, {y}", "v_accvgpr_write_b32 a{a}, {p}"):
                for k, n in enumerate(acc[i:i + 8]):
                    x.put(f.format(p=v(p[k]), a=n, y=ty))
        for i in range(8):
            x.put("v_fma_f32 %s, %s, %%[scale], -%%[m%d]" % (v(p[i]), v(sc[i]), qb))
        for i in range(8):
            x.put("v_exp_f32 %s, %s" % (v(p[i]), v(p[i])))
        x.put("s_nop 0")
        ts = v(self.TS + qb)
        x.put("v_add_f32 %s, %s, %s" % (ts, v(p[0]), v(p[1])))
        for i in range(2, 8):
            x.put("v_add_f32 %s, %s, %s" % (ts, ts, v(p[i])))
        for i in range(4):
            x.put("%s %s, %s, %s" % (x.pack_name, v(self.PP + 4 * qb + i), v(p[2 * i]), v(p[2 * i + 1])))
        x.put("s_nop 7")
        x.put("s_setpc_b64 %s" % s(self.RET, 2))

    def row_max(self, mx, ty):
        """The largest of the four lanes 16 apart."""
        x = self.x
        for swap in ("v_permlane32_swap_b32", "v_permlane16_swap_b32"):
            x.put("v_mov_b32 %s, %s" % (ty, mx))
            x.put("s_nop 1")
            x.put("%s %s, %s" % (swap, mx, ty))
            x.put("s_nop 1")
            x.put("v_max_f32 %s, %s, %s" % (mx, mx, ty))

    def reference(self):
        """m from the scores of the first 64 keys, whichever split has them (where they are masked, or there are none, it stays very
        low): a row's reference, by which its P is rounded, is then the same with and without splits."""
        x, split = self.x, self.copies == 8
        if split:
            x.put("s_mov_b32 %s, 0" % s(self.KEY))
            x.put("s_lshl_b32 %s, %%[key], 11" % s(self.T))      # 32 keys on is the next stream's tile
            for ks in range(4):
                x.put("v_subrev_u32 %s, %s, %%[rk%d]" % (v(self.VT + ks), s(self.T), ks))
        for st in range(2):
            if split and st:
                for ks in range(4):
                    x.put("v_add_u32 %s, 0x%x, %s" % (v(self.VT + ks), self.STAGES * self.STAGEB, v(self.VT + ks)))
            for i in range(8):
                text = self.k_read(i, 0 if split else st * self.STAGEB)
                x.lds(re.sub(r"%\[rk(\d)\]", lambda a: v(self.VT + int(a[1])), text) if split else text, self.KF + 4 * i, 4, "k")
            for m in range(32):
                self.scores_mfma(m // 16, m % 16)
            x.settle()
            x.put("s_cmp_gt_i32 %s, %%[mlim]" % s(self.KEY))
            x.put("s_cbranch_scc1 %s" % self.ref("FIRST%d" % st))
            self.label("FIRSTED%d" % st)
            x.put("s_add_u32 %s, %s, 32" % (s(self.KEY), s(self.KEY)))
            for qb in range(4):
                p, mx = self.probs(qb), v(self.TS + qb)
                for i in range(8):
                    x.put("v_mul_f32 %s, %%[scale], %s" % (v(p[i]), v(self.S + 8 * qb + i)))
                rest = p if st else p[1:]
                first = mx if st else v(p[0])
                x.put("v_max3_f32 %s, %s, %s, %s" % (mx, first, v(rest[0]), v(rest[1])))
                for i in range(2, len(rest) - 1, 2):
                    x.put("v_max3_f32 %s, %s, %s, %s" % (mx, mx, v(rest[i]), v(rest[i + 1])))
                if len(rest) % 2:
                    x.put("v_max_f32 %s, %s, %s" % (mx, mx, v(rest[-1])))
        x.put("s_mov_b32 %s, %%[key]" % s(self.KEY))
        for qb in range(4):
            self.row_max(v(self.TS + qb), v(self.TY))
            x.put("v_max_f32 %%[m%d], %%[m%d], %s" % (qb, qb, v(self.TS + qb)))

    def scores_mfma(self, group, m):
        """MFMA m of 16: S of a group, a block after the other."""
        qb, ks, kb = 2 * group + m // 8, m % 8 // 2, m % 2
        d, frag = self.S + 4 * (2 * qb + kb), self.KF + 4 * (m % 8)
        need = set(range(frag, frag + 8)) if m < 8 and m % 2 == 0 else set(range(frag, frag + 4))      # one wait for two fragments
        self.x.wait(need)
        self.x.mfma(v(d, 4), v(frag, 4), "%%[q%d%d]" % (qb, ks), v(d, 4) if ks else "0", [(v(frag, 4), "k")])

    def out_mfma(self, group, m):
        """MFMA m of 16: O of a group."""
        qb, t = 2 * group + m // 8, m % 8
        frag, acc = self.VT + 4 * t, "a[%d:%d]" % (32 * (2 * group + m // 8) + 4 * (m % 8), 32 * (2 * group + m // 8) + 4 * (m % 8) + 3)
        self.x.wait(set(range(frag, frag + 8)) if m < 8 and m % 2 == 0 else set(range(frag, frag + 4)))
        self.x.mfma(acc, v(frag, 4), v(self.PP + 4 * qb, 4), acc)
        if t == 7:
            acc = "a[%d:%d]" % (self.SUMS + 4 * qb, self.SUMS + 4 * qb + 3)
            self.x.mfma(acc, v(self.ONES, 4), v(self.PP + 4 * qb, 4), acc)

    B_HEAD = 15                                    # MFMAs of the tile beneath which B's softmax begins; the rest of it is in the next tile

    def b_softmax(self, head):
        todo = self.softmax(2) + self.softmax(3)
        n = (len(todo) * self.B_HEAD + 13) // (self.B_HEAD + 12)
        return todo[:n] if head else todo[n:]

    def body(self, stage, masked, without_a=False):
        """The code of a tile; where it lies behind the rows of group A their product is left out."""
        x, issue, work = self.x, {}, {}
        name = "%s%d" % ("L" if without_a else "M" if masked else "T", stage)
        for at, d, n, text, what in self.reads(stage):
            issue.setdefault(at, []).append((text, d, n, what))

        def spread(todo, first, slots):
            for i, f in enumerate(todo):
                work.setdefault(first + slots * i // len(todo), []).append(f)
        spread(self.b_softmax(False), 0, 12)
        work.setdefault(14, []).append(lambda: self.check(1, name))
        spread(self.softmax(0) + self.softmax(1), 17, 27)
        work.setdefault(45, []).append(lambda: self.check(0, name))
        spread(self.b_softmax(True), 49, self.B_HEAD)
        next_rows = dict(zip(range(18, 40, 4), self.to_next_rows()))
        for m in range(64):
            gap = 16 // self.copies
            copy = (m - 49) // gap if m >= 49 and (m - 49) % gap == 0 and (m - 49) // gap < self.copies else None
            if copy is not None:
                self.copy(copy, (stage + 3) % self.STAGES, True)
            if masked and m in (16, 48):
                x.settle()
                if m == 16:
                    self.mask_lanes(self.CX, self.CY)
                self.mask(self.S, v(self.NEG), self.CX, self.CY, (0, 1) if m == 16 else (2, 3))
            if m == self.AT_BARRIER:
                x.put("s_waitcnt vmcnt(%d)" % self.copies)     # the next tile has landed ..
                x.put("s_barrier")                 # .. all of it, and everybody has what it needs of the tile before
            if m == 48 and without_a:
                x.wait(set(range(self.VT, self.VT + 32)))
            if m < 48 or not without_a:
                (self.scores_mfma, self.out_mfma)[m // 16 % 2]((0, 1, 1, 0)[m // 16], m % 16)
            if copy is not None:
                self.copy(copy, 0, False)
            for text, d, n, what in issue.get(m, []):
                x.lds(text, d, n, what)
            for f in work.get(m, []):
                f()
            for line in next_rows.get(m, []):
                x.put(line)
        x.put("s_add_u32 %s, %s, %%[keystep]" % (s(self.KEY), s(self.KEY)))

    def last_b(self, name):
        """The product of the last tile's group B."""
        x = self.x
        x.resume(self.begin[0])
        x.reads = []
        for f in self.b_softmax(False):
            f()
            if x.trans:
                x.put("s_nop 0")
        self.check(1, name)
        x.put("s_nop 3")
        for m in range(16):
            self.out_mfma(1, m)

    def idle(self, stage):
        """A tile behind all rows of the wavefront: its share of the copies, and the others' meeting point."""
        x = self.x
        for line in sum(self.to_next_rows(), []):
            x.put(line)
        x.put("s_waitcnt vmcnt(%d)" % self.copies)
        x.put("s_barrier")
        for i in range(self.copies):
            self.copy(i, (stage + 3) % self.STAGES, True)
            x.put("s_nop 0")
            self.copy(i, 0, False)

    def tile(self, stage):
        x = self.x
        x.put("s_cmp_gt_i32 %s, %%[mlim]" % s(self.KEY))
        x.put("s_cbranch_scc1 %s" % self.ref("MASKED%d" % stage))
        self.begin[stage] = x.state()
        self.body(stage, False)
        self.label("DONE%d" % stage)

    def text(self):
        x, self.stubs, self.begin = self.x, [], {}
        self.enter()
        for line in sum(self.rows_left(), []):
            x.put(line)
        x.put("v_mov_b32 %s, 0xff800000" % v(self.NEG))
        x.put("s_waitcnt vmcnt(%d)" % self.copies)
        x.put("s_barrier")                         # the first two tiles are there
        self.reference()
        # the group B of a tile in front of the first: no scores, no values
        for i in range(16):
            x.put("v_mov_b32 %s, %s" % (v(self.S + 16 + i), v(self.NEG)))
        for i in range(32):
            x.put("v_mov_b32 %s, 0" % v(self.VT + i))
        for i in range(4):
            x.put("v_mov_b32 %s, %s" % (v(self.ONES + i), self.ones))
        x.put("s_mov_b32 %s, 0x43800000" % s(self.BOUND))
        x.put("s_nop 3")
        for i in range(36):
            x.put("%s a[%d:%d], %s, %s, 0" % (x.mfma_name, 4 * i, 4 * i + 3, v(self.VT, 4), v(self.VT, 4)))
        for f in self.b_softmax(True):
            f()
            if x.trans:
                x.put("s_nop 0")
        self.loop(self.tile, self.first_reads)
        end = [set(r) for r in x.reads]
        for stage in range(self.STAGES):
            self.label("MASKED%d" % stage)
            x.put("s_cmp_gt_i32 %s, %%[alim]" % s(self.KEY))
            x.put("s_cbranch_scc1 %s" % self.ref("LATE%d" % stage))
            for without_a in (False, True):
                if without_a:
                    self.label("LATE%d" % stage)
                    x.put("s_add_u32 %s, %%[alim], 32" % s(self.T))
                    x.put("s_cmp_gt_i32 %s, %s" % (s(self.KEY), s(self.T)))
                    x.put("s_cbranch_scc1 %s" % self.ref("IDLE%d" % stage))
                x.resume(self.begin[stage])
                x.pad = without_a
                self.body(stage, True, without_a)
                x.pad = False
                assert x.reads == end[len(end) - len(x.reads):], "the masked tile ends otherwise"
                x.put("s_branch %s" % self.ref("DONE%d" % stage))
        for stage in range(self.STAGES):
            self.label("IDLE%d" % stage)
            x.put("s_waitcnt lgkmcnt(0)")
            x.put("s_nop 15")
            x.put("s_call_b64 %s, %s" % (s(self.BACK, 2), self.ref("LASTB")))
            x.put("s_branch %s" % self.ref("REST%d" % stage))
        for stage in range(self.STAGES):
            self.label("REST%d" % stage)
            self.idle(stage)
            x.put("s_sub_u32 %[rem], %[rem], 1")
            x.put("s_cmp_lg_u32 %[rem], 0")
            x.put("s_cbranch_scc%d %s" % ((1, self.ref("REST0")) if stage == self.STAGES - 1 else (0, self.ref("RESTED"))))
        self.label("RESTED")
        x.put("s_waitcnt vmcnt(0)")
        x.put("s_branch %s" % self.ref("WRITE"))
        self.label("LASTB")
        self.last_b("R")
        x.put("s_setpc_b64 %s" % s(self.BACK, 2))
        self.leave()
        self.last_b("E")
        self.label("WRITE")
        x.put("s_nop 15")
        x.put("s_nop 7")
        x.put("s_barrier")                         # everyone is done with the tiles
        for qb in range(4):
            x.put("v_accvgpr_read_b32 %%[n%d], a%d" % (qb, self.SUMS + 4 * qb))
        for qb in range(4):
            for t in range(8):
                x.put("ds_write_b128 %%[wo%d], a[%d:%d] offset:%d" % (t, 32 * qb + 4 * t, 32 * qb + 4 * t + 3, 8192 * qb))
        x.put("s_waitcnt lgkmcnt(0)")
        x.put("s_branch %s" % self.ref("OUT"))
        for st in range(2):
            self.label("FIRST%d" % st)
            self.mask_lanes(self.CX, self.CY)
            self.mask(self.S, v(self.NEG), self.CX, self.CY)
            x.put("s_branch %s" % self.ref("FIRSTED%d" % st))
        for group, name in self.stubs:
            self.label("GROW%d%s" % (group, name))
            for qb in (2 * group, 2 * group + 1):
                x.put("s_call_b64 %s, %s" % (s(self.RET, 2), self.ref("MOVE%d" % qb)))
            x.put("s_branch %s" % self.ref("GROWN%d%s" % (group, name)))
        for qb in range(4):
            self.move(qb)
        self.label("OUT")
        return x.lines


def define(name, lines):
    return "#define %s \\\n" % name + " \\\n".join('  "%s\\n\\t"' % l for l in lines) + "\n"


def clobbers(name, first_v, last_v, first_s, last_s, agprs=0):
    names = ["a%d" % i for i in range(agprs)] + ["v%d" % i for i in range(first_v, last_v + 1)] + ["s%d" % i for i in range(first_s, last_s + 1)] + ["vcc", "scc", "m0", "memory"]
    return "#define %s %s\n" % (name, ", ".join('"%s"' % n for n in names))


def generate():
    out = ["// Written by attn_loops.py.\n#pragma once\n"]
    for dtype in ("bf16", "f16"):
        for ds in (False, True):
            out.append(define("DH_DKV128_LOOP_%s%s" % (dtype.upper(), "_DS" if ds else ""), DKV(dtype, ds).text()))
        for copies in (4, 8):
            out.append(define("DH_DQ128_LOOP_%s_%d" % (dtype.upper(), copies), DQ(dtype, copies).text()))
        for copies in (4, 8):
            out.append(define("DH_FWD128_LOOP_%s_%d" % (dtype.upper(), copies), FWD(dtype, copies).text()))
    out.append(clobbers("DH_DKV128_CLOBBERS", DKV.KEEP, DKV.NEG, DKV.RSQ, DKV.PADS + 7))
    out.append(clobbers("DH_DQ128_CLOBBERS", DQ.KEEP, DQ.ZERO, Keys.RSC, Keys.T))
    out.append(clobbers("DH_FWD128_CLOBBERS", FWD.KEEP, FWD.ONES + 3, Keys.RSC, FWD.BACK + 1, FWD.SUMS + 16))
    return "".join(out)


if __name__ == "__main__":
    with open(sys.argv[1], "w") as f:
        f.write(generate())
