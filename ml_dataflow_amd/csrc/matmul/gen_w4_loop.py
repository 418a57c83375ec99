#!/usr/bin/env python3
"""Writes gemm_w4_loop.inc: the k-loops of the four-wave GEMM kernels of gemm_w4_kernel.h as inline-assembly text
(gemm_bf16_w4_kernel: classes Mult and Loader, described here; gemm_bf16_w4d_kernel: class Wide, gemm_bf16_w4k_kernel: class Ring, described there).  Run
by the Makefile; the output is a build product.

The kernel: 256 threads, one wave per SIMD, work-group tile 256 (m) x 288 (n) x 64 (k).  The waves have two roles.

  Wave 0 loads.  It requests the operands from global memory into its own registers (buffer_load_dwordx4 into
  accumulation registers, 68 chunks of 1 KiB per k-tile: 32 of P, 36 of Q, a chunk being eight rows of 128 bytes or, for
  a k-major operand, two k-rows of 256 rows) and writes them to the LDS stages with ds_write_b128.  The stream is a
  sequence of slots, 68 per k-tile; which chunk a slot carries (its global offset and its LDS address are per-slot
  registers) is up to the caller, who rotates the chunks by work-group so that the work-groups which share an operand
  panel ask for a given line at different times.  The stream is one sliding window: behind the write of slot t comes the
  load of slot t + 60, into the registers that the write of slot t - 8 has left, so 60 KiB are in flight at any time,
  also across k-tiles and barriers.  A wave that issues a load
  while the memory pipeline of the compute unit is full waits until the load is accepted; this wave has nothing else to do.
  Waves 1-3 multiply.  Wave w owns columns [96 (w - 1), 96 w) of the tile and all 256 rows: 16 x 6 blocks of 16 x 16,
  v_mfma_f32_16x16x32_bf16, accumulators in a[0:255] and v[0:127].  They read fragments from the LDS and never touch
  global memory, so nothing but the barrier ever holds their matrix instructions up.

One barrier per k-tile: when the loader has written k-tile g+1 and the multiplying waves have read the last fragment of
k-tile g.  One asm statement per role covers the k-tiles of one output tile.

State from statement to statement (tile to tile): LDS stage 0 holds k-tile 0 of the tile, visible to all waves; the
loader's registers hold chunks 0..59 of k-tile 1, landed (the statement ends with s_waitcnt vmcnt(0)); chunks 60..67 of
k-tile 1 are the first loads of the next statement.  k-tile counts are even; the loader fetches the next tile's first
k-tiles while the last ones of this tile are multiplied (a next tile that does not exist has an empty buffer: zeros).

Multiplying wave, step g (stage p = g & 1), MFMA m = 0..191 in the order k-step s, row block i, column block j:
  * the fragment of P for row block a = 16 s + i goes to ring slot a % 4, read right behind the last MFMA of block a - 4;
  * the six fragments of Q of k-step 1 are read during k-step 0 into the second buffer, those of k-step 0 of the next
    k-tile behind the barrier;
  * behind MFMA 179: s_waitcnt lgkmcnt(0), s_barrier, then the first reads of stage 1 - p; 12 MFMAs are left to cover them.
s_waitcnt lgkmcnt values come from a simulation of the in-order LDS queue.
"""
import os
import sys

P_STAGE = 32768          # bytes of one P stage (256 rows x 64 k)
Q_STAGE = 36864          # bytes of one Q stage (288 rows x 64 k)
CHUNKS_P, CHUNKS_Q = 32, 36
CHUNKS = CHUNKS_P + CHUNKS_Q
WINDOW = 60              # chunks in flight
LAG = CHUNKS - WINDOW

# loader registers
L_VOFFP, L_VOFFQ, L_VOFFQ_NEXT, L_WR = 16, 48, 84, 120        # v[0:15]: slots 64..67; then offsets; LDS write address of every slot
# multiplying-wave registers
M_BF, M_AF, M_ARD, M_BRD = 128, 176, 192, 200                 # v[0:127]: accumulator groups 16..23

# schedule parameters (W4_OPTS="key=value,..." overrides them for experiments; ablations give wrong results, timing only)
OPTS = {"abl": "", "pre": 4, "first": 2, "every": 3, "qfirst": 14, "qevery": 13}
for kv in os.environ.get("W4_OPTS", "").split(","):
    if "=" in kv and kv.split("=", 1)[0] in OPTS:
        k_, v_ = kv.split("=", 1)
        OPTS[k_] = type(OPTS[k_])(v_)
ABL = set(OPTS["abl"].split("+")) if OPTS["abl"] else set()


class Asm:
    def __init__(self):
        self.L = []
        self.issued, self.prod, self.known_done = 0, {}, -1

    def e(self, x):
        if ("noloads" in ABL and x.startswith("buffer_load")) or ("nowrites" in ABL and x.startswith("ds_write")) or \
           ("nobar" in ABL and x == "s_barrier") or ("nomfma" in ABL and x.startswith("v_mfma")) or \
           ("noreads" in ABL and x.startswith("ds_read_b")) or ("nolgkm" in ABL and x.startswith("s_waitcnt lgkmcnt(") and not x.endswith("(0)")) or ("novm" in ABL and x.startswith("s_waitcnt vmcnt") and "lgkm" not in x):
            return
        if "oob" in ABL and (x.startswith("s_cselect_b32 s66,") or x.startswith("s_cselect_b32 s70,")):
            x = "s_mov_b32 s%s, 0" % x.split()[1][1:3]
        self.L.append(x)

    def lds(self, text, key=None):
        self.e(text)
        if key is not None:
            self.prod[key] = self.issued
        self.issued += 1

    def need(self, *keys):
        n = max(self.prod.get(k, -1) for k in keys)
        if n > self.known_done:
            after = self.issued - 1 - n
            assert 0 <= after <= 15, after
            self.e("s_waitcnt lgkmcnt(%d)" % after)
            self.known_done = n

    def barrier(self):
        self.e("s_barrier")

    def lds_drain(self):
        self.e("s_waitcnt lgkmcnt(0)")
        self.known_done = self.issued - 1


def vr(lo, n):
    return "v%d" % lo if n == 1 else "v[%d:%d]" % (lo, lo + n - 1)


# ================================================================================================ multiplying waves
class Mult(Asm):
    """s40: k-tiles (even), s41 bit 0: first tile of the work-group"""

    def __init__(self, PKM):
        Asm.__init__(self)
        self.PKM = PKM
        self.name = "W4_MULT_%s" % ("PKM" if PKM else "PKC")

    def acc(self, i, j):
        g = (i // 4) * 6 + j
        lo = (i % 4) * 4
        if g < 16:
            return "a[%d:%d]" % (16 * g + lo, 16 * g + lo + 3)
        return "v[%d:%d]" % (16 * (g - 16) + lo, 16 * (g - 16) + lo + 3)

    def read_A(self, stage, a):
        s, i = divmod(a, 16)
        dst = M_AF + (a % 4) * 4
        if not self.PKM:
            self.lds("ds_read_b128 %s, v%d offset:%d" % (vr(dst, 4), M_ARD + s, stage * P_STAGE + i * 2048), ("A", a % 4))
        else:
            off = stage * P_STAGE + s * 32 * 512 + (i // 8) * 256
            self.lds("ds_read_b64_tr_b16 %s, v%d offset:%d" % (vr(dst, 2), M_ARD + (i % 8), off))
            self.lds("ds_read_b64_tr_b16 %s, v%d offset:%d" % (vr(dst + 2, 2), M_ARD + (i % 8), off + 4 * 512), ("A", a % 4))

    def read_B(self, stage, s, j):
        dst = M_BF + s * 24 + j * 4
        self.lds("ds_read_b128 %s, v%d offset:%d" % (vr(dst, 4), M_BRD + s * 2 + stage, j * 2048), ("B", s, j))

    def tail_reads(self, stage, which, blocks=6):
        if which == 0:
            self.read_B(stage, 0, 0)
            self.read_A(stage, 0)
            for j in range(1, blocks):
                self.read_B(stage, 0, j)
            self.read_A(stage, 1)
        else:
            self.read_A(stage, 1 + which)

    def loop_head_state(self, blocks=6):
        self.issued, self.known_done, self.prod = 0, -1, {}
        keep, self.L = self.L, []
        for which in range(3):
            self.tail_reads(0, which, blocks)
        self.L = keep

    def step(self, p):
        after = {}

        def at(m, fn):
            after.setdefault(m, []).append(fn)

        for a in range(4, 32):
            at(6 * (a - 4) + 5, lambda a=a: self.read_A(p, a))
        for j in range(6):
            at(30 + 6 * j + 2, lambda j=j: self.read_B(p, 1, j))

        def barrier():
            self.lds_drain()
            self.barrier()
            self.tail_reads(1 - p, 0)
        at(179, barrier)
        at(185, lambda: self.tail_reads(1 - p, 1))
        at(191, lambda: self.tail_reads(1 - p, 2))
        if p == 1:
            at(187, lambda: self.e("s_add_u32 s76, s76, 2"))
            at(188, lambda: self.e("s_cmp_lt_u32 s76, s40"))
        for m in range(192):
            s, rem = divmod(m, 96)
            i, j = divmod(rem, 6)
            if i & 1:
                j = 5 - j                        # one operand stays from each MFMA to the next: 0.8 % less time at the card's power limit
            a = s * 16 + i
            self.need(("A", a % 4), ("B", s, j))
            self.e("v_mfma_f32_16x16x32_bf16 %s, %s, %s, %s" % (self.acc(i, j), vr(M_AF + (a % 4) * 4, 4), vr(M_BF + s * 24 + j * 4, 4), self.acc(i, j)))
            for fn in after.get(m, []):
                fn()

    def generate(self):
        e = self.e
        e("s_mov_b32 s76, 0")
        e("s_bitcmp1_b32 s41, 0")
        e("s_cbranch_scc0 2f")
        e("s_barrier")                      # first tile: the loader has written k-tile 0
        e("2:")
        for which in range(3):
            self.tail_reads(0, which)
        e("3:")
        self.loop_head_state()
        self.step(0)
        self.loop_head_state()
        self.step(1)
        e("s_cbranch_scc1 3b")
        e("s_waitcnt lgkmcnt(0)")
        for _ in range(3):
            e("s_nop 7")
        return self.L

    def clobbers(self):
        return ["v%d" % i for i in range(M_BF, M_ARD)] + ["s76", "scc", "memory"]


# ================================================================================================ loader wave
class Loader(Asm):
    """s[40:47] this tile's cursor at k-tile 0 (P base lo, hi, extent lo, hi, then Q), s[48:55] the next tile's,
    s56 k-tiles (even), s57 bit 0: first tile of the work-group, s58 / s59 bytes per k-tile of P / Q.
    Working registers: s[64:67] / s[68:71] buffer descriptors of P / Q at the k-tile being loaded, s[72:73] / s[74:75]
    bytes left from there, s76 the k-tile being written, s77 scratch."""

    def __init__(self, GATHER):
        Asm.__init__(self)
        self.GATHER = GATHER
        self.name = "W4_LOAD_%s" % ("GATHER" if GATHER else "PACKED")

    def chunk_regs(self, c):
        return "a[%d:%d]" % (4 * c, 4 * c + 3) if c < 64 else "v[%d:%d]" % (4 * (c - 64), 4 * (c - 64) + 3)

    def load(self, c):
        if c < CHUNKS_P:
            self.e("buffer_load_dwordx4 %s, v%d, s[64:67], 0 offen" % (self.chunk_regs(c), L_VOFFP + c))
        else:
            self.e("buffer_load_dwordx4 %s, v%d, s[68:71], 0 offen" % (self.chunk_regs(c), L_VOFFQ + c - CHUNKS_P))

    def write(self, stage, c):
        self.lds("ds_write_b128 v%d, %s offset:%d" % (L_WR + c, self.chunk_regs(c), stage * (P_STAGE if c < CHUNKS_P else Q_STAGE)))

    def set_cursor(self, src):
        for (d, ext, o) in ((64, 72, 0), (68, 74, 4)):
            for ins in ("s_mov_b32 s%d, s%d" % (d, src + o), "s_mov_b32 s%d, s%d" % (d + 1, src + o + 1),
                        "s_mov_b32 s%d, s%d" % (ext, src + o + 2), "s_mov_b32 s%d, s%d" % (ext + 1, src + o + 3),
                        "s_cmp_lg_u32 s%d, 0" % (ext + 1), "s_cselect_b32 s%d, -1, s%d" % (d + 2, ext),
                        "s_mov_b32 s%d, 0x00020000" % (d + 3)):
                self.e(ins)

    def advance(self):
        """cursor one k-tile on: base += ktile, extent -= ktile (not below zero), num_records = min(extent, 2^32 - 1)"""
        for (d, ext, kt) in ((64, 72, 58), (68, 74, 59)):
            for ins in ("s_add_u32 s%d, s%d, s%d" % (d, d, kt), "s_addc_u32 s%d, s%d, 0" % (d + 1, d + 1),
                        "s_sub_u32 s%d, s%d, s%d" % (ext, ext, kt), "s_subb_u32 s%d, s%d, 0" % (ext + 1, ext + 1),
                        "s_cselect_b32 s%d, 0, s%d" % (ext, ext), "s_cselect_b32 s%d, 0, s%d" % (ext + 1, ext + 1),
                        "s_cmp_lg_u32 s%d, 0" % (ext + 1), "s_cselect_b32 s%d, -1, s%d" % (d + 2, ext)):
                self.e(ins)

    def step(self, stage, check_switch):
        """writes the k-tile s76 into `stage`; its chunks 60..67 and chunks 0..59 of the next k-tile are requested"""
        e = self.e
        for c in range(CHUNKS):
            e("s_waitcnt vmcnt(%d)" % (WINDOW - 1))
            self.write(stage, c)
            if c == LAG:
                # the loads move on to k-tile s76 + 1: of this tile, or the first of the next
                if check_switch:
                    e("s_add_u32 s77, s76, 1")
                    e("s_cmp_eq_u32 s77, s56")
                    e("s_cbranch_scc0 5f")
                    self.set_cursor(48)
                    if self.GATHER:
                        for q in range(CHUNKS_Q):
                            e("v_mov_b32 v%d, v%d" % (L_VOFFQ + q, L_VOFFQ_NEXT + q))
                    e("s_branch 6f")
                    e("5:")
                    self.advance()
                    e("6:")
                else:
                    self.advance()
            self.load(c + WINDOW if c < LAG else c - LAG)
        e("s_waitcnt lgkmcnt(0)")
        self.barrier()

    def generate(self):
        e = self.e
        self.set_cursor(40)
        e("s_bitcmp1_b32 s57, 0")
        e("s_cbranch_scc1 1f")
        self.advance()                       # chunks 0..59 of k-tile 1 are here; the next loads are its last eight
        e("s_branch 2f")
        e("1:")
        # first tile: request chunks 0..59 of k-tile 0, then the generic step writes it into stage 0
        for c in range(WINDOW):
            self.load(c)
        e("s_mov_b32 s76, 0")
        self.step(0, False)
        e("2:")
        e("s_mov_b32 s76, 1")
        e("3:")
        self.step(1, True)
        e("s_add_u32 s76, s76, 1")
        self.step(0, False)
        e("s_add_u32 s76, s76, 1")
        e("s_cmp_le_u32 s76, s56")
        e("s_cbranch_scc1 3b")
        e("s_waitcnt vmcnt(0)")
        return self.L

    def clobbers(self):
        return ["s%d" % i for i in range(64, 78)] + ["scc", "memory"]


# ================================================================================================ four symmetric waves, 256 x 384
QW_STAGE = 49152         # bytes of one Q stage of the wide tile (384 rows x 64 k)
SHORT = (5, 4, 3, 2)     # column blocks of a wave in a tile of fewer rows
D_VP, D_VQ, D_VQ_NEXT, D_AT = 208, 216, 228, 240              # this lane's offsets of the wave's 8 chunks of P, 12 of Q, the next tile's Q, of D


class Tail(Asm):
    """The epilogue of the kernels below, a part of their statements: the compiler, given 256 accumulators or more to read, kept 16 to 40
    of them in scratch memory, waited there for its own stores, and for every second load of C.  A wave's results are groups of 64 (m) x 16
    (n), two accumulators of 8 per lane; they leave as whole 128-byte lines without the LDS:
      1. Pairs of row blocks change lane rows (v_permlane16_swap_b32: lane rows 1 and 3 of block i with lane rows 0 and 2 of block
         i + 1): a lane then holds m = 8 (grp / 2) .. + 7 of block i + (grp & 1), 16 bytes, and the four lane rows of one n hold 64
         consecutive bytes.
      2. Two such pairs (blocks i, i + 1 and i + 2, i + 3) are merged across the halves of a lane row (a DPP rotation by eight
         lanes, written to one half only): one store carries both pairs of eight n, 128 consecutive bytes per n.
    The first store of a group carries n = 0-7 (lanes 0-7 of a lane row the first pair, lanes 8-15 the second), the second n = 8-15 (the
    other way round).  s32 / s33: address of the wave's first element of D, s34: bytes from there to the end of its rows, s35: bytes of 16
    rows, s38: alpha.  v[at + 2 h], v[at + 2 h + 1]: this lane's offset of the first and the second store of group (0, h), outside any buffer
    where its columns do not exist.  Rows that do not exist lie past s34.  All stores are issued always: the waits of the next statement
    count them."""

    def valu(self, text, dst, cross=()):
        """a vector instruction that writes the registers `dst`; the cross-lane reads `cross` need two others behind their writer"""
        behind = min([self.count - self.written.get(v, -9) for v in cross] + [3])
        if behind <= 2:
            self.e("s_nop %d" % (2 - behind))
            self.count += 3 - behind
        self.e(text)
        for v in dst:
            self.written[v] = self.count
        self.count += 1

    def swap(self, a, b):
        self.valu("v_permlane16_swap_b32 v%d, v%d" % (a, b), (a, b), (a, b))

    def dpp(self, dst, src, ctrl, bank):
        self.valu("v_mov_b32_dpp v%d, v%d %s row_mask:0xf bank_mask:0x%x" % (dst, src, ctrl, bank), (dst,), (src,))

    def descriptor(self, d, address):
        for ins in ("s_mov_b32 s%d, s%d" % (d, address), "s_mov_b32 s%d, s%d" % (d + 1, address + 1), "s_mov_b32 s%d, s34" % (d + 2),
                    "s_mov_b32 s%d, 0x00020000" % (d + 3)):
            self.e(ins)

    def accumulators(self, group, t, scale):
        """the 16 results of a group, as registers (copied to t .. t + 15 from the accumulation registers), times alpha"""
        src = t
        if group < 16:
            for r in range(16):
                self.valu("v_accvgpr_read_b32 v%d, a%d" % (t + r, 16 * group + r), (t + r,))
        else:
            src = 16 * (group - 16)
        if scale:
            for r in range(16):
                self.valu("v_mul_f32 v%d, s38, v%d" % (t + r, src + r), (t + r,))
            src = t
        return src

    def store_group(self, src, t, at):
        """16 results to D; t .. t + 3 and t + 16 .. t + 19 carry the stores"""
        for k in range(8):
            self.valu("v_cvt_pk_bf16_f32 v%d, v%d, v%d" % (t + k, src + 2 * k, src + 2 * k + 1), (t + k,))
        for a in (t, t + 1, t + 4, t + 5):
            self.swap(a, a + 2)
        for k in range(4):
            self.valu("v_mov_b32 v%d, v%d" % (t + 16 + k, t + k), (t + 16 + k,))
        for k in range(4):
            self.dpp(t + k, t + 4 + k, "row_ror:8", 0xC)
        for k in range(4):
            self.dpp(t + 16 + k, t + 4 + k, "row_ror:8", 0x3)
        self.e("buffer_store_dwordx4 %s, v%d, s[92:95], 0 offen nt" % (vr(t, 4), at))
        self.e("buffer_store_dwordx4 %s, v%d, s[92:95], 0 offen nt" % (vr(t + 16, 4), at + 1))
        self.count += 2

    def next_rows(self, at, n):
        for k in range(n):
            self.valu("v_add_u32 v%d, s35, v%d" % (at + k, at + k), (at + k,))


class Wide(Mult, Tail):
    """gemm_bf16_w4d_kernel: tile 256 (m) x 384 (n) x 64 (k), four waves that all do both jobs.  Wave w multiplies columns
    [96 w, 96 w + 96) of the tile like a multiplying wave above (same fragment reads, same MFMA order) and loads a quarter
    of every k-tile -- chunks 8 w .. 8 w + 7 of P and 12 w .. 12 w + 11 of Q, 20 KiB -- straight into the LDS
    (buffer_load_dwordx4 ... lds), so the two stages fill all 160 KiB and there is no epilogue scratch.

    The rows of Q that a wave loads are the rows it multiplies: nobody else reads them.  So the Q part of a stage needs no
    barrier: in step g (stage p = g & 1) the wave reads its fragments of Q for the second k-step first and, with them in
    registers, loads the Q rows of k-tile g + 2 into stage p (from MFMA `qfirst` on, every `qevery` MFMAs), with most of
    two steps to land.  P is
    read by all waves: behind MFMA 179 the wave waits for its loads of k-tile g + 1 (all but the twelve newest, which are
    the Q rows of k-tile g + 2: loads complete in order) and for its fragment reads of stage p, then the barrier; the P
    rows of k-tile g + 2 follow, `pre` of them behind MFMAs 180, 183, ... and the rest behind MFMAs first, first + every, ...
    of the next step.  Loads are in flight all the time, also across the barrier.

    The two cursors (buffer descriptors of P and of Q at the k-tile being loaded) move on where their loads begin; when
    the tile has no k-tile g + 2 they switch to the next tile's first one.

    s[40:47] this tile's cursor at k-tile 0, s[48:55] the next tile's (empty buffers when there is none), s56 k-tiles
    (even), s57 bit 0: first tile of the work-group, s58 / s59 bytes per k-tile of P / Q, s60 LDS address of the stages,
    s61 / s62 of the wave's first chunk of P / Q in stage 0, s63 bytes from s60 to the wave's rows of Q.  Working registers as in the loader above.

    Short tiles: a tile of at most 64 n rows, n one of SHORT, has bit 14 - n of s57 set, and wave w multiplies rows [16 n w, 16 n w + 16 n) of
    it, n column blocks instead of six: the steps are the same with fewer multiplies.  Its loads of Q from the 2 n-th on read zeros.

    State from statement to statement: stage 0 holds k-tile 0 of the tile, visible to all waves; the rows of Q and P of k-tile 1 are
    in flight into stage 1, and behind them the 48 stores of the tile before; the Q offsets of the tile are in v[D_VQ ...], of
    gathered rows those of the next in v[D_VQ_NEXT ...].  Epilogue as
    in class Tail; s57 bit 2: alpha is not 1.  Three macros: what every tile starts with, the first tile's loads and the loop, the first two
    steps, which come in front of the loop but stand behind it, and the epilogue."""

    LOADS_P, LOADS_Q = 8, 12

    def __init__(self, PKM, GATHER):
        Mult.__init__(self, PKM)
        self.GATHER = GATHER
        self.parts = []
        self.name = "W4D_%s_%s" % ("PKM" if PKM else "PKC", "GATHER" if GATHER else "PACKED")

    # which: 0 = P (descriptor s[64:67], bytes left s[72:73]), 1 = Q (s[68:71], s[74:75])
    def set_cursor(self, src, which):
        d, ext, o = ((64, 72, 0), (68, 74, 4))[which]
        for ins in ("s_mov_b32 s%d, s%d" % (d, src + o), "s_mov_b32 s%d, s%d" % (d + 1, src + o + 1),
                    "s_mov_b32 s%d, s%d" % (ext, src + o + 2), "s_mov_b32 s%d, s%d" % (ext + 1, src + o + 3),
                    "s_cmp_lg_u32 s%d, 0" % (ext + 1), "s_cselect_b32 s%d, -1, s%d" % (d + 2, ext),
                    "s_mov_b32 s%d, 0x00020000" % (d + 3)):
            self.e(ins)

    def advance(self, which):
        d, ext, kt = ((64, 72, 58), (68, 74, 59))[which]
        for ins in ("s_add_u32 s%d, s%d, s%d" % (d, d, kt), "s_addc_u32 s%d, s%d, 0" % (d + 1, d + 1),
                    "s_sub_u32 s%d, s%d, s%d" % (ext, ext, kt), "s_subb_u32 s%d, s%d, 0" % (ext + 1, ext + 1),
                    "s_cselect_b32 s%d, 0, s%d" % (ext, ext), "s_cselect_b32 s%d, 0, s%d" % (ext + 1, ext + 1),
                    "s_cmp_lg_u32 s%d, 0" % (ext + 1), "s_cselect_b32 s%d, -1, s%d" % (d + 2, ext)):
            self.e(ins)

    def dma_p(self, stage, u):
        self.e("s_add_u32 m0, s61, %d" % (stage * P_STAGE + u * 1024))
        self.e("s_nop 0")
        self.e("buffer_load_dwordx4 v%d, s[64:67], 0 offen lds" % (D_VP + u))

    def dma_q(self, stage, q):
        self.e("s_add_u32 m0, s62, %d" % (stage * QW_STAGE + q * 1024))
        self.e("s_nop 0")
        self.e("buffer_load_dwordx4 v%d, s[68:71], 0 offen lds" % (D_VQ + q))

    def move_on(self, which, check_switch):
        """cursor `which` to k-tile s76 + 2 (of this tile, or the first of the next)"""
        e = self.e
        if check_switch:
            e("s_add_u32 s77, s76, 2")
            e("s_cmp_eq_u32 s77, s56")
            e("s_cbranch_scc0 5f")
            self.set_cursor(48, which)
            if self.GATHER and which == 1:
                for q in range(12):
                    e("v_mov_b32 v%d, v%d" % (D_VQ + q, D_VQ_NEXT + q))
            e("s_branch 6f")
            e("5:")
            self.advance(which)
            e("6:")
        else:
            self.advance(which)

    def step(self, p, start=False, blocks=6):
        """`blocks`: column blocks of a wave"""
        after = {}

        def at(m, fn):
            after.setdefault(m, []).append(fn)

        count, behind = 32 * blocks, 30 * blocks - 1         # MFMAs; the one behind which two of the four slots of P's fragments are free again
        pre, first, every, qfirst, qevery = (OPTS[k] for k in ("pre", "first", "every", "qfirst", "qevery"))
        if blocks < 6:                           # all twelve loads of Q go out (the next tile may have the rows), closer together
            every, qfirst = min(every, blocks - 1), min(qfirst, 4 * blocks)
            qevery = (behind - 1 - qfirst) // (self.LOADS_Q - 1)
        assert 1 <= pre <= 4 and first + every * (self.LOADS_P - pre - 1) < qfirst
        assert qfirst >= 8 and qfirst + qevery * (self.LOADS_Q - 1) < behind
        # the rest of the P rows of k-tile g + 1, into the other stage
        if not start:                        # of the first k-tile they are out in front of the epilogue
            for n, u in enumerate(range(pre, self.LOADS_P)):
                at(first + every * n, lambda u=u: self.dma_p(1 - p, u))
        # the fragments of Q of k-step 1 first: with them in registers the wave's Q rows of this stage are free
        for j in range(blocks):
            at(j, lambda j=j: self.read_B(p, 1, j))
        # this wave's Q rows of k-tile g + 2, into the stage being multiplied
        at(qfirst, lambda: self.need(*[("B", 1, j) for j in range(blocks)]))
        at(qfirst, lambda: self.move_on(1, p == 0))
        for q in range(self.LOADS_Q):
            at(qfirst + qevery * q, lambda q=q: self.dma_q(p, q))
        for a in range(4, 32):
            at(blocks * (a - 3) - 1, lambda a=a: self.read_A(p, a))

        def barrier():
            if start:                            # behind the first tile's loads, or the stores of the tile before
                self.e("s_bitcmp1_b32 s57, 0")
                self.e("s_cbranch_scc0 7f")
                self.e("s_waitcnt vmcnt(%d)" % self.LOADS_Q)
                self.e("7:")
                self.e("s_waitcnt vmcnt(%d)" % (self.LOADS_Q + 48))
            else:
                self.e("s_waitcnt vmcnt(%d)" % self.LOADS_Q)
            self.lds_drain()
            self.barrier()
            self.tail_reads(1 - p, 0, blocks)
        at(behind, barrier)
        at(behind + 1, lambda: self.move_on(0, p == 0))
        for u in range(pre):
            at(behind + 1 + blocks * u // 2, lambda u=u: self.dma_p(p, u))
        at(behind + blocks, lambda: self.tail_reads(1 - p, 1))
        at(behind + 2 * blocks, lambda: self.tail_reads(1 - p, 2))
        for m in range(count):
            s, rem = divmod(m, 16 * blocks)
            i, j = divmod(rem, blocks)
            if i & 1:
                j = blocks - 1 - j               # one operand stays from each MFMA to the next: 0.8 % less time at the card's power limit
            a = s * 16 + i
            self.need(("A", a % 4), ("B", s, j))
            self.e("v_mfma_f32_16x16x32_bf16 %s, %s, %s, %s" % (self.acc(i, j), vr(M_AF + (a % 4) * 4, 4), vr(M_BF + s * 24 + j * 4, 4), "0" if start and s == 0 else self.acc(i, j)))
            for fn in after.get(m, []):
                fn()

    def addresses(self):
        """fragment read addresses of this lane, from its number (kept out of the compiler's hands: it has eight registers across the
        statement): row l % 16, chunk 4 s + l / 16 of a k-contiguous operand, four k-rows from 8 (l / 16) on of a k-major one"""
        e = self.e
        l15, g4, sw, t = M_BF, M_BF + 1, M_BF + 2, M_BF + 3
        e("v_mbcnt_lo_u32_b32 v%d, -1, 0" % t)
        e("v_mbcnt_hi_u32_b32 v%d, -1, v%d" % (t, t))
        e("v_and_b32 v%d, 15, v%d" % (l15, t))
        e("v_lshrrev_b32 v%d, 4, v%d" % (g4, t))
        if self.PKM:                             # k-row 8 g4 + l15 / 4, rows 16 i + 4 (l15 % 4), swizzled as kmajor_swizzle does
            e("v_lshrrev_b32 v%d, 2, v%d" % (sw, l15))
            e("v_lshl_add_u32 v%d, v%d, 3, v%d" % (t, g4, sw))
            e("v_lshlrev_b32 v%d, 5, v%d" % (sw, sw))
            e("v_and_b32 v%d, 0x60, v%d" % (sw, sw))
            e("v_and_b32 v%d, 1, v%d" % (t + 1, g4))
            e("v_lshlrev_b32 v%d, 4, v%d" % (t + 1, t + 1))
            e("v_xor_b32 v%d, v%d, v%d" % (sw, sw, t + 1))
            e("v_lshlrev_b32 v%d, 9, v%d" % (t, t))
            e("v_add_u32 v%d, s60, v%d" % (t, t))
            e("v_and_b32 v%d, 3, v%d" % (t + 1, l15))
            e("v_lshlrev_b32 v%d, 2, v%d" % (t + 1, t + 1))
            for n in range(8):
                e("v_add_u32 v%d, %d, v%d" % (M_ARD + n, 16 * n, t + 1))
                e("v_xor_b32 v%d, v%d, v%d" % (M_ARD + n, M_ARD + n, sw))
                e("v_lshl_add_u32 v%d, v%d, 1, v%d" % (M_ARD + n, M_ARD + n, t))
        e("v_lshrrev_b32 v%d, 1, v%d" % (sw, l15))
        e("v_lshlrev_b32 v%d, 7, v%d" % (l15, l15))
        e("v_add_u32 v%d, s60, v%d" % (l15, l15))
        for s in range(2):
            e("v_add_u32 v%d, %d, v%d" % (t, 4 * s, g4))
            e("v_xor_b32 v%d, v%d, v%d" % (t, t, sw))
            e("v_lshl_add_u32 v%d, v%d, 4, v%d" % (t, t, l15))
            if not self.PKM:
                e("v_mov_b32 v%d, v%d" % (M_ARD + s, t))
            e("v_add_u32 v%d, s63, v%d" % (M_BRD + 2 * s, t))
            e("v_add_u32 v%d, %d, v%d" % (M_BRD + 2 * s + 1, QW_STAGE, M_BRD + 2 * s))

    def generate(self):
        e = self.e
        self.addresses()
        self.set_cursor(40, 0)
        self.set_cursor(40, 1)
        e("s_mov_b32 s76, 0")
        e("s_bitcmp1_b32 s57, 0")
        e("s_cbranch_scc0 2f")
        self.part("HEAD")
        for u in range(self.LOADS_P):        # first tile: k-tile 0, then the first loads of k-tile 1
            self.dma_p(0, u)
        for q in range(self.LOADS_Q):
            self.dma_q(0, q)
        e("s_waitcnt vmcnt(0)")
        e("s_barrier")
        self.advance(0)
        self.advance(1)
        for u in range(OPTS["pre"]):
            self.dma_p(1, u)
        for q in range(self.LOADS_Q):
            self.dma_q(1, q)
        e("s_branch 12f")
        e("3:")
        self.two_steps(False)
        e("s_cbranch_scc1 3b")
        e("s_branch 9f")
        self.part("ASM")
        e("12:")                             # the rest of the first tile's P
        for u in range(OPTS["pre"], self.LOADS_P):
            self.dma_p(1, u)
        e("s_branch 4f")
        e("2:")
        self.advance(0)
        self.advance(1)
        e("4:")
        for blocks in SHORT:
            e("s_bitcmp1_b32 s57, %d" % (14 - blocks))
            e("s_cbranch_scc1 %df" % (30 + blocks))
        for which in range(3):
            self.tail_reads(0, which)
        self.two_steps(True)                 # the first two k-tiles start the sums
        e("s_cbranch_scc1 3b")
        e("s_branch 9f")
        for blocks in SHORT:
            e("%d:" % (30 + blocks))
            for which in range(3):
                self.tail_reads(0, which, blocks)
            self.two_steps(True, blocks)
            e("s_cbranch_scc0 9f")
            e("%d:" % (40 + blocks))
            self.two_steps(False, blocks)
            e("s_cbranch_scc1 %db" % (40 + blocks))
            e("s_branch 9f")
        e("9:")
        e("s_waitcnt lgkmcnt(0)")
        for u in range(OPTS["pre"], self.LOADS_P):
            self.dma_p(1, u)
        self.descriptor(92, 32)
        for _ in range(3):
            e("s_nop 7")
        e("s_bitcmp1_b32 s57, 2")
        e("s_cbranch_scc1 10f")
        self.epilogue(False)
        e("s_branch 11f")
        e("10:")
        self.epilogue(True)
        e("11:")
        self.part("END")
        return self.parts

    def part(self, name):
        """the lines since the last part, as a macro of their own"""
        self.parts.append(("%s_%s" % (self.name, name), self.L))
        self.L = []

    def two_steps(self, start, blocks=6):
        self.loop_head_state(blocks)
        self.step(0, start, blocks)
        self.loop_head_state(blocks)
        self.step(1, False, blocks)
        self.e("s_add_u32 s76, s76, 2")
        self.e("s_cmp_lt_u32 s76, s56")

    def epilogue(self, scale):
        self.count, self.written = 0, {}
        for n in range(24):
            j, h = divmod(n, 4)
            if h == 0 and j:
                self.next_rows(D_AT, 8)
            t = M_BF + 24 * (n & 1)
            self.store_group(self.accumulators(6 * h + j, t, scale), t, D_AT + 2 * h)

    def clobbers(self):
        return ["v%d" % i for i in range(D_VP)] + ["a%d" % i for i in range(256)] + ["s%d" % i for i in range(64, 78)] + \
               ["s%d" % i for i in range(92, 96)] + ["m0", "scc", "memory"]


# ================================================================================================ four waves, ragged reduction
R_SLICE, R_SLOTS = 32768, 5                                   # bytes of a slice of both operands (2 x 32 k x 256 rows), slices in the LDS
R_C, R_PRD, R_QRD, R_VP, R_VQ, R_AT, R_CAT = 64, 192, 200, 208, 212, 216, 220
R_MAP, R_MAPN, R_MAP0, R_MAP1, R_SEL, R_SEL0, R_KB, R_COL, R_T = 224, 225, 226, 227, 228, 229, 230, 231, 233      # gathered k-rows


class Ring(Tail):
    """gemm_bf16_w4k_kernel: tile 256 (m) x 256 (n), both operands k-major, four waves as 2 x 2, each 128 x 128 (8 x 8 blocks, all 256
    accumulators in a[0:255]).  The stream is one of slices of 32 k, 16 KiB of P behind 16 KiB of Q, in a ring of five slots that runs on
    across tiles; every wave loads a quarter of each slice (eight chunks of 1 KiB, two k-rows each) straight into the LDS.

    Slice s, two halves of 32 MFMAs, row block by row block: columns 0-3, then 4-7.  All operands of a slice are in registers once, and
    each is read again right behind its last MFMA: those of columns 4-7 (of this slice) in the first half, between the halves the one
    barrier, then those of columns 0-3 and row by row those of P (of the next slice), 28 MFMAs in front of their use.  In front of the
    barrier the wave waits for its loads of slice s + 1, and for its reads of slice s, whose slot takes the loads of slice s + 5: three to
    four slices, 96 to 128 KiB, are in flight at any time.

    C has 128 registers: its tile is read in the first eight slices, four lines of 16 rows each, and has the rest of the tile's multiplies
    to arrive; the stores of D go out behind the last multiply and drain under the next tile's.

    s[40:47] the cursor (as for the loader above) of this tile, at slice 0 for the work-group's first tile and at slice 5 for any other,
    s[48:55] the next tile's at slice 0, s56 slices (at least `least`), s57 bit 0: first tile, bit 2: alpha is not 1, s58 / s59 bytes per
    slice of P / Q, s60 byte offset of slice 0's slot, s61 / s62 LDS address of the wave's rows of P / Q in slot 0, s63 of its first chunk.
    s[32:39] as w4_output gives them (D, bytes, bytes of 16 rows, C, alpha, beta).  Working registers: s[64:75] as in the loader above,
    s76 the slot, s77 scratch, s78 where the loads go, s79 the slice, s[84:87] C's descriptor, s[92:95] D's.

    State from statement to statement: slices 0-4 of the tile are on their way or there, slice 0 visible to all waves; behind them the 32
    stores of the tile before.

    GATHER: the k-rows of P are scattered over a source, by a map.  The cursor of P stays at the tile's first column of the source; s42 the
    source's bytes from there, s43 its rows, s58 bytes of one of them (s50 and s51 of the next tile).  s[80:83] / s[88:91] buffers over this / the
    next tile's map.  A wave's rows of eight slices, 8 r + j the j-th row of the r-th slice, are held one per lane, as the byte offset of the
    source's row (R_MAP; a row that does not exist, outside any buffer), each load takes its two from there by a ds_bpermute, and the
    offsets of the next eight slices are on their way (R_MAPN; of the next tile's first sixteen R_MAP0 and R_MAP1, which therefore are asked
    for a tile ahead: a load between two tiles would wait for the stores in front of it).  R_SEL: where the slice's first row is, four bytes a
    lane; R_KB, R_SEL0, R_COL: this lane's place in the map, in a slice, and column of the source, of even and of odd loads.  s96 bytes of the
    map to the eight slices behind those held, s97 slices to them.  A tile has eight slices at least.  State: R_MAP the tile's first eight slices, R_SEL at
    the sixth of them, R_MAPN the next eight."""

    LOADS, STORES = 8, 32

    def __init__(self, HAS_C, GATHER=False):
        Asm.__init__(self)
        self.C, self.GATHER = HAS_C, GATHER
        self.least = 8 if HAS_C or GATHER else 5           # slices a tile has at least
        self.head = 8 if HAS_C else 4            # slices in front of the loop
        self.name = "W4K_%s%s" % ("C" if HAS_C else "NOC", "_GATHER" if GATHER else "")

    def set_p(self, src):
        """the buffer of P, gathered"""
        for n, ins in enumerate(("s%d" % src, "s%d" % (src + 1), "s%d" % (src + 2), "0x00020000")):
            self.e("s_mov_b32 s%d, %s" % (64 + n, ins))

    def load_map(self, dst, buffer, at=None):
        self.e("buffer_load_dword v%d, v%d, s[%d:%d], 0 offen" % (dst, R_KB if at is None else at, buffer, buffer + 3))

    def hold(self, raw, buffer, at=None):
        """the offsets of the rows `raw`, entries of the map from byte `at` (a register) or 0 on"""
        e = self.e
        where = R_KB
        if at:
            e("v_add_u32 v%d, %s, v%d" % (R_T, at, R_KB))
            where = R_T
        e("v_cmp_gt_u32 vcc, s%d, v%d" % (buffer + 2, where))
        e("v_min_u32 v%d, s43, v%d" % (R_MAP, raw))
        e("v_mul_lo_u32 v%d, v%d, s58" % (R_MAP, R_MAP))
        e("v_mov_b32 v%d, 0xfffffc00" % R_T)
        e("v_cndmask_b32 v%d, v%d, v%d, vcc" % (R_MAP, R_T, R_MAP))

    def next_rows_of_map(self):
        """in front of the loads of slice s79 + 5: its rows among those held"""
        e = self.e
        e("s_sub_u32 s97, s97, 1")
        e("s_add_u32 s77, s79, %d" % R_SLOTS)
        e("s_cmp_eq_u32 s77, s56")
        e("s_cbranch_scc1 21f")
        e("s_cmp_eq_u32 s97, 0")
        e("s_cbranch_scc0 23f")
        self.hold(R_MAPN, 80, "s96")             # the next eight slices of the tile
        e("s_mov_b32 s97, 8")
        e("s_add_u32 s96, s96, 1024")
        e("s_add_u32 s77, s77, 8")
        e("s_cmp_lt_u32 s77, s56")               # and those behind them, if there are any
        e("s_cbranch_scc0 23f")
        e("v_add_u32 v%d, s96, v%d" % (R_T, R_KB))
        self.load_map(R_MAPN, 80, R_T)
        e("s_branch 23f")
        e("21:")                                 # the next tile's first eight
        e("s_waitcnt vmcnt(%d)" % (3 * self.LOADS))        # asked for at least three slices ago
        self.hold(R_MAP0, 88)
        e("v_mov_b32 v%d, v%d" % (R_MAPN, R_MAP1))
        e("v_mov_b32 v%d, v%d" % (R_SEL, R_SEL0))
        e("s_mov_b32 s97, 16")                   # no more than five of them are loaded in this statement
        e("23:")

    def take_rows(self, u):
        self.lds("ds_bpermute_b32 v%d, v%d, v%d offset:%d" % (R_VP + u, R_SEL, R_MAP, 8 * u))

    def add_column(self, u):
        self.e("v_add_u32 v%d, v%d, v%d" % (R_VP + u, R_COL + (u & 1), R_VP + u))

    def next_slice_of_map(self):
        self.e("v_add_u32 v%d, 32, v%d" % (R_SEL, R_SEL))

    set_cursor, advance = Wide.set_cursor, Wide.advance

    def need(self, *keys):
        n = max(self.prod.get(k, -1) for k in keys)
        if n > self.known_done:
            after = min(self.issued - 1 - n, 15)
            self.e("s_waitcnt lgkmcnt(%d)" % after)
            self.known_done = self.issued - 1 - after

    def read(self, which, n):
        """operand n (16 rows) of P or Q, both halves of its 32 k"""
        dst = 4 * n + (0 if which == "P" else 32)
        addr = (R_PRD if which == "P" else R_QRD) + n
        self.lds("ds_read_b64_tr_b16 %s, v%d" % (vr(dst, 2), addr))
        self.lds("ds_read_b64_tr_b16 %s, v%d offset:%d" % (vr(dst + 2, 2), addr, 4 * 512), (which, n))

    def dma(self, u):
        self.e("s_add_u32 m0, s78, %d" % ((u % 4) * 1024 + (16384 if u >= 4 else 0)))
        self.e("s_nop 0")
        self.e("buffer_load_dwordx4 v%d, s[%s], 0 offen lds" % (R_VP + u, "64:67" if u < 4 else "68:71"))

    def load_c(self, j, k):
        self.e("buffer_load_dwordx4 %s, v%d, s[84:87], 0 offen nt" % (vr(R_C + 16 * j + 4 * k, 4), R_CAT + k))
        self.e("v_add_u32 v%d, s35, v%d" % (R_CAT + k, R_CAT + k))

    def move_on(self):
        """the cursor, which stands at slice s79 + 5 of this tile, to the next tile's first one if there is none"""
        self.e("s_add_u32 s77, s79, %d" % R_SLOTS)
        self.e("s_cmp_eq_u32 s77, s56")
        self.e("s_cbranch_scc0 6f")
        if self.GATHER:
            self.set_p(48)
        else:
            self.set_cursor(48, 0)
        self.set_cursor(48, 1)
        self.e("6:")

    def vm_count(self, s):
        """of the operations behind the loads of slice s + 1, how many may be in flight at the barrier of slice s < head"""
        ops = []
        for t in range(1, R_SLOTS):
            ops += ["L%d" % t] * self.LOADS
        ops += ["S"] * self.STORES + (["M"] * 2 if self.GATHER else [])
        for t in range(s + 1):
            ops += ["C"] * (4 if self.C else 0)
            if t < s:
                ops += ["L%d" % (t + R_SLOTS)] * self.LOADS
        last = max(n for n, o in enumerate(ops) if o == "L%d" % (s + 1))
        return min(63, len(ops) - 1 - last)

    def slice(self, s):
        """s: the slice's number, or None in the loop"""
        after = {}

        def at(m, fn):
            after.setdefault(m, []).append(fn)

        e = self.e
        for n in range(4):
            at(2 * n, lambda n=n: self.read("Q", 4 + n))
        # the read addresses move to the next slot (the reads of this one are out)
        at(8, lambda: e("s_add_u32 s78, s63, s76"))
        at(8, lambda: e("s_mov_b32 s77, s76"))
        at(9, lambda: e("s_add_u32 s76, s76, %d" % R_SLICE))
        at(9, lambda: e("s_cmp_eq_u32 s76, %d" % (R_SLOTS * R_SLICE)))
        at(9, lambda: e("s_cselect_b32 s76, 0, s76"))
        at(9, lambda: e("s_sub_u32 s77, s76, s77"))
        for n in range(16):
            at(10 + n, lambda n=n: e("v_add_u32 v%d, s77, v%d" % (R_PRD + n, R_PRD + n)))
        if self.GATHER:
            at(7, self.next_rows_of_map)
            for u in range(4):
                at(12 + 3 * u, lambda u=u: self.take_rows(u))
                at(32 + u // 2, lambda u=u: self.add_column(u))
            at(35, self.next_slice_of_map)
        if self.C and s is not None and s < 8:
            for k in range(4):
                at(11 + 4 * k, lambda k=k: self.load_c(s, k))

        def barrier():
            e("s_waitcnt vmcnt(%d)" % (self.LOADS * 3 if s is None else self.vm_count(s)))
            self.lds_drain()
            self.barrier()
        at(31, barrier)
        for n in range(4):
            at(32 + n, lambda n=n: self.read("Q", n))
        for i in range(8):
            at(35 + 4 * i, lambda i=i: self.read("P", i))
        at(34, self.move_on)
        for u in range(self.LOADS):
            at(36 + 3 * u, lambda u=u: self.dma(u))
        if not self.GATHER:
            at(58, lambda: self.advance(0))
        at(59, lambda: self.advance(1))
        at(60, lambda: e("s_add_u32 s79, s79, 1"))
        for m in range(64):
            half, rem = divmod(m, 32)
            i, j = divmod(rem, 4)
            if i & 1:
                j = 3 - j                        # one operand stays from each MFMA to the next
            j += 4 * half
            acc = "a[%d:%d]" % (16 * (8 * (i // 4) + j) + 4 * (i % 4), 16 * (8 * (i // 4) + j) + 4 * (i % 4) + 3)
            self.need(("P", i), ("Q", j))
            self.e("v_mfma_f32_16x16x32_bf16 %s, %s, %s, %s" % (acc, vr(4 * i, 4), vr(32 + 4 * j, 4), "0" if s == 0 else acc))
            for fn in after.get(m, []):
                fn()

    def entry_state(self):
        """the reads in flight at the start of a slice, as the second half of the one before leaves them"""
        self.issued, self.known_done, self.prod = 0, -1, {}
        keep, self.L = self.L, []
        for n in range(4):
            self.read("Q", n)
        for i in range(8):
            self.read("P", i)
        self.L = keep

    def addresses(self):
        """fragment read addresses of this lane in the slot s60: k-row 8 g4 + l15 / 4, rows 16 i + 4 (l15 % 4), swizzled as
        kmajor_swizzle does"""
        e = self.e
        l15, g4, sw, t, row = 0, 1, 2, 3, 4
        e("v_mbcnt_lo_u32_b32 v%d, -1, 0" % t)
        e("v_mbcnt_hi_u32_b32 v%d, -1, v%d" % (t, t))
        e("v_and_b32 v%d, 15, v%d" % (l15, t))
        e("v_lshrrev_b32 v%d, 4, v%d" % (g4, t))
        e("v_lshrrev_b32 v%d, 2, v%d" % (sw, l15))
        e("v_lshl_add_u32 v%d, v%d, 3, v%d" % (t, g4, sw))
        e("v_lshlrev_b32 v%d, 5, v%d" % (sw, sw))
        e("v_and_b32 v%d, 1, v%d" % (row, g4))
        e("v_lshlrev_b32 v%d, 4, v%d" % (row, row))
        e("v_xor_b32 v%d, v%d, v%d" % (sw, sw, row))
        e("v_lshlrev_b32 v%d, 9, v%d" % (t, t))
        e("v_add_u32 v%d, s60, v%d" % (t, t))
        e("v_and_b32 v%d, 3, v%d" % (row, l15))
        e("v_lshlrev_b32 v%d, 2, v%d" % (row, row))
        for n in range(8):
            e("v_add_u32 v%d, %d, v%d" % (R_PRD + n, 16 * n, row))
            e("v_xor_b32 v%d, v%d, v%d" % (R_PRD + n, R_PRD + n, sw))
            e("v_lshl_add_u32 v%d, v%d, 1, v%d" % (R_PRD + n, R_PRD + n, t))
            e("v_add_u32 v%d, s62, v%d" % (R_QRD + n, R_PRD + n))
            e("v_add_u32 v%d, s61, v%d" % (R_PRD + n, R_PRD + n))

    def generate(self):
        e = self.e
        self.addresses()
        if self.GATHER:
            self.set_p(40)
        else:
            self.set_cursor(40, 0)
        self.set_cursor(40, 1)
        if self.C:
            for n, ins in enumerate(("s36", "s37", "s34", "0x00020000")):
                e("s_mov_b32 s%d, %s" % (84 + n, ins))
        e("s_mov_b32 s76, s60")
        e("s_mov_b32 s79, 0")
        if self.GATHER:
            e("s_mov_b32 s96, 1024")
            e("s_mov_b32 s97, 4")                # slices 5, 6 and 7 are held; counted down in front of each
        e("s_bitcmp1_b32 s57, 0")
        e("s_cbranch_scc0 2f")
        if self.GATHER:
            self.load_map(R_MAP0, 80)
            e("v_add_u32 v%d, s96, v%d" % (R_T, R_KB))
            self.load_map(R_MAPN, 80, R_T)
            e("s_waitcnt vmcnt(0)")
            self.hold(R_MAP0, 80)
            e("v_mov_b32 v%d, v%d" % (R_SEL, R_SEL0))
        for t in range(R_SLOTS):                 # first tile (its first slot is slot 0)
            e("s_add_u32 s78, s63, %d" % (t * R_SLICE))
            if self.GATHER:
                for u in range(4):
                    self.take_rows(u)
                e("s_waitcnt lgkmcnt(0)")
                for u in range(4):
                    self.add_column(u)
                self.next_slice_of_map()
            for u in range(self.LOADS):
                self.dma(u)
            if not self.GATHER:
                self.advance(0)
            self.advance(1)
        e("s_waitcnt vmcnt(0)")
        e("s_barrier")
        e("2:")
        if self.GATHER:
            self.load_map(R_MAP0, 88)
            e("v_add_u32 v%d, s96, v%d" % (R_T, R_KB))
            self.load_map(R_MAP1, 88, R_T)
        for n in range(4):
            self.read("Q", n)
        for i in range(8):
            self.read("P", i)
        for s in range(self.head):
            self.entry_state()
            self.slice(s)
        e("s_cmp_lt_u32 s79, s56")
        e("s_cbranch_scc0 4f")
        e("3:")
        self.entry_state()
        self.slice(None)
        e("s_cmp_lt_u32 s79, s56")
        e("s_cbranch_scc1 3b")
        e("4:")
        e("s_waitcnt lgkmcnt(0)")
        self.descriptor(92, 32)
        if self.C:                               # C is here: 8 loads went out behind it for each slice from the eighth on
            e("s_cmp_ge_u32 s56, 11")
            e("s_cbranch_scc1 5f")
            e("s_waitcnt vmcnt(%d)" % self.LOADS)
            e("5:")
            e("s_waitcnt vmcnt(%d)" % (4 * self.LOADS))
        for _ in range(3):
            e("s_nop 7")
        e("s_bitcmp1_b32 s57, 2")
        e("s_cbranch_scc1 10f")
        self.epilogue(False)
        e("s_branch 11f")
        e("10:")
        self.epilogue(True)
        e("11:")
        return self.L

    def add_c(self, src, c):
        """beta C on the 16 results from src on; c .. c + 3 and c + 4 .. c + 7: the lines' halves as they were loaded, 16 bytes of each
        row in a lane.  The swap undoes what the one in front of a store does"""
        for a in (c, c + 1, c + 4, c + 5):
            self.swap(a, a + 2)
        for k in range(8):
            for half in range(2):
                self.valu(("v_and_b32 v60, 0xffff0000, v%d" if half else "v_lshlrev_b32 v60, 16, v%d") % (c + k), (60,))
                self.valu("v_fmac_f32 v%d, s39, v60" % (src + 2 * k + half), (src + 2 * k + half,))

    def epilogue(self, scale):
        self.count, self.written = 0, {}
        for n in range(16):
            j, h = divmod(n, 2)
            if h == 0 and j:
                self.next_rows(R_AT, 4)
            t = 24 * (n & 1)
            src = self.accumulators(8 * h + j, t, scale)
            if self.C:
                self.add_c(src, R_C + 16 * j + 8 * h)
            self.store_group(src, t, R_AT + 2 * h)

    def clobbers(self):
        return ["v%d" % i for i in range(R_VP)] + ["a%d" % i for i in range(256)] + ["s%d" % i for i in range(64, 80)] + \
               ["s%d" % i for i in list(range(84, 88)) + list(range(92, 98 if self.GATHER else 96))] + (["vcc"] if self.GATHER else []) + ["m0", "scc", "memory"]


def main():
    out = sys.argv[1] if len(sys.argv) > 1 else os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_w4_loop.inc")
    with open(out, "w") as f:
        f.write("/* generated by gen_w4_loop.py -- do not edit */\n")
        for v in (Mult(False), Mult(True), Loader(False), Loader(True), Wide(False, False), Wide(False, True), Wide(True, False), Wide(True, True), Ring(False), Ring(True), Ring(False, True), Ring(True, True)):
            parts = v.generate()
            if not isinstance(v, Wide):
                parts = [(v.name + "_ASM", parts)]
            for name, lines in parts:
                f.write("#define %s \\\n" % name + " \\\n".join('\t"%s\\n\\t"' % x for x in lines) + "\n")
            f.write("#define %s_CLOBBERS %s\n" % (v.name, ", ".join('"%s"' % c for c in v.clobbers())))
        # multiplying waves: accumulator groups g[0..23] (group 6 (i / 4) + j holds row blocks 4 (i / 4) .. + 3 of column block
        # j), the lane block lb (fragment read addresses), k-tiles and flags
        ops = ['"+{a[%d:%d]}"(g[%d])' % (16 * n, 16 * n + 15, n) for n in range(16)]
        ops += ['"+{v[%d:%d]}"(g[%d])' % (16 * (n - 16), 16 * (n - 16) + 15, n) for n in range(16, 24)]
        f.write("#define W4_MULT_OUTPUTS(g) %s\n" % ", ".join(ops))
        f.write('#define W4_MULT_INPUTS(lb, nkt, flags) "{v[%d:%d]}"(lb), "{s40}"(nkt), "{s41}"(flags)\n' % (M_ARD, M_ARD + 15))
        f.write("#define W4_M_ARD 0\n#define W4_M_BRD %d\n" % (M_BRD - M_ARD))
        # loader: slot registers st[0..7] (a[0:255]) and st8 (v[0:15]), offsets of P (vp) and Q (vq, vq4), of the next tile's
        # Q (gathered; vn, vn4), LDS write address of every slot (wr[0..1], wr4), cursors sa, sb, the block sc
        ops = ['"+{a[%d:%d]}"(st[%d])' % (32 * n, 32 * n + 31, n) for n in range(8)] + ['"+{v[0:15]}"(st8)']
        f.write("#define W4_LOAD_OUTPUTS(st, st8) %s\n" % ", ".join(ops))
        f.write('#define W4_LOAD_OUTPUTS_Q(vq, vq4) "+{v[%d:%d]}"(vq), "+{v[%d:%d]}"(vq4)\n' % (L_VOFFQ, L_VOFFQ + 31, L_VOFFQ + 32, L_VOFFQ + 35))
        f.write('#define W4_LOAD_INPUTS(vp, wr, wr4, sa, sb, sc) "{v[%d:%d]}"(vp), "{v[%d:%d]}"(wr[0]), "{v[%d:%d]}"(wr[1]), "{v[%d:%d]}"(wr4), "{s[40:47]}"(sa), "{s[48:55]}"(sb), "{s[56:63]}"(sc)\n' %
                (L_VOFFP, L_VOFFP + 31, L_WR, L_WR + 31, L_WR + 32, L_WR + 63, L_WR + 64, L_WR + 67))
        f.write('#define W4_LOAD_INPUTS_NEXT(vn, vn4) "{v[%d:%d]}"(vn), "{v[%d:%d]}"(vn4)\n' % (L_VOFFQ_NEXT, L_VOFFQ_NEXT + 31, L_VOFFQ_NEXT + 32, L_VOFFQ_NEXT + 35))
        # wide symmetric kernel: the lane's load offsets vo (8 of P, 12 of Q, 12 of the next tile's Q) and its eight of D (in and out, though
        # those of P do not change: of an input the compiler kept a copy in scratch memory), the blocks of scalars sd, sa, sb, sc
        f.write('#define W4D_OUTPUTS(vo, at) "+{v[%d:%d]}"(vo), "+{v[%d:%d]}"(at)\n' % (D_VP, D_VP + 31, D_AT, D_AT + 7))
        f.write('#define W4D_INPUTS(sd, sa, sb, sc) "{s[32:39]}"(sd), "{s[40:47]}"(sa), "{s[48:55]}"(sb), "{s[56:63]}"(sc)\n')
        f.write("#define W4D_PRE %d\n" % OPTS["pre"])
        f.write("#define W4D_VP 0\n#define W4D_VQ %d\n#define W4D_VQ_NEXT %d\n" % (D_VQ - D_VP, D_VQ_NEXT - D_VP))

        # sliced kernel: the lane's load offsets vo (4 of P, 4 of Q) and its four of D and four of C, the blocks of scalars sd, sa, sb, sc
        f.write('#define W4K_OUTPUTS(vo, at) "+{v[%d:%d]}"(vo), "+{v[%d:%d]}"(at)\n' % (R_VP, R_VP + 7, R_AT, R_AT + 7))
        # gathered k-rows: the registers from R_MAP on and the two buffers over maps
        f.write('#define W4K_GATHER_OUTPUTS(vg) "+{v[%d:%d]}"(vg)\n' % (R_MAP, R_MAP + 15))
        f.write('#define W4K_GATHER_INPUTS(mc, mn) "{s[80:83]}"(mc), "{s[88:91]}"(mn)\n')
        f.write("#define W4K_SEL0 %d\n#define W4K_KB %d\n#define W4K_COL %d\n" % (R_SEL0 - R_MAP, R_KB - R_MAP, R_COL - R_MAP))
        for v in (Ring(False), Ring(True), Ring(False, True), Ring(True, True)):
            f.write("#define %s_LEAST %d\n" % (v.name, v.least))

if __name__ == "__main__":
    main()
