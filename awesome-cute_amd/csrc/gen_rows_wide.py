#!/usr/bin/env python3
"""Writes the loop of the rows kernel over 128 columns (w4a16_rows_wide.hip) as one
inline-assembly statement with fixed registers.

Why assembly: a wave keeps weights requested three chunks ahead and activations
two, next to 128 accumulators and the operands in use, in 256 registers.  The
compiler moves registers that are still being loaded from one turn of the loop to
the next, which waits for everything in flight, and puts twelve vector operations
in a row before the MFMAs that need them.  Here every wait lets exactly the later
requests stay in flight, and the operations of the unpack go behind the MFMAs of
the operand before.

A wave works by itself: no barriers.  A chunk is 64 k-values: four rows of B, 16 MB
rows of A.  Its 16 operands of 16 columns x 32 k-values are taken in the order
  j (16-column group), then (h, q) = (0,0) (1,0) (0,1) (1,1)
(h: columns 0-7 or 8-15 of the group; q: k-values 0-7 or 8-15 of a row of B), each
with MB MFMAs, one for a row block.

Register map (v = VGPR, a = AGPR, s = SGPR):
  a[4(o MB + m) : +3]  accumulator of operand o = 2j + h, row block m
  v[16r + 4i : +3]     packed weights, ring slot r (chunk % 3), row i of the chunk
  v[48 + 4r : +3]      group scales of ring slot r
  v[60 + 4x : +3]      unpacked operand ring, x = operand % 3
  v[72 + 4(2m + q):+3] activation operands of row block m
  v[104 .. 107]        words shifted by 8
  v[108 + i]           byte offset of this lane's piece of rows 8i ... 8i+7 of A
  v116 v117            per-lane byte offsets into B and into the scale rows
  v118 v119            LDS addresses of the operand reads, q = 0, 1
  v120 v121            0x64006400; -72 (fp16 x2)
  s[40:43] s[44:47] s[48:51]   buffer resources of A, B, scales
  s52 s53              first chunk of this wave, end (at least one chunk is computed)
  s54 s55              bytes per row of B; bytes per scale row
  s56                  LDS address of this wave's first slot
  s57 ...              loop state and constants
"""
import sys

RING = 3
SLOT = 8192  # a chunk's activations in LDS (a power of two)
W0, S0, OP0, A0, WT0, AL0 = 0, 48, 60, 72, 104, 108
VB, VS, VRD, VEX, VNEG72 = 116, 117, (118, 119), 120, 121
RA, RB, RS = 40, 44, 48
S_BEGIN, S_END, S_BROW, S_N2, S_LDS = 52, 53, 54, 55, 56
(S_C, S_T, S_SA, S_SB, S_SS, S_FULLA, S_FULLB, S_FULLS, S_LOMASK, S_HIMASK, S_NEG1032,
 S_SIXTEENTH) = range(57, 69)


def set_blocks(mb):
    """row blocks of 16"""
    global MB
    MB = mb


def W(r, i): return W0 + 16 * r + 4 * i
def SC(r): return S0 + 4 * r
def OP(x): return OP0 + 4 * x
def AV(m, q): return A0 + 4 * (2 * m + q)
def q4(r): return f"v[{r}:{r + 3}]"
def a4(r): return f"a[{r}:{r + 3}]"
def s4(r): return f"s[{r}:{r + 3}]"


class Emitter:
    """Collects instructions and works out the s_waitcnt immediates: loads and LDS
    reads each complete in order of issue, and a wait lets exactly those issued
    after what it waits for stay in flight."""

    def __init__(self):
        self.lines, self.vm, self.lgkm = [], [], []

    def emit(self, text):
        self.lines.append(text)

    def wait(self, vm=(), lgkm=()):
        def after(queue, tags):
            found = [len(queue) - 1 - max(i for i, t in enumerate(queue) if t == tag) for tag in tags if tag in queue]
            return min(found) if found else None
        parts = []
        n = after(self.vm, vm)
        if n is not None:
            parts.append(f"vmcnt({min(n, 63)})")
            del self.vm[:len(self.vm) - n]
        n = after(self.lgkm, lgkm)
        if n is not None:
            parts.append(f"lgkmcnt({min(n, 15)})")
            del self.lgkm[:len(self.lgkm) - n]
        if parts:
            self.emit("s_waitcnt " + " ".join(parts))


def load_rows(e, c, i):
    """rows 8i ... 8i+7 of chunk c's activations to LDS, where m0 says"""
    e.emit(f"buffer_load_dwordx4 v{AL0 + i}, {s4(RA)}, s{S_SA} offen lds")
    e.vm.append(("A", c))


def rows_scalars(e, ahead):
    """chunk `ahead` after s57: past the end, an empty buffer (zeros)"""
    e.emit(f"s_add_i32 s{S_T}, s{S_C}, {ahead}")
    e.emit(f"s_cmp_lt_i32 s{S_T}, s{S_END}")
    e.emit(f"s_cselect_b32 s{RA + 2}, s{S_FULLA}, 0")
    e.emit(f"s_lshl_b32 s{S_SA}, s{S_T}, 7")


def weight_scalars(e, ahead, group):
    e.emit(f"s_add_i32 s{S_T}, s{S_C}, {ahead}")
    e.emit(f"s_cmp_lt_i32 s{S_T}, s{S_END}")
    e.emit(f"s_cselect_b32 s{RB + 2}, s{S_FULLB}, 0")
    if group:
        e.emit(f"s_cselect_b32 s{RS + 2}, s{S_FULLS}, 0")
        e.emit(f"s_lshr_b32 s{S_SS}, s{S_T}, 1")
        e.emit(f"s_mul_i32 s{S_SS}, s{S_SS}, s{S_N2}")
    e.emit(f"s_lshl_b32 s{S_SB}, s{S_T}, 2")
    e.emit(f"s_mul_i32 s{S_SB}, s{S_SB}, s{S_BROW}")


def load_weights(e, c, i):
    r = c % RING
    e.emit(f"buffer_load_dwordx4 {q4(W(r, i))}, v{VB}, {s4(RB)}, s{S_SB} offen nt")
    e.vm.append(("W", c))
    if i < 3:
        e.emit(f"s_add_i32 s{S_SB}, s{S_SB}, s{S_BROW}")


def load_scales(e, c):
    e.emit(f"buffer_load_dwordx4 {q4(SC(c % RING))}, v{VS}, {s4(RS)}, s{S_SS} offen")
    e.vm.append(("W", c))


def read_rows(e, c, m, q):
    e.emit(f"ds_read_b128 {q4(AV(m, q))}, v{VRD[q]} offset:{2048 * m}")
    e.lgkm.append(("A", c, m, q))


def swap32(r, j):
    return [f"v_permlane32_swap_b32 v{W(r, 0) + j}, v{W(r, 2) + j}",
            f"v_permlane32_swap_b32 v{W(r, 1) + j}, v{W(r, 3) + j}"]


def swap16(r, j):
    return [f"v_permlane16_swap_b32 v{W(r, 0) + j}, v{W(r, 1) + j}",
            f"v_permlane16_swap_b32 v{W(r, 2) + j}, v{W(r, 3) + j}"]


ORDER = [(j, h, q) for j in range(4) for h, q in ((0, 0), (1, 0), (0, 1), (1, 1))]


def unpack(group, r, g):
    """operand g of the chunk in ring slot r, the four words in lockstep"""
    j, h, q = ORDER[g]
    d = OP(g_slot(g))
    out = []
    if (h, q) == (1, 0):
        out += [f"v_lshrrev_b32 v{WT0 + t}, 8, v{W(r, t) + j}" for t in range(4)]
    src = [f"v{WT0 + t}" if h else f"v{W(r, t) + j}" for t in range(4)]
    mask = S_HIMASK if q else S_LOMASK
    out += [f"v_and_or_b32 v{d + t}, {src[t]}, s{mask}, v{VEX}" for t in range(4)]
    if q == 0:
        out += [f"v_pk_add_f16 v{d + t}, v{d + t}, s{S_NEG1032} op_sel_hi:[1,0]" for t in range(4)]
    else:
        out += [f"v_pk_fma_f16 v{d + t}, v{d + t}, s{S_SIXTEENTH}, v{VNEG72} op_sel_hi:[1,0,0]" for t in range(4)]
    if group:
        sel = "op_sel:[1,0] op_sel_hi:[1,1]" if h else "op_sel_hi:[0,1]"
        out += [f"v_pk_mul_f16 v{d + t}, v{SC(r) + j}, v{d + t} {sel}" for t in range(4)]
    return out


PHASE = 0  # operands before this chunk, modulo the operand ring


def g_slot(g):
    return (PHASE + g) % 3


def chunk(e, group, u):
    """Chunk s57, ring slot u.  Behind the MFMAs of operand g, one MFMA early (an
    operand has to be complete two instructions before its first MFMA): the unpack
    of operand g + 1.  Rows of the chunk after the next follow the last read of this
    one's, weights the last word used."""
    global PHASE
    nslots = 16 * MB
    c = CHUNK
    valu = [[] for _ in range(nslots)]
    # unpack of operand g + 1 in slots MB g - 1 ... MB g + MB - 2 (operand 1's first part comes
    # with slot 0, operand 0 of the next chunk ends MB - 1 slots before this one's end)
    for g in range(16):
        if g < 15:
            ops = unpack(group, u, g + 1)
            if g + 1 == 15:
                ops = [("wait", c + 1)] + swap32((u + 1) % RING, 0) + ops
            elif ORDER[g + 1][1:] == (1, 1):
                ops = swap32(u, ORDER[g + 1][0] + 1) + ops
            elif ORDER[g + 1][1:] == (0, 0):
                ops = swap16(u, ORDER[g + 1][0]) + ops
        else:
            PHASE += 16
            ops = swap16((u + 1) % RING, 0) + unpack(group, (u + 1) % RING, 0)
            PHASE -= 16
        lo = max(0, MB * g - 1)
        hi = MB * g + MB - 1  # one past the last slot
        n = hi - lo
        for k, op in enumerate(ops):
            valu[lo + k * n // len(ops)].append(op)
    mem = [[] for _ in range(nslots)]
    for m in range(MB):
        mem[m].append(lambda m=m: read_rows(e, c, m, 1))
        # q = 0 operands are free behind group 13
        mem[14 * MB + m].append(lambda m=m: read_rows(e, c + 1, m, 0))
    # LDS addresses: the next chunk's slot before its first read
    for k in (0, 1):
        valu[14 * MB - 1].insert(0, f"v_xor_b32 v{VRD[k]}, {SLOT}, v{VRD[k]}")
    # rows of chunk c + 2, into this chunk's slot (its reads have all come back by slot 3 MB)
    first, last = 3 * MB + 1, 13 * MB
    na = 2 * MB
    for i in range(na):
        at = first + i * (last - first) // na
        if i == 0:
            mem[at - 1].append(lambda: rows_scalars(e, 2))
            mem[at - 1].append(lambda: e.emit(f"s_mov_b32 m0, s{S_LDS}"))
        mem[at].append(lambda i=i: load_rows(e, c + 2, i))
        if i < na - 1:
            mem[at].append(lambda: e.emit("s_add_u32 m0, m0, 0x400"))
    mem[last].append(lambda: e.emit(f"s_xor_b32 s{S_LDS}, s{S_LDS}, {SLOT}"))
    # weights of chunk c + 3: the last word of this one is unpacked by slot 15 MB - 2
    mem[15 * MB - 1].append(lambda: weight_scalars(e, 3, group))
    for i in range(4):
        mem[15 * MB + i * MB // 4].append(lambda i=i: load_weights(e, c + 3, i))
    if group:
        mem[16 * MB - 1].append(lambda: load_scales(e, c + 3))
    for s in range(nslots):
        g, m = divmod(s, MB)
        j, h, q = ORDER[g]
        e.wait(lgkm=[("A", c, m, q)])
        if s == 14 * MB:
            e.wait(vm=[("A", c + 1)])
        acc = 4 * ((2 * j + h) * MB + m)
        e.emit(f"v_mfma_f32_16x16x32_f16 {a4(acc)}, {q4(OP(g_slot(g)))}, {q4(AV(m, q))}, {a4(acc)}")
        ops = valu[s]
        half = (len(ops) + 1) // 2
        for k, op in enumerate(ops):
            if k == half:
                for f in mem[s]:
                    f()
            if isinstance(op, tuple):
                e.wait(vm=[("W", op[1])])
            else:
                e.emit(op)
        if len(ops) <= half:
            for f in mem[s]:
                f()
    PHASE += 16


def generate(group):
    global PHASE, CHUNK
    e = Emitter()
    PHASE = 0
    for s, w in ((S_FULLA, RA + 2), (S_FULLB, RB + 2), (S_FULLS, RS + 2), (S_C, S_BEGIN)):
        e.emit(f"s_mov_b32 s{s}, s{w}")
    # requests in the loop's order
    for c in range(3):
        weight_scalars(e, c, group)
        for i in range(4):
            load_weights(e, c, i)
        if group:
            load_scales(e, c)
        if c < 2:
            rows_scalars(e, c)
            e.emit(f"s_mov_b32 m0, s{S_LDS}")
            for i in range(2 * MB):
                e.emit("s_nop 0")
                load_rows(e, c, i)
                e.emit("s_add_u32 m0, m0, 0x400")
            e.emit(f"s_xor_b32 s{S_LDS}, s{S_LDS}, {SLOT}")
    e.emit(f"s_mov_b32 s{S_LOMASK}, 0x000f000f")
    e.emit(f"s_mov_b32 s{S_HIMASK}, 0x00f000f0")
    e.emit(f"s_mov_b32 s{S_NEG1032}, 0xe408")      # fp16 -1032
    e.emit(f"s_mov_b32 s{S_SIXTEENTH}, 0x2c00")    # fp16 1/16
    e.emit(f"v_mov_b32 v{VEX}, 0x64006400")
    e.emit(f"v_mov_b32 v{VNEG72}, 0xd480")         # fp16 -72
    for n in range(32 * MB):
        e.emit(f"v_accvgpr_write_b32 a{n}, 0")
    e.wait(vm=[("W", 0)])
    for op in swap32(0, 0) + ["s_nop 1"] + swap16(0, 0) + unpack(group, 0, 0):
        e.emit(op)
    e.wait(vm=[("A", 0)])
    for m in range(MB):
        read_rows(e, 0, m, 0)
    for u in range(RING):
        CHUNK = u
        if u == 0:
            e.emit(".Lrw_loop_%=:")
        chunk(e, group, u)
        e.emit(f"s_add_i32 s{S_C}, s{S_C}, 1")
        e.emit(f"s_cmp_lt_i32 s{S_C}, s{S_END}")
        e.emit("s_cbranch_scc0 .Lrw_done_%=" if u < RING - 1 else "s_cbranch_scc1 .Lrw_loop_%=")
    # 16 operands a chunk: the operand ring does not come round with the weights' ring of
    # three unless 48 operands are a multiple of it
    assert PHASE % 3 == 0
    e.emit(".Lrw_done_%=:")
    e.emit("s_nop 15")  # the last MFMAs' results are not readable before
    e.emit("s_nop 15")
    e.emit("s_waitcnt vmcnt(0) lgkmcnt(0)")
    return e.lines


def statement(group):
    out = ["// generated by gen_rows_wide.py -- do not edit", "asm volatile("]
    out += [f'    "{l}\\n\\t"' for l in generate(group)]
    outs = [f'"={{a[{4 * (s * MB + m)}:{4 * (s * MB + m) + 3}]}}"(acc[{s}][{m}])' for s in range(8) for m in range(MB)]
    outs += [f'"+{{s[{RA}:{RA + 3}]}}"(ra_words)', f'"+{{s[{RB}:{RB + 3}]}}"(rb_words)',
             f'"+{{s[{RS}:{RS + 3}]}}"(rs_words)', f'"+{{s{S_LDS}}}"(lds_slot)',
             f'"+{{v{VRD[0]}}}"(a_rd[0])', f'"+{{v{VRD[1]}}}"(a_rd[1])']
    out.append("    : " + ",\n      ".join(outs))
    ins = [f'"{{s{S_BEGIN}}}"(c0)', f'"{{s{S_END}}}"(c1)', f'"{{s{S_BROW}}}"(b_row)', f'"{{s{S_N2}}}"(s_row)']
    ins += [f'"{{v{AL0 + i}}}"(a_src[{i}])' for i in range(2 * MB)]
    ins += [f'"{{v{VB}}}"(b_src)', f'"{{v{VS}}}"(s_src)']
    out.append("    : " + ",\n      ".join(ins))
    clob = [f'"v{n}"' for n in list(range(0, AL0)) + [VEX, VNEG72]]
    clob += [f'"s{n}"' for n in range(S_C, S_SIXTEENTH + 1)] + ['"scc"', '"memory"']
    out.append("    : " + ", ".join(clob) + ");")
    return "\n".join(out) + "\n"


if __name__ == "__main__":
    outdir = sys.argv[1] if len(sys.argv) > 1 else "."
    for blocks in (3, 4):
        set_blocks(blocks)
        for group, name in ((True, "group"), (False, "chan")):
            with open(f"{outdir}/w4a16_rows_wide_{name}{16 * blocks}.inc", "w") as f:
                f.write(statement(group))
