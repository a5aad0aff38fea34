#!/usr/bin/env python3
"""Writes the main loops of the dense fp16 kernel (f16_streamk.hip) as inline
assembly statements with fixed registers, one per tile shape.

A workgroup has four waves, one per SIMD, each with a 128 x 128 fp32
accumulator (all 256 AGPRs): 256 x 256 tiles with a wave per quarter, and 128 x
256 tiles with two waves per 128 columns, each taking every other 32-deep k step
(128 x 128 tiles with four waves that take every fourth were 3 to 30 % slower than
eight waves of 64 x 64: two slabs of 128 k-values leave a load half a
microsecond, and two rounds through LDS add four waves' sums).  Why assembly: with
the accumulators filling their register file the compiler's allocator would
move and spill them, and the LDS reads have to be placed and waited for one by
one.

Why that shape: every operand read from LDS (one ds_read_b128) feeds eight
MFMAs, 16 reads per 64 MFMAs where eight waves of 128 x 64 take 24, and 16 instead
of 32 with 128-row tiles (64 x 64 each).  Fewer reads leave the matrix pipe more of
the power that bounds the loop: 4096^3 101 -> 96 us, the pipe busy 76 % of the
cycles, LDS reads 21 %.

A step is 64 MFMAs: row blocks i = 0 ... 7 of 16 rows, operands o = 0 ... 7 of
16 columns.  Its A operands are read three row blocks ahead into a ring of four,
the eight B operands of the next step into the other of two buffers.  A slab is
what the workgroup stages in LDS at once, in a ring of two or three; the request
for the slab after the ring's last goes into the slab just finished:

  inner step (256 x 256 only: the next step is in the same slab)
     A and B reads dealt out evenly
  outer step (the next step is in the next slab)
     row blocks 0-4   the last A operands of this slab
     then             my loads of the next slab have landed, my reads of this
                      one too; barrier: so have everybody's
     row blocks 5-7   B and A operands of the next step, alternating with the
                      request for the slab that goes where this one was; what
                      does not fit follows in the next step

Every memory operation gets an MFMA to itself: two behind one MFMA cost more
than its time.  All s_waitcnt are computed from the order of issue.

Registers (v = VGPR, a = AGPR, s = SGPR):
  a[32i+4o : +3]     accumulator of row block i, operand o
  v[32b+4o : +3]     B operands, buffer b (step parity)
  v[64+4x : +3]      A operand ring, x = row block % 4
  v[80+j] v[88+j]    LDS addresses of the A and B reads, j = slot (x 2 + step of the slab)
  v[96+t]            byte offsets of this lane's loads, A then B
  s[40:43] s[44:47]  buffer resources of A and B (their sizes become 0 past the last slab)
  s48 s49 s50 s51    byte offset of the next request; slabs; requested; left
  s52 s53            sizes of A and B
  s[54:56] s[57:59]  LDS addresses of this wave's part of the slots, A and B
"""
import sys

AHEAD = 3
RA, RB = 40, 44
S_AT, S_N, S_REQ, S_LEFT, S_FULLA, S_FULLB, S_MA, S_MB = 48, 49, 50, 51, 52, 53, 54, 57
V_A, V_B, V_OFF = 80, 88, 96


class Shape:
    def __init__(self, tm, tn, wk, ring):
        self.name, self.wk, self.ring = f"{tm}x{tn}", wk, ring
        self.slab = (tm + tn) * ROW
        self.steps = 2 // wk                       # steps of a wave per slab
        self.ta = tm * ROW // 4096                 # load instructions per wave: 1 KiB each
        self.loads = self.ta + tn * ROW // 4096


ROW = 128          # bytes of a row in a slab: 64 k-values
BLOCK = 16 * ROW
SHAPES = [Shape(256, 256, 1, 2), Shape(128, 256, 2, 3)]
TAIL = 12  # loads requested right behind the barrier


def q(base): return f"v[{base}:{base + 3}]"
def aq(base): return f"a[{base}:{base + 3}]"
def sq(base): return f"s[{base}:{base + 3}]"
def BOP(b, o): return 32 * b + 4 * o
def AOP(i): return 64 + 4 * (i & 3)


class Emitter:
    def __init__(self):
        self.lines = []
        self.lds = []  # destinations of LDS reads in flight, oldest first

    def emit(self, text):
        self.lines.append(text)

    def read(self, dst, addr, off):
        assert 0 <= off < 65536
        self.emit(f"ds_read_b128 {q(dst)}, v{addr} offset:{off}")
        self.lds.append(dst)

    def need(self, *regs):
        """wait until the reads into `regs` have landed (LDS reads land in order)"""
        last = max([i for i, r in enumerate(self.lds) if r in regs], default=-1)
        if last >= 0:
            self.lds = self.lds[last + 1:]
            assert len(self.lds) <= 15
            self.emit(f"s_waitcnt lgkmcnt({len(self.lds)})")


def request_head(e, sh, slot):
    """what the loads of the next slab need: sizes (zero past the end), m0"""
    e.emit(f"s_cmp_lt_u32 s{S_REQ}, s{S_N}")
    e.emit(f"s_cselect_b32 s{RA + 2}, s{S_FULLA}, 0")
    e.emit(f"s_cselect_b32 s{RB + 2}, s{S_FULLB}, 0")
    e.emit(f"s_add_u32 s{S_REQ}, s{S_REQ}, 1")
    e.emit(f"s_mov_b32 m0, s{S_MA + slot}")


def request(e, sh, slot, t):
    """load t of a slab; m0 is left ready for load t + 1 (an MFMA or a nop lies between)"""
    e.emit(f"buffer_load_dwordx4 v{V_OFF + t}, {sq(RA if t < sh.ta else RB)}, s{S_AT} offen lds")
    if t == sh.ta - 1:
        e.emit(f"s_mov_b32 m0, s{S_MB + slot}")
    elif t < sh.loads - 1:
        e.emit("s_add_u32 m0, m0, 0x400")
    else:
        e.emit(f"s_add_u32 s{S_AT}, s{S_AT}, {ROW}")


def assign(ops, n):
    """(preferred MFMA, operation) -> {MFMA: operation}, distinct, in the order of preference"""
    at, last = {}, -1
    for pref, fn in sorted(ops, key=lambda x: x[0]):
        last = max(last + 1, int(pref))
        at[last] = fn
    assert last < n, last
    return at


def read_a(e, sh, j, i):
    e.read(AOP(i), V_A + j, (i & 7) * BLOCK)


def read_b(e, sh, j, b, o):
    e.read(BOP(b, o), V_B + j, o * BLOCK)


def next_operands(sh, j, b):
    """the reads of the next step that an outer step issues, in order"""
    ops = [lambda e, o=o: read_b(e, sh, j, b, o) for o in range(8)]
    ops.insert(1, lambda e: read_a(e, sh, j, 0))
    ops += [lambda e, i=i: read_a(e, sh, j, i) for i in range(1, AHEAD)]
    return ops


def step(e, sh, slot, h, b, carry):
    """one step; carry: (slot, first load) of a request that the step before left unfinished"""
    steps = sh.steps
    outer = h == steps - 1
    j = slot * steps + h
    nslot = (slot + 1) % sh.ring if outer else slot
    jn = nslot * steps + (0 if outer else h + 1)
    ops = [(8 * i, lambda e, i=i: read_a(e, sh, j, i + AHEAD)) for i in range(8 - AHEAD)]
    for x, t in enumerate(range(carry[1], sh.loads) if carry else ()):
        ops.append((2 + 4 * x, lambda e, t=t: request(e, sh, carry[0], t)))
    left = None
    if outer:
        bar = 8 * (8 - AHEAD)

        def barrier(e):
            e.emit(f"s_waitcnt vmcnt({(sh.ring - 2) * sh.loads}) lgkmcnt(0)")
            e.lds = []
            e.emit("s_barrier")
            request_head(e, sh, slot)

        ops.append((bar - 1, barrier))
        ops += [(bar + 2 * x, fn) for x, fn in enumerate(next_operands(sh, jn, b ^ 1))]
        tail = min(TAIL, sh.loads)
        ops += [(bar + 1 + 2 * t, lambda e, t=t: request(e, sh, slot, t)) for t in range(tail)]
        left = (slot, tail) if tail < sh.loads else None
    else:
        ops += [(8 * (8 - AHEAD + i), lambda e, i=i: read_a(e, sh, jn, i)) for i in range(AHEAD)]
        ops += [(8 * o + 4, lambda e, o=o: read_b(e, sh, jn, b ^ 1, o)) for o in range(8)]
    at = assign(ops, 64)
    for i in range(8):
        for o in range(8):
            e.need(AOP(i), *([BOP(b, o)] if i == 0 else []))
            acc = 32 * i + 4 * o
            e.emit(f"v_mfma_f32_16x16x32_f16 {aq(acc)}, {q(BOP(b, o))}, {q(AOP(i))}, {aq(acc)}")
            if 8 * i + o in at:
                at[8 * i + o](e)
    return left


def generate(sh):
    e = Emitter()
    # prologue: every slot requested (the last one as far as an outer step would
    # have), the accumulators zeroed, the first step's operands read
    e.emit(f"s_mov_b32 s{S_FULLA}, s{RA + 2}")
    e.emit(f"s_mov_b32 s{S_FULLB}, s{RB + 2}")
    e.emit(f"s_mov_b32 s{S_REQ}, 0")
    e.emit(f"s_mov_b32 s{S_LEFT}, s{S_N}")
    for s in range(1, sh.ring):
        e.emit(f"s_add_u32 s{S_MA + s}, s{S_MA}, {s * sh.slab}")
        e.emit(f"s_add_u32 s{S_MB + s}, s{S_MB}, {s * sh.slab}")
    last = min(TAIL, sh.loads)
    for s in range(sh.ring):
        request_head(e, sh, s)
        for t in range(sh.loads if s < sh.ring - 1 else last):
            e.emit("s_nop 0")
            request(e, sh, s, t)
    for n in range(256):
        e.emit(f"v_accvgpr_write_b32 a{n}, 0")
    e.emit(f"s_waitcnt vmcnt({(sh.ring - 2) * sh.loads + last})")
    e.emit("s_barrier")
    for fn in next_operands(sh, 0, 0):
        fn(e)
    start = list(e.lds)
    carry = (sh.ring - 1, last) if last < sh.loads else None
    first_carry = carry
    e.emit(".Ldn_loop_%=:")
    b = 0
    turns = 2 if sh.ring * sh.steps % 2 else 1  # slots and operand buffers come round together
    for turn in range(turns):
        for slot in range(sh.ring):
            for h in range(sh.steps):
                carry = step(e, sh, slot, h, b, carry)
                b ^= 1
            e.emit(f"s_sub_u32 s{S_LEFT}, s{S_LEFT}, 1")
            e.emit(f"s_cmp_eq_u32 s{S_LEFT}, 0")
            if turn == turns - 1 and slot == sh.ring - 1:
                e.emit("s_cbranch_scc0 .Ldn_loop_%=")
            else:
                e.emit("s_cbranch_scc1 .Ldn_done_%=")
    assert b == 0 and e.lds == start and carry == first_carry
    e.emit(".Ldn_done_%=:")
    # the last MFMAs' results are not readable for 18 cycles, and the hardware
    # does not interlock that for what follows; nothing may be on its way into
    # LDS or registers either
    e.emit("s_nop 15")
    e.emit("s_nop 15")
    e.emit("s_waitcnt vmcnt(0) lgkmcnt(0)")
    return e.lines


def statement(sh):
    out = ["// generated by gen_dense.py -- do not edit", "asm volatile("]
    out += [f'    "{l}\\n\\t"' for l in generate(sh)]
    outs = [f'"={{{aq(32 * i + 4 * o)}}}"(acc[{i}][{o}])' for i in range(8) for o in range(8)]
    outs += [f'"+{{{sq(RA)}}}"(ra_words)', f'"+{{{sq(RB)}}}"(rb_words)', f'"+{{s{S_AT}}}"(s_at)']
    out.append("    : " + ",\n      ".join(outs))
    reads = sh.ring * sh.steps
    ins = [f'"{{s{S_N}}}"(slabs)', f'"{{s{S_MA}}}"(lds_a)', f'"{{s{S_MB}}}"(lds_b)']
    ins += [f'"{{v{V_A + j}}}"(a_rd[{j}])' for j in range(reads)]
    ins += [f'"{{v{V_B + j}}}"(b_rd[{j}])' for j in range(reads)]
    ins += [f'"{{v{V_OFF + t}}}"(src[{t}])' for t in range(sh.loads)]
    clob = [f"v{n}" for n in range(80)]
    out.append("    : " + ",\n      ".join(ins))
    clob += [f"s{n}" for n in range(S_REQ, S_FULLB + 1)]
    clob += [f"s{S_MA + s}" for s in range(1, sh.ring)] + [f"s{S_MB + s}" for s in range(1, sh.ring)]
    clob += ["scc", "memory"]  # (m0 is the compiler's to reserve; it keeps nothing there)
    out.append("    : " + ", ".join(f'"{c}"' for c in clob) + ");")
    return "\n".join(out) + "\n"


if __name__ == "__main__":
    outdir = sys.argv[1] if len(sys.argv) > 1 else "."
    for sh in SHAPES:
        with open(f"{outdir}/f16_dense_{sh.name}.inc", "w") as f:
            f.write(statement(sh))
