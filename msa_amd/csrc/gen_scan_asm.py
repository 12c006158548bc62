#!/usr/bin/env python3
"""Writes ``scan_asm.inc``: the instruction-level K step of the large-tile routing scan (``score_scan4_kernel``), and
``gemm_asm.inc``: the same step for the tiled products (``tile_gemm_kernel``).

The scan's 256 x 256 tile is computed by four wavefronts, one per SIMD, 128 x 128 each: 8 x 8 blocks of 16 x 16 in the 256
accumulation registers a0-a255, eight fragments of each operand in v128-v191.  One K step (64 elements of K) is one asm statement
whose issue order is fixed here: two sub-steps of 64 ``v_mfma_f32_16x16x32_bf16`` (the 32 x 32 x 16 form costs more power a FLOP: it
passes an accumulator twice as often for the same products, and these loops run at the clock the power allows).

* A sub-step walks over the four quadrants (half of the A fragments x half of the B fragments, sixteen MFMAs each) so that
  neighbouring quadrants share a half and every half's last use comes a quadrant or two before its successor's first: the
  fragments are single-buffered.  Each quadrant requests the four that the next but none needs (one read behind each of its MFMAs
  1 - 4) and begins with the four that arrived last changing slowest, so that each wait covers one read and has had at least
  sixteen MFMAs' time; the other operand goes to and fro, so that neighbouring MFMAs share an operand.
* The eight 1 KB blocks of the K_r tile two steps ahead are requested during the first two quadrants and those of the query tile two
  steps ahead during the last two, one ``buffer_load_dwordx4 ... lds`` behind every fourth MFMA (the compute unit's address unit
  takes about that long per load of four wavefronts), M0 set one instruction earlier.
* The step's only wait for memory (everything but the eight newest loads) and the workgroup barrier sit at the start of the last but
  one quadrant, the barrier behind its first MFMA so that the matrix pipe runs while the wavefronts meet; behind the barrier the
  stages this step has finished with are refilled and the first fragments of the next step are read.

LDS: two stages of the query tile at 0 / 0x8000, three of the K_r tile at 0x10000 / 0x18000 / 0x20000, rows of 128
bytes whose 16-byte units are XOR-swizzled by (row >> 1) & 7.

Registers the statements own (the kernel's compiler-allocated code stays below v128, below v96 where queries lie in units, and uses
no accumulation registers): v128-v159 fragments A0-A7, v160-v191 B0-B7, v192-v197 LDS addresses of the step, v198-v201 per-lane LDS offsets of the
two sub-steps (A, then B), v208-v215 global offsets of the wavefront's eight 1 KB blocks, v216-v223 tile pool and prefetch values
(see the kernel), v224-v231 the maxima of the tile just finished (row block of 32 rows i and column group of 64 columns p in
v224 + 2 i + p, lane l column 64 p + l; in the folding form the maxima over all rows, column group p in v224 + p), v232-v239 their
parts before the lanes are joined, v96-v127 those of units of eight rows (unit u of row block i in v96 + 8 i + 4 p + u, lane l column
64 p + l), v240-v247 scratch of the reduction and the fold, v248-v252 per-lane constants of the fold,
s76-s95 scratch.

The reduction of a finished tile (per lane the maximum of each block's four values, then of the blocks below it, then over the four
lanes that hold a column: two half-wave swaps and a swap of rows of sixteen for four column blocks) rides in the first sub-step of
the next tile's first K step, a block in front of the MFMA that overwrites it: with one wavefront per SIMD the matrix pipe runs
under it.  When the wavefront's rows belong to one query and all count and the tile lies inside the bank, the fold of the
column maxima over the chunks of a document (order-preserving key, segmented max-scan over the 64
lanes by row moves, one atomic per document run) follows in the same statement, dealt out behind the MFMAs of
the second sub-step; its atomics are issued behind the step's wait so that the wait does not count them.  Short queries lie in units
of eight rows, four units a row block, unit u in rows 4 u .. 4 u + 3 of either sixteen: a lane has a unit's maximum of its column
without an exchange, and the joining becomes a transposition of (column block, unit), the same swaps without the maxima.

In the products the A operand is the weights and the B operand the tokens; each has row offsets of its own (v208-v215 the eight blocks
of the A tile, v216-v223 those of the B tile), neither is read non-temporal, and a finished tile's accumulators are read behind its
last step.

Run ``python gen_scan_asm.py`` after changing the schedule; ``scan_asm.inc`` is committed, ``gemm_asm.inc`` (a copy of the step for every
column of every end) is written by every build.
"""
import os
import sys

FA, FB = 128, 160
VT_A0, VT_B0, VT_A1, VT_B1, VT_AN, VT_BN = range(192, 198)
VADDR = 198          # A of sub-steps 0 and 1, B of sub-steps 0 and 1
VOFF = 208
VOFF_B = 216         # of the products' B operand
VMAX = 224
VPART = 232
VUNIT = 96
VRED = 240           # 8 scratch registers; the fold's temporaries: pair p in v(240 + 4 p) .. v(243 + 4 p)
V_LOWMASK, V_DISTBASE, V_L32P1, V_IS31, V_L15 = 248, 249, 250, 251, 252
VDOC = 220           # documents of the wavefront's columns: group p in v(220 + p)
S_HALF = "s[86:87]"  # lanes 32 - 63
S_M0, S_AN, S_BN, S_BLD = "s92", "s93", "s94", "s95"
B0, BEND = 0x10000, 0x28000

QUADS = [[(0, 0), (0, 1), (1, 1), (1, 0)], [(0, 1), (0, 0), (1, 0), (1, 1)]]      # (A half, B half) in the order of a sub-step
# the fragments requested during a quadrant (operand, half, address register)
READS = [[("b", 1, VT_B0), ("a", 1, VT_A0), ("a", 0, VT_A1), ("b", 1, VT_B1)],
         [("b", 0, VT_B1), ("a", 1, VT_A1), ("a", 0, VT_AN), ("b", 0, VT_BN)]]
BARRIER = (1, 2)


class Tile:
    """A wavefront's blocks (rows of A x rows of B, in sixteens) and what follows from them: LDS stages, loads of a wavefront."""

    def __init__(self, a_blocks=8, b_blocks=8):
        self.a, self.b = a_blocks, b_blocks
        self.stage_a, self.stage_b = a_blocks * 4096, b_blocks * 4096
        self.b0 = 2 * self.stage_a
        self.b_end = self.b0 + 3 * self.stage_b

    def acc(self, i, j):
        b = (i * self.b + j) * 4
        return f"a[{b}:{b + 3}]"


SCAN = Tile()


def frag(kind, n):
    b = (FA if kind == "a" else FB) + 4 * n
    return f"v[{b}:{b + 3}]"


def order(sub, q, tile=SCAN):
    """The quadrant's blocks: the fragments that arrived last change slowest, the others go to and fro."""
    ha, hb = QUADS[sub][q]
    na, nb = tile.a // 2, tile.b // 2
    slow, fast = (na, nb) if q >= 2 else (nb, na)
    out = []
    for n in range(slow):
        for m in range(fast):
            x = m if n % 2 == 0 else fast - 1 - m
            out.append((na * ha + n, nb * hb + x) if q >= 2 else (na * ha + x, nb * hb + n))
    return out


class Reduction:
    """The maxima of a finished tile, a block at a time in the order of the first sub-step's quadrants."""

    def __init__(self, joined, units=False):
        self.joined, self.units, self.seen, self.flip = joined, units, set(), 0

    def part(self, i, j):
        if self.units:
            return VUNIT + 4 * ((i >> 1) * 2 + (j >> 2)) + (j & 3)
        # joined: one row of parts per column group, over all rows; otherwise one per row block of 32 inside the quadrant
        return VPART + (4 * (j >> 2) if self.joined else 4 * ((i >> 1) & 1)) + (j & 3)

    def block(self, i, j):
        b = (i * 8 + j) * 4
        r = [f"v{VRED + self.flip + x}" for x in range(4)]
        self.flip ^= 4
        m = f"v{self.part(i, j)}"
        key = (j,) if self.joined else (i >> 1, j)
        out = [f"v_accvgpr_read_b32 {r[x]}, a{b + x}" for x in range(4)]
        out.append(f"v_max3_f32 {r[0]}, {r[0]}, {r[1]}, {r[2]}")
        out.append(f"v_max3_f32 {m}, {m}, {r[0]}, {r[3]}" if key in self.seen else f"v_max_f32 {m}, {r[0]}, {r[3]}")
        self.seen.add(key)
        return out

    def after(self, q):
        """What a quadrant's parts allow: the lanes of a column group joined, lane l column l of the group."""
        ha, hb = QUADS[0][q]
        if self.units:
            firsts = [VUNIT + 4 * ((2 * ha + r) * 2 + hb) for r in range(2)]
            return [f"{op} v{first + x}, v{first + y}" for op, x, y in (("v_permlane32_swap_b32", 0, 2), ("v_permlane32_swap_b32", 1, 3),
                                                                        ("v_permlane16_swap_b32", 0, 1), ("v_permlane16_swap_b32", 2, 3))
                    for first in firsts]
        if self.joined:
            groups = [(VPART + 4 * hb, VMAX + hb)] if q >= 2 else []
        else:
            groups = [(VPART, VMAX + 2 * (2 * ha) + hb), (VPART + 4, VMAX + 2 * (2 * ha + 1) + hb)]
        out = []
        for step in ("v_permlane32_swap_b32 {0}, {2}", "v_permlane32_swap_b32 {1}, {3}", "v_max_f32 {0}, {0}, {2}", "v_max_f32 {1}, {1}, {3}",
                     "v_permlane16_swap_b32 {0}, {1}", "v_max_f32 {r}, {0}, {1}"):
            for first, result in groups:
                out.append(step.format(*(f"v{first + x}" for x in range(4)), r=f"v{result}"))
        return out


def fold_pair(p):
    """Document fold of column group p (maxima over the rows in v(VMAX + p), documents of
    the 64 columns in v(VDOC + p)): returns (instructions, the masked atomic).  [okey]: the query's row of keys."""
    R, doc = f"v{VMAX + p}", f"v{VDOC + p}"
    t0, t1, t2, t3 = (f"v{VRED + 4 * p + x}" for x in range(4))
    sc = f"s[{80 + 2 * p}:{81 + 2 * p}]"        # a condition
    shl, shh = f"s{76 + 2 * p}", f"s{77 + 2 * p}"   # run heads, one bit per lane
    sx = "s[88:89]"                             # exec saved around the atomic
    o = []
    o.append(f"v_ashrrev_i32 {t0}, 31, {R}")               # order-preserving key of the float
    o.append(f"v_or_b32 {t0}, 0x80000000, {t0}")
    o.append(f"v_xor_b32 {R}, {R}, {t0}")
    o.append(f"v_mov_b32 {t1}, {doc}")                     # the document of the lane below (lane 0: its own)
    o.append(f"v_mov_b32_dpp {t1}, {doc} wave_shr:1 row_mask:0xf bank_mask:0xf")
    o.append(f"v_cmp_ne_u32_e64 s[{shl[1:]}:{shh[1:]}], {t1}, {doc}")
    o.append(f"s_or_b32 {shl}, {shl}, 1")                  # lanes 0 and 32 open a run
    o.append(f"s_or_b32 {shh}, {shh}, 1")
    o.append(f"v_mov_b32 {t1}, {shl}")
    o.append(f"v_mov_b32 {t2}, {shh}")
    o.append(f"v_cndmask_b32_e64 {t1}, {t1}, {t2}, {S_HALF}")      # the heads of the lane's half
    o.append(f"v_and_b32 {t2}, v{V_LOWMASK}, {t1}")        # heads at or below the lane (never empty)
    o.append(f"v_ffbh_u32 {t2}, {t2}")
    o.append(f"v_add_u32 {t2}, {t2}, v{V_DISTBASE}")       # distance from the run's first lane: l32 - 31 + leading zeros
    o.append(f"v_lshrrev_b32 {t3}, v{V_L32P1}, {t1}")
    o.append(f"v_and_b32 {t3}, 1, {t3}")
    o.append(f"v_or_b32 {t3}, {t3}, v{V_IS31}")            # non-zero: last lane of its run
    for k in (1, 2, 4, 8):                                 # segmented max-scan inside the rows of 16 lanes
        o.append(f"v_max_u32_dpp {t0}, {R}, {R} row_shr:{k} row_mask:0xf bank_mask:0xf bound_ctrl:0")
        o.append(f"v_cmp_le_u32_e64 {sc}, {k}, {t2}")
        o.append(f"v_cndmask_b32_e64 {R}, {R}, {t0}, {sc}")
    o.append(f"v_mov_b32 {t0}, 0")                         # lane 15 of the lower row joins the runs that cross into the upper
    o.append(f"v_mov_b32_dpp {t0}, {R} row_bcast:15 row_mask:0xa bank_mask:0xf")
    o.append(f"v_max_u32 {t0}, {t0}, {R}")
    o.append(f"v_cmp_gt_u32_e64 {sc}, {t2}, v{V_L15}")
    o.append(f"v_cndmask_b32_e64 {R}, {R}, {t0}, {sc}")
    o.append(f"v_lshlrev_b32 {t0}, 2, {doc}")
    o.append(f"v_cmp_ne_u32_e64 {sc}, 0, {t3}")
    atomic = [f"s_and_saveexec_b64 {sx}, {sc}", f"global_atomic_umax {t0}, {R}, %[okey]", f"s_mov_b64 exec, {sx}"]
    return o, atomic


def interleave(a, b):
    out = []
    for x, y in zip(a, b):
        out += [x, y]
    return out + a[len(b):] + b[len(a):]


def written_vgprs(line):
    """Vector registers an instruction writes (first operand of v_* / ds_read*; v_permlane32_swap writes both)."""
    import re
    op, _, rest = line.partition(" ")
    if not (op.startswith("v_") or op.startswith("ds_read")) or op.startswith("v_mfma") or op.startswith("v_cmp"):
        return set()
    ops = [x.strip() for x in rest.split(",")]
    targets = ops[:2] if op.startswith("v_permlane") else ops[:1]
    regs = set()
    for t in targets:
        m = re.match(r"v\[(\d+):(\d+)\]", t)
        if m:
            regs |= set(range(int(m.group(1)), int(m.group(2)) + 1))
        else:
            m = re.match(r"v(\d+)$", t)
            if m:
                regs.add(int(m.group(1)))
    return regs


def fix_lane_move_hazards(lines):
    """A DPP operand or a half-wave swap reads its registers two wait states after a VALU write at the earliest."""
    import re
    out = []
    for line in lines:
        op = line.split(" ")[0]
        if op.endswith("_dpp") or op.startswith("v_permlane"):
            reads = {int(x) for x in re.findall(r"\bv(\d+)\b", line)}
            dist = 0
            need = 0
            for prev in reversed(out):
                if dist >= 2:
                    break
                if written_vgprs(prev) & reads:
                    need = 2 - dist
                    break
                dist += int(prev.split(" ")[1]) + 1 if prev.startswith("s_nop") else 1
            if need:
                out.append(f"s_nop {need - 1}")
        out.append(line)
    return out


def kstep(fresh, reduce=None, tile=SCAN, voff_b=VOFF, nt=" nt", woff=("woff", "woff"), fillers=(), stores=(), early_fillers=()):
    """One K step.  Operands: [sa] / [sb] LDS stage of the step's A / B tile (advanced to the next step's),
    [ra] / [rb] resources the loads of this step read, [k] their byte offset inside a row, [woff] the wavefront's part of a stage.
    fresh: a tile's first step (the first sub-step multiplies into zero); reduce: it also reduces the accumulators the
    previous tile left, "blocks" to one maximum per row block, "units" per eight rows, "fold" on to the key plane ([okey]: the query's keys).
    fillers go behind the MFMAs, stores (of the tile before) behind the step's wait so that it does not count them;
    early_fillers: a list per block in front of the MFMA that overwrites it."""
    out = []
    e = out.append
    fillers, atomics, stores = list(fillers), [], list(stores)
    red = Reduction(reduce == "fold", reduce == "units") if reduce else None
    if reduce == "fold":
        (a0, at0), (a1, at1) = fold_pair(0), fold_pair(1)
        fillers = interleave(a0, a1)
        atomics = at0 + at1
    blocks = tile.a * tile.b
    per_slot = -(-len(fillers) // 44) if reduce else -(-len(fillers) // (blocks + blocks // 2 - 12)) if fillers else 0
    # The step's scalar and address arithmetic stands behind its first MFMAs, not in front of them (a wavefront that
    # is alone on its SIMD pays for every instruction the matrix pipe does not run under): `early` is what the first
    # LDS read and the first tile load need, `later` the rest, two instructions per MFMA.
    early = [f"s_mov_b32 {S_M0}, m0",
             f"v_add_u32 v{VT_B0}, %[sb], v{VADDR + 2}", f"v_add_u32 v{VT_A0}, %[sa], v{VADDR}",
             f"s_sub_u32 {S_BLD}, %[sb], {tile.stage_b:#x}", f"s_cmp_lt_u32 {S_BLD}, {tile.b0:#x}",
             f"s_cselect_b32 {S_BLD}, {tile.b_end - tile.stage_b:#x}, {S_BLD}", f"s_add_u32 {S_BLD}, {S_BLD}, %[{woff[1]}]"]
    later = [f"v_add_u32 v{VT_A1}, %[sa], v{VADDR + 1}", f"v_add_u32 v{VT_B1}, %[sb], v{VADDR + 3}",
             f"s_add_u32 {S_BN}, %[sb], {tile.stage_b:#x}", f"s_cmp_eq_u32 {S_BN}, {tile.b_end:#x}", f"s_cselect_b32 {S_BN}, {tile.b0:#x}, {S_BN}",
             f"s_xor_b32 {S_AN}, %[sa], {tile.stage_a:#x}", f"v_add_u32 v{VT_AN}, {S_AN}, v{VADDR}", f"v_add_u32 v{VT_BN}, {S_BN}, v{VADDR + 2}"]
    if reduce == "fold":
        later += ["s_mov_b32 s86, 0", "s_mov_b32 s87, -1"]
    half = {"a": tile.a // 2, "b": tile.b // 2}
    pending = [("a", n) for n in range(half["a"])] + [("b", n) for n in range(half["b"])]      # reads in flight, oldest first: the step before left these
    quad = blocks // 4                                     # MFMAs of a quadrant
    every = {0: 2 * quad // tile.b, 1: 2 * quad // tile.a}  # MFMAs between two tile loads of a sub-step's
    nload = {0: 0, 1: 0}
    read_from = 1 if quad > half["a"] else 0
    for sub in range(2):
        for q in range(4):
            kind, which, addr = READS[sub][q]
            for n, (i, j) in enumerate(order(sub, q, tile)):
                if (sub, q) == BARRIER and n == 0:
                    e(f"s_waitcnt vmcnt({tile.b}) lgkmcnt(0)")
                    pending = []
                need = max([pending.index(x) for x in (("a", i), ("b", j)) if x in pending], default=-1)
                if need >= 0:
                    pending = pending[need + 1:]
                    e(f"s_waitcnt lgkmcnt({len(pending)})")
                do_load = n % every[sub] == every[sub] - 1 and q // 2 == sub
                if do_load:
                    if nload[sub]:
                        e("s_add_u32 m0, m0, 0x400")
                    elif sub == 0:
                        e(f"s_mov_b32 m0, {S_BLD}")
                    else:
                        e(f"s_add_u32 m0, %[sa], %[{woff[0]}]")
                if red and sub == 0:
                    out.extend(red.block(i, j))
                if early_fillers and sub == 0:
                    out.extend(early_fillers[i][j])
                c = "0" if (fresh and sub == 0) else tile.acc(i, j)
                e(f"v_mfma_f32_16x16x32_bf16 {tile.acc(i, j)}, {frag('a', i)}, {frag('b', j)}, {c}")
                if (sub, q) == BARRIER and n == 0:
                    e("s_barrier")
                if (sub, q, n) == (0, 0, 0):
                    out.extend(early)
                if (sub, q) == (0, 0) and n >= min(4, quad // 2):
                    for _ in range(max(2, -(-len(later) // (quad - n)))):
                        if later:
                            e(later.pop(0))
                if (sub == 1 and n > (4 if q == 2 else 0)) if reduce else ((sub, q) not in ((0, 0), (1, 3)) and not ((sub, q) == BARRIER and n < 2)):
                    for _ in range(per_slot):
                        if fillers:
                            e(fillers.pop(0))
                if (sub, q) == (1, 3) and n in (10, 12) and atomics:
                    assert not fillers
                    for _ in range(3):
                        e(atomics.pop(0))
                if (sub, q) == (1, 3) and stores:
                    assert not fillers
                    if n % max(1, quad // len_stores) == 0:
                        e(stores.pop(0))
                elif (sub, q) == (1, 2):
                    len_stores = max(1, len(stores))
                if read_from <= n < read_from + half[kind]:
                    idx = which * half[kind] + n - read_from
                    e(f"ds_read_b128 {frag(kind, idx)}, v{addr} offset:{idx * 2048}")
                    pending.append((kind, idx))
                if do_load:
                    if sub == 0:
                        e(f"buffer_load_dwordx4 v{voff_b + nload[0]}, %[rb], %[k] offen{nt} lds")
                    else:
                        e(f"buffer_load_dwordx4 v{VOFF + nload[1]}, %[ra], %[k] offen lds")
                    nload[sub] += 1
            if red and sub == 0:
                out.extend(red.after(q))
    e(f"s_mov_b32 %[sa], {S_AN}")
    e(f"s_mov_b32 %[sb], {S_BN}")
    e(f"s_mov_b32 m0, {S_M0}")
    assert not fillers and not atomics and not later and not stores and nload == {0: tile.b, 1: tile.a}
    scc = [l.split()[0] for l in out if l.startswith(("s_cmp", "s_cselect", "s_add_u32", "s_sub_u32", "s_xor", "s_or_b32", "s_and_save"))]
    assert all(scc[n - 1].startswith("s_cmp") for n, l in enumerate(scc) if l == "s_cselect_b32")
    assert pending[-half["b"]:] == [("b", n) for n in range(half["b"])]
    return fix_lane_move_hazards(out)


def reduction(units=False):
    """The reduction by itself, behind a workgroup's last tile (an MFMA's result may be read 18 wait states after its
    issue at the earliest)."""
    red, out = Reduction(False, units), ["s_nop 15", "s_nop 7"]
    for q in range(4):
        for i, j in order(0, q):
            out += red.block(i, j)
        out += red.after(q)
    return fix_lane_move_hazards(out)


def define(name, lines):
    """(@NT in a line stands for the macro's parameter)"""
    body = " \\\n".join(f'  "{l}\\n\\t"' for l in lines).replace("@NT", '" NT "')
    return f"#define {name} \\\n{body}\n"


def frags0():
    """Fragments of the first quadrant out of the stages [sa] / [sb] (in front of the first step)."""
    lines = [f"v_add_u32 v{VT_AN}, %[sa], v{VADDR}", f"v_add_u32 v{VT_BN}, %[sb], v{VADDR + 2}"]
    for kind, addr in (("a", VT_AN), ("b", VT_BN)):
        lines += [f"ds_read_b128 {frag(kind, n)}, v{addr} offset:{n * 2048}" for n in range(4)]
    return lines


def load8(voff, nt=""):
    """The wavefront's eight blocks of one operand tile into the LDS stage at [dst] (+ wave * 8 KB already added)."""
    lines = [f"s_mov_b32 {S_M0}, m0", "s_mov_b32 m0, %[dst]", "s_nop 4"]
    for i in range(8):
        lines.append(f"buffer_load_dwordx4 v{voff + i}, %[r], %[k] offen{nt} lds")
        if i < 7:
            lines += ["s_add_u32 m0, m0, 0x400", "s_nop 0"]
    return lines + [f"s_mov_b32 m0, {S_M0}"]


def set_registers(first, count):
    return [f"v_mov_b32 v{first + s}, %{s}" for s in range(count)]


def clobbers(name, first=128):
    regs = [f"v{r}" for r in range(first, 256)] + [f"a{r}" for r in range(256)] + [f"s{r}" for r in range(76, 96)] + ["vcc", "scc", "memory"]
    return f"#define {name} " + ", ".join(f'"{x}"' for x in regs) + "\n"


HEADER = "// Generated by gen_scan_asm.py (the schedule and the register map are described there).  Do not edit.\n"


def scan_text():
    return "\n".join([
        HEADER,
        define("MSA_SCAN4_KSTEP", kstep(False)),
        define("MSA_SCAN4_KSTEP_FRESH", kstep(True)),
        define("MSA_SCAN4_KSTEP_FRESH_REDUCE", kstep(True, "blocks")),
        define("MSA_SCAN4_KSTEP_FRESH_FOLD", kstep(True, "fold")),
        define("MSA_SCAN4_KSTEP_FRESH_UNITS", kstep(True, "units")),
        define("MSA_SCAN4_REDUCE", reduction()),
        define("MSA_SCAN4_REDUCE_UNITS", reduction(True)),
        *(define(f"MSA_SCAN4_UNIT_READ_{i}", [f"v_mov_b32 %{x}, v{VUNIT + 8 * i + x}" for x in range(8)]) for i in range(4)),
        define("MSA_SCAN4_MAX_READ", [f"v_mov_b32 %{x}, v{VMAX + x}" for x in range(8)]),
        define("MSA_SCAN4_FRAGS0", frags0()),
        define("MSA_SCAN4_LOAD8", load8(VOFF)),
        define("MSA_SCAN4_LOAD8_NT", load8(VOFF, " nt")),
        define("MSA_SCAN4_SET_ADDR", set_registers(VADDR, 4)),
        define("MSA_SCAN4_SET_VOFF", set_registers(VOFF, 8)),
        # the fold's per-lane constants from l32 = lane & 31 (operand 0)
        define("MSA_SCAN4_SET_FOLD", [
            f"v_lshlrev_b32 v{V_LOWMASK}, %0, 2", f"v_add_u32 v{V_LOWMASK}, -1, v{V_LOWMASK}",      # (2 << l32) - 1
            f"v_add_u32 v{V_DISTBASE}, -31, %0", f"v_add_u32 v{V_L32P1}, 1, %0",
            f"v_cmp_eq_u32 vcc, 31, %0", f"v_cndmask_b32 v{V_IS31}, 0, 1, vcc", f"v_and_b32 v{V_L15}, 15, %0"]),
        clobbers("MSA_SCAN4_CLOBBERS"),
        clobbers("MSA_SCAN4_UNITS_CLOBBERS", VUNIT)])


# ---------------------------------------------------------------------------------------------------------------
# The tiled products' ends under the next tile's steps (tile_flow_kernel).  A tile's first step rounds the accumulators of the tile
# before to bf16, a block in front of the MFMA that overwrites it, into 128 held registers; each of the next eight steps finishes one
# column block of them (128 weight rows x 16 tokens) behind its MFMAs and stores it.  Held registers of column j, row block i, pair of
# rows p: number 16 j + 2 i + p.
HOLD_LOW = 24                       # compiler code has the registers below
TEMP = list(range(202, 208)) + list(range(248, 255))
V_GELU = 255                        # a constant of gelu
LOG2E = 1.4426950408889634
S_LOW, S_ROW = "s[76:77]", "s78"    # lanes whose token is one of the first eight of its sixteen; byte offset of the column's rows


def hold(n):
    return HOLD_LOW + n if n < 128 - HOLD_LOW else 224 + n - (128 - HOLD_LOW)


def hex_f32(x):
    import struct
    return f"{struct.unpack('<I', struct.pack('<f', x))[0]:#010x}"


def pack_block(tile, i, j, t):
    """Four accumulators, rounded, into two held registers; t: four scratch registers."""
    b, h = (i * tile.b + j) * 4, 16 * j + 2 * i
    return [f"v_accvgpr_read_b32 v{t[x]}, a{b + x}" for x in range(4)] + \
           [f"v_cvt_pk_bf16_f32 v{hold(h + p)}, v{t[2 * p]}, v{t[2 * p + 1]}" for p in range(2)]


def gelu_pair(r, t):
    """The tanh form of gelu of the two values in r: z / (1 + 2^(z (a + b z^2)))."""
    a, b = -1.5957691216057308 * LOG2E, -1.5957691216057308 * 0.044715 * LOG2E
    lo, hi, u, w = t
    return [f"v_lshlrev_b32 v{lo}, 16, v{r}", f"v_and_b32 v{hi}, 0xffff0000, v{r}",
            f"v_mul_f32 v{u}, v{lo}, v{lo}", f"v_mul_f32 v{w}, v{hi}, v{hi}",
            f"v_fmamk_f32 v{u}, v{u}, {hex_f32(b)}, v{V_GELU}", f"v_fmamk_f32 v{w}, v{w}, {hex_f32(b)}, v{V_GELU}",
            f"v_mul_f32 v{u}, v{u}, v{lo}", f"v_mul_f32 v{w}, v{w}, v{hi}",
            f"v_exp_f32 v{u}, v{u}", f"v_exp_f32 v{w}, v{w}", "s_nop 0",
            f"v_add_f32 v{u}, 1.0, v{u}", f"v_add_f32 v{w}, 1.0, v{w}",
            f"v_rcp_f32 v{u}, v{u}", f"v_rcp_f32 v{w}, v{w}", "s_nop 0",
            f"v_mul_f32 v{lo}, v{lo}, v{u}", f"v_mul_f32 v{hi}, v{hi}, v{w}",
            f"v_cvt_pk_bf16_f32 v{r}, v{lo}, v{hi}"]


def gated_pair(mode, gate, up, t):
    """The two gated units of the gates in one register and the ups in another, into the gates' register."""
    g0, g1, e0, e1, u0, u1 = t
    o = [f"v_lshlrev_b32 v{g0}, 16, v{gate}", f"v_and_b32 v{g1}, 0xffff0000, v{gate}",
         f"v_lshlrev_b32 v{u0}, 16, v{up}", f"v_and_b32 v{u1}, 0xffff0000, v{up}"]
    if mode == "glu":
        o += [f"v_min_f32 v{g0}, %[limit], v{g0}", f"v_min_f32 v{g1}, %[limit], v{g1}",
              f"v_max_f32_e64 v{u0}, -%[limit], v{u0}", f"v_max_f32_e64 v{u1}, -%[limit], v{u1}",
              f"v_min_f32 v{u0}, %[limit], v{u0}", f"v_min_f32 v{u1}, %[limit], v{u1}",
              f"v_mul_f32 v{e0}, %[rate], v{g0}", f"v_mul_f32 v{e1}, %[rate], v{g1}",
              f"v_add_f32 v{u0}, %[shift], v{u0}", f"v_add_f32 v{u1}, %[shift], v{u1}"]
    else:
        o += [f"v_mul_f32 v{e0}, {hex_f32(-LOG2E)}, v{g0}", f"v_mul_f32 v{e1}, {hex_f32(-LOG2E)}, v{g1}"]
    return o + [f"v_exp_f32 v{e0}, v{e0}", f"v_exp_f32 v{e1}, v{e1}", "s_nop 0",
                f"v_add_f32 v{e0}, 1.0, v{e0}", f"v_add_f32 v{e1}, 1.0, v{e1}",
                f"v_rcp_f32 v{e0}, v{e0}", f"v_rcp_f32 v{e1}, v{e1}", "s_nop 0",
                f"v_mul_f32 v{g0}, v{g0}, v{e0}", f"v_mul_f32 v{g1}, v{g1}, v{e1}",
                f"v_mul_f32 v{g0}, v{g0}, v{u0}", f"v_mul_f32 v{g1}, v{g1}, v{u1}",
                f"v_cvt_pk_bf16_f32 v{gate}, v{g0}, v{g1}"]


def whole_lines(p0, p1, at, so):
    """Two 16-byte groups of every token, 32 columns apart: token t's lanes and those of token t + 8 change halves, so that a store
    writes whole cache lines of eight tokens.  at: registers for the two stores' offsets.  (instructions, stores)"""
    t = TEMP[2:6]
    o = [f"v_add_u32 v{at[0]}, {S_ROW}, %[{so}]", f"v_add_u32 v{at[1]}, %[row8], v{at[0]}"]
    o += [f"v_cndmask_b32_e64 v{t[k]}, v{p0 + k}, v{p1 + k}, {S_LOW}" for k in range(4)]
    o += [f"v_mov_b32_dpp v{t[k]}, v{t[k]} row_ror:8 row_mask:0xf bank_mask:0xf" for k in range(4)]
    o += [f"v_cndmask_b32_e64 v{p0 + k}, v{t[k]}, v{p0 + k}, {S_LOW}" for k in range(4)]
    o += [f"v_cndmask_b32_e64 v{p1 + k}, v{p1 + k}, v{t[k]}, {S_LOW}" for k in range(4)]
    return o, [f"buffer_store_dwordx4 v[{p}:{p + 3}], v{v}, %[ro], 0 offen@NT" for p, v in ((p0, at[0]), (p1, at[1]))]


def finish_column(mode, j):
    """(instructions, stores) of column block j."""
    h = lambda n: hold(16 * j + n)
    o, stores = [f"s_mov_b32 s76, 0x00ff00ff", "s_mov_b32 s77, 0x00ff00ff", f"s_mul_i32 {S_ROW}, %[row16], {j}"], []
    if mode == "gelu":
        for n in range(0, 16, 2):
            o += interleave(gelu_pair(h(n), TEMP[0:4]), gelu_pair(h(n + 1), TEMP[6:10]))
    if mode in ("silu", "glu"):
        for m in range(2):
            for n in range(0, 4, 2):
                o += interleave(gated_pair(mode, h(8 * m + n), h(8 * m + 4 + n), TEMP[0:6]),
                                gated_pair(mode, h(8 * m + n + 1), h(8 * m + 5 + n), TEMP[6:12]))
        a, b = whole_lines(h(0), h(8), (TEMP[0], TEMP[1]), "so0")
        return o + a, stores + b
    for m, so, at in ((0, "so0", (TEMP[0], TEMP[1])), (2, "so1", (TEMP[6], TEMP[7]))):
        a, b = whole_lines(h(4 * m), h(4 * m + 4), at, so)
        o, stores = o + a, stores + b
    return o, stores


SETTLE = ["s_nop 15", "s_nop 7"]     # an MFMA's result may be read 18 wait states after its issue at the earliest


def pack_all(tile):
    return SETTLE + [x for i in range(tile.a) for j in range(tile.b) for x in pack_block(tile, i, j, TEMP[0:4] if j % 2 else TEMP[6:10])]


def piece(tile):
    """The accumulators as they are, 1 KB a block, to a partial tile ([rp], [vp] the lane's offset, [sp] the wavefront's)."""
    out = SETTLE + ["s_mov_b32 s79, %[sp]"]
    for n, (j, i) in enumerate((j, i) for j in range(tile.b) for i in range(tile.a)):
        t = TEMP[2:6] if n % 2 else TEMP[6:10]
        out += [f"v_accvgpr_read_b32 v{t[x]}, a{(i * tile.b + j) * 4 + x}" for x in range(4)]
        out.append(f"buffer_store_dwordx4 v[{t[0]}:{t[3]}], %[vp], %[rp], s79 offen offset:{n % 4 * 1024}")
        if n % 4 == 3:
            out.append("s_add_u32 s79, s79, 0x1000")
    return out


def gemm_text():
    tile = SCAN
    step = lambda fresh, **kw: kstep(fresh, voff_b=VOFF_B, nt="", **kw)
    parts = [HEADER,
             define("MSA_GEMM_KSTEP", step(False)),
             define("MSA_GEMM_KSTEP_FRESH", step(True)),
             define("MSA_GEMM_FRAGS0", frags0()),
             define("MSA_GEMM_LOAD8_A", load8(VOFF)),
             define("MSA_GEMM_LOAD8_B", load8(VOFF_B)),
             define("MSA_GEMM_SET_ADDR", set_registers(VADDR, 4)),
             *(define(f"MSA_GEMM_SET_VOFF_{name}{h}", set_registers(first + 4 * h, 4)) for name, first in (("A", VOFF), ("B", VOFF_B)) for h in range(2)),
             define("MSA_GEMM_SETTLE", SETTLE)]
    # four of the eight row blocks of a column block, sixteen accumulators
    for j in range(8):
        for h in range(2):
            parts.append(define(f"MSA_GEMM_ACC_{j}_{h}", [f"v_accvgpr_read_b32 %{4 * i + r}, a{((4 * h + i) * 8 + j) * 4 + r}"
                                                          for i in range(4) for r in range(4)]))
    packs = [[pack_block(tile, i, j, TEMP[0:4] if j % 2 else TEMP[6:10]) for j in range(tile.b)] for i in range(tile.a)]
    parts.append(define("MSA_GEMM_KSTEP_FRESH_PACK", step(True, early_fillers=packs)))
    parts.append(define("MSA_GEMM_PACK", pack_all(tile)))
    parts.append(define("MSA_GEMM_PIECE", piece(tile)))
    parts.append(define("MSA_GEMM_SET_GELU", [f"v_mov_b32 v{V_GELU}, {hex_f32(-1.5957691216057308 * LOG2E)}"]))
    for mode in ("store", "gelu", "silu", "glu"):
        for j in range(tile.b):
            work, stores = finish_column(mode, j)
            parts.append(define(f"MSA_GEMM_KSTEP_{mode.upper()}_{j}(NT)", step(False, fillers=work, stores=stores)))
            parts.append(define(f"MSA_GEMM_END_{mode.upper()}_{j}(NT)", fix_lane_move_hazards(work + stores)))
    parts.append(clobbers("MSA_GEMM_CLOBBERS"))
    parts.append(clobbers("MSA_GEMM_FLOW_CLOBBERS", HOLD_LOW))
    return "\n".join(parts)


def main():
    """``scan_asm.inc`` (``--check``: is it what would be written?) and, always, ``gemm_asm.inc``, which every build writes again."""
    here = os.path.dirname(os.path.abspath(__file__))
    path, text = os.path.join(here, "gemm_asm.inc"), gemm_text()
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as f:
            f.write(text)
    path, text = os.path.join(here, "scan_asm.inc"), scan_text()
    if len(sys.argv) > 1 and sys.argv[1] == "--check":
        return 0 if open(path).read() == text else 1
    with open(path, "w") as f:
        f.write(text)
    return 0


if __name__ == "__main__":
    sys.exit(main())
