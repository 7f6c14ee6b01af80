#!/usr/bin/env python3
"""Generator of the hand-scheduled gfx950 assembly of the fused fp32 Winograd F(2x2,3x3) kernel on
the bf16 matrix instructions.

Every fp32 operand is split into three bf16 pieces, x = h + m + l (round to nearest each, exact:
3 x 8 significant bits and two signs cover the 24 of fp32), and a product of two operands is the
sum of six products of pieces, U_l V_h + U_h V_l + U_h V_m + U_m V_h + U_h V_h + U_m V_m, on
v_mfma_f32_32x32x16_bf16 with its fp32 accumulators; the three products that are left out are below
2^-25 of the result's terms.  An 8-channel chunk is three MFMAs per position, filter group and column
group: the 16 values of K hold two pieces of the lane half's four channels.

Why: v_mfma_f32_32x32x2_f32 takes 64 cycles for 2 channels and shares the SIMD's ALUs with every
vector instruction; 3 bf16 MFMAs take 96 cycles for 8 channels, and vector instructions run next to
them.  Against 64 bits the sums are nearer than those of the fp32 MFMA (relative 2-norm error of a
dot product over 64 / 512 / 1024 channels: 1.1e-7 / 3.4e-7 / 4.9e-7 against 1.5e-7 / 4.1e-7 /
5.7e-7): there are fewer roundings on the way.

Range: bf16 has no exponents below fp32's, so the pieces of a value below 2^-110 would fall off the end of
bf16's grid, 2^-133.  Every operand is therefore split times 2^16: fp32's own grid, 2^-149, then lies on
bf16's, and the pieces are exact for every value up to 2^112.  The outputs are stored times 2^-32.  V gets
its factor in the input transform (six instructions a patch), U in front of its split (one a value):
14 of 241 vector instructions a unit, 0.4 ... 2.4 % of a call (N=1 C=K=64 14x14 19.7 -> 20.2 us,
N=128 C=K=512 7x7 106.0 -> 106.5).  Deciding by the magnitude of operands or outputs instead where the pieces would lose
bits takes both operands' largest and smallest values, of all waves; an output's neighbours do not tell.

What the pieces cannot hold: infinities and NaNs (their residual is NaN), operands of 2^112 or more and
outputs of 2^94 or more (infinite once scaled).  A lane therefore sums the magnitudes of the outputs it stores;
where a sum is not finite, or close to it, the workgroup computes the tiles that it stores once more with
v_mfma_f32_32x32x2_f32 (exact_chunk), which is what gen_wino_f32_asm.py's kernels always use, and
stores them again: a launch then takes 2 to 5 times as long (one NaN, fused kernel: N=128 C=K=128 28x28 98 -> 244 us,
N=128 C=K=512 7x7 106 -> 252, N=32 C=K=512 7x7 38 -> 183, whose tiles the second pass does not cut).

What bounds it: power on layers that fill the chip (N=128 C=K=512 7x7 runs at 2.07 GHz, the fp32 MFMA
kernel at 2.49; with every wait taken out it takes as long, at a lower clock), issue on small ones (two
waves per SIMD, some 370 instructions a unit each; without its MFMAs a unit takes 96 % of the time).
Fused kernel on the fp32 MFMA / here, us: N=64 C=K=64 56x56 64.4 / 59.7, N=128 C=K=128 28x28 110 / 97,
C=K=256 14x14 106 / 95, C=K=512 7x7 127 / 105, N=1 C=K=64 14x14 22.5 / 17.8.  Layers of 17 to 48 channels run
these kernels, and packed columns that break quads of images where their units are few; the others, of those figures too,
the kernels of gen_wino_f32_half_asm.py, which take this one's place with three products instead of six.

Workgroup: eight waves, one tile of 64 filters x 64 columns (2 x 2 MFMA tiles) for all 16 positions.
Wave w holds positions 2w and 2w + 1: every U and every V element is read, and split, by one wave of
the workgroup only; two waves per SIMD, so that one's vector instructions run next to the other's
MFMAs.  The position pairs meet in the output transform, through LDS: two rounds (one per
filter group) of 128 KB.

LDS, 160 KB: V[pos][channel][column] of one chunk is 32 KB (columns of odd channels swapped in halves
against bank conflicts); the two buffers are the first and the last 32 KB, so that the 128 KB next to
the live one are contiguous for the output transform.

Units, ranges, cursors, place() and the hand-over protocol are those of gen_wino_f32_asm.py; all
merges of a published partial tile happen in the output transform.

Usage: gen_wino_f32_split_asm.py > wino_f32_split_asm.s
"""
import sys

from gen_wino_f32_asm import FLAGS, OOB, Alloc, Kernel, a, cached_forms, s, v

BUFFER_SWAP = 0x20000       # the two V buffers: bytes 0 .. 32K and 128K .. 160K
LDS_BYTES = 160 * 1024
STORES = 32                 # stores of an output transform, per wave
SUM_LARGE = 0x7E800000      # 2^126
SCALE = 0x47800000          # 2^16, on U and on V
UNSCALE = 0x2F800000        # 2^-32


class KernelSplit(Kernel):
    SLAB_CHANNELS = 1
    SCALARS = ["MaskHi", "Scale", "Unscale"]  # registers of constants()
    SPLIT_SCALES = {"A": "Scale"}  # scalar registers that operands meet in front of their split

    def __init__(self, KW, ragged=False, packed=False):
        """KW = 2: the line of tiles is filter-block major.  KW = 4: the two blocks of a pair of filter
        blocks are neighbours on the line, column block by column block, and share patches in L2."""
        self.KW = KW
        self.ragged = ragged
        self.packed = packed
        self.lines = []
        self.outofline = []
        self.nlabel = 0
        self.name = f"wino_f32_asm_kw{KW}" + ("_packed" if packed else "_ragged" if ragged else "")
        self.alloc()

    # ------------------------------------------------------------------ registers
    def alloc_sgprs(self):
        S = Alloc(42, 102)
        names = ["N", "H", "W", "Chunks", "TilesW", "Ngroups", "Colgroups", "Colblocks", "Q", "HWN4",
                 "UnitsQ", "UnitsRem", "UswBytes", "GridPerXcd", "Mch", "Sch", "Mcb", "Scb", "Mng",
                 "Sng", "Mtw", "Stw", "Creal", "Kreal", "Timeline", "TimelineHi"]
        self.S = {n: 16 + i for i, n in enumerate(names)}
        self.S.update(X=8, U=10, Y=12, Sync=14, Status=4, SpinLimit=6)
        for n in ["L", "Wave", "Begin", "Nunits", "G", "Tp", "Cp", "Tq", "Cq", "Tm", "Cm",
                  "SegEnd", "Kind", "ColStep", "RowStep", "Uoff0", "Uoff1",
                  "Dkb", "DkbPrev", "DkbM", "Spin", "Stamps", "Bad", "Buf", *self.SCALARS, "PlaceTn"]:
            self.S[n] = S.get(n)
        self.S["RsrcX"] = S.get("RsrcX", 4, 4)
        self.S["RsrcU"] = S.get("RsrcU", 4, 4)
        self.S["RsrcY"] = S.get("RsrcY", 4, 4)
        self.S["Fl"] = S.get("Fl", 2, 2)
        self.S["M"] = S.get("M", 2, 2)
        self.S["T"] = S.get("T", 8, 2)
        self.S.update(PlaceM=3, PlaceS=7, PlaceG=self.S["GridPerXcd"])
        self.sgpr_count = S.next

    def alloc_vgprs(self):
        V = Alloc(1, 128)
        self.V = {}
        for n, cnt, al in [("Lane16", 1, 1), ("Lds0", 1, 1), ("Lds1", 1, 1), ("LdsWr", 1, 1),
                           ("EffP", 1, 1), ("EffPrev", 1, 1), ("Tmp", 2, 1), ("Eff", 4, 1),
                           ("Sum", 1, 1), ("VOFF", 16, 1), ("P", 16, 1), ("U", 16, 4),
                           # 64 registers that hold nothing between two chunks: the output transform's
                           ("EX", 64, 4)]:
            self.V[n] = V.get(n, cnt, al)
        ex = self.V["EX"]
        # constants of the flag accesses, written in front of them
        self.V["One"], self.V["Zero"] = self.V["Tmp"], self.V["Tmp"] + 1
        self.V.update(A0=ex, A1=ex + 6, B0=ex + 12, B1=ex + 20, S4=ex + 28, VR=ex + 32, T=ex + 48)
        self.vgpr_count = V.next

    # ------------------------------------------------------------------ tiles
    def split_tile(self, T):
        """Workgroup tile T -> Dkb (block of 64 filters) and T0 (block of 64 columns)."""
        t = self.t
        self.place(T)
        self.div(self.sr("Dkb"), t(5), self.sr("Mcb"), self.sr("Scb"))
        self.e(f"s_mul_i32 {t(0)}, {self.sr('Dkb')}, {self.sr('Colblocks')}")
        self.e(f"s_sub_u32 {t(0)}, {t(5)}, {t(0)}")
        if self.KW == 4:  # Colblocks counts the column blocks of both filter blocks of a pair
            self.e(f"s_lshl_b32 {self.sr('Dkb')}, {self.sr('Dkb')}, 1")
            self.e(f"s_and_b32 {t(1)}, {t(0)}, 1")
            self.e(f"s_add_u32 {self.sr('Dkb')}, {self.sr('Dkb')}, {t(1)}")
            self.e(f"s_lshr_b32 {t(0)}, {t(0)}, 1")

    def vdiv(self, dst, x, m, sh, tmp):
        """dst = x / d per lane, the magic number in two SGPRs; tmp: an even pair of T registers."""
        T = lambda i, n=1: self.vr("T", i, n)
        self.e(f"v_mul_lo_u32 {T(tmp)}, {x}, {m}")
        self.e(f"v_mul_hi_u32 {T(tmp + 1)}, {x}, {m}")
        self.e(f"v_lshrrev_b64 {T(tmp, 2)}, {sh}, {T(tmp, 2)}")
        self.e(f"v_mov_b32 {dst}, {T(tmp)}")

    def decode(self, tile):
        """Tile -> Dkb, and per lane (= column of the tile) T[0] = batch element * 4, T[1] = 2*ty,
        T[2] = 2*tx, T[3] = 0 or, for a column that does not exist, the out-of-range bit."""
        t, e = self.t, self.e
        T = lambda i: self.vr("T", i)
        self.split_tile(tile)
        e(f"v_mov_b32 {T(15)}, 0x{OOB:x}")  # for the range checks here and in the offsets
        e(f"v_mov_b32 {T(14)}, 0")
        e(f"v_lshrrev_b32 {T(8)}, 4, {self.vr('Lane16')}")                  # lane
        e(f"s_add_u32 {t(2)}, {self.sr('H')}, 1")
        e(f"s_lshr_b32 {t(2)}, {t(2)}, 1")                                  # tile rows
        if self.packed:
            # column (spatial tile, n) of the line lies at tile * N + n; the slot Mng / Sng divides by N
            e(f"s_lshl_b32 {t(0)}, {t(0)}, 6")
            e(f"v_add_u32 {T(1)}, {t(0)}, {T(8)}")
            self.vdiv(T(6), T(1), self.sr("Mng"), self.sr("Sng"), 4)        # spatial tile
            e(f"v_mul_lo_u32 {T(5)}, {T(6)}, {self.sr('N')}")
            e(f"v_sub_u32 {T(0)}, {T(1)}, {T(5)}")                          # batch element
            e(f"s_mul_i32 {t(4)}, {t(2)}, {self.sr('TilesW')}")
            e(f"v_cmp_gt_u32 vcc, {t(4)}, {T(6)}")
            e(f"v_cndmask_b32 {T(3)}, {T(15)}, {T(14)}, vcc")
        else:
            e(f"s_lshl_b32 {t(0)}, {t(0)}, 1")
            e(f"v_lshrrev_b32 {T(1)}, 5, {T(8)}")
            e(f"v_add_u32 {T(1)}, {t(0)}, {T(1)}")                          # column tile of 32
            e(f"v_cmp_gt_u32 vcc, {self.sr('Colgroups')}, {T(1)}")
            e(f"v_cndmask_b32 {T(3)}, {T(15)}, {T(14)}, vcc")
            # divisor: the spatial tiles (bit 6 of the shift) or the image groups, whichever is the fast index
            self.vdiv(T(6), T(1), self.sr("Mng"), self.sr("Sng"), 4)
            e(f"v_mul_lo_u32 {T(5)}, {T(6)}, {self.sr('Ngroups')}")
            e(f"v_sub_u32 {T(7)}, {T(1)}, {T(5)}")
            e(f"s_bitcmp1_b32 {self.sr('Sng')}, 6")
            e(f"s_cselect_b64 vcc, -1, 0")
            e(f"v_cndmask_b32 {T(0)}, {T(7)}, {T(6)}, vcc")                 # image group
            e(f"v_cndmask_b32 {T(6)}, {T(6)}, {T(7)}, vcc")                 # spatial tile
            e(f"v_and_b32 {T(5)}, 31, {T(8)}")
            e(f"v_lshl_add_u32 {T(0)}, {T(0)}, 5, {T(5)}")                  # batch element
            if self.ragged:
                e(f"v_cmp_gt_u32 vcc, {self.sr('N')}, {T(0)}")
                e(f"v_cndmask_b32 {T(3)}, {T(15)}, {T(3)}, vcc")
        self.vdiv(T(1), T(6), self.sr("Mtw"), self.sr("Stw"), 4)            # row-major reading
        e(f"v_mul_lo_u32 {T(5)}, {T(1)}, {self.sr('TilesW')}")
        e(f"v_sub_u32 {T(2)}, {T(6)}, {T(5)}")
        if not self.packed:
            # bit 6 of the shift Stw: strips of two tile rows, zigzag (see Kernel.decode)
            e(f"v_or_b32 {T(4)}, 1, {T(1)}")
            e(f"v_cmp_gt_u32 vcc, {t(2)}, {T(4)}")                          # the strip has two rows
            e(f"s_bitcmp1_b32 {self.sr('Stw')}, 6")
            e(f"s_cselect_b64 {s(self.S['T'] + 6, 2)}, -1, 0")
            e(f"s_and_b64 vcc, vcc, {s(self.S['T'] + 6, 2)}")
            e(f"v_and_b32 {T(4)}, 1, {T(1)}")
            e(f"v_mul_lo_u32 {T(4)}, {T(4)}, {self.sr('TilesW')}")
            e(f"v_add_u32 {T(4)}, {T(4)}, {T(2)}")                          # position inside the strip
            e(f"v_and_b32 {T(5)}, -2, {T(1)}")
            e(f"v_and_b32 {T(6)}, 1, {T(4)}")
            e(f"v_or_b32 {T(5)}, {T(5)}, {T(6)}")
            e(f"v_lshrrev_b32 {T(4)}, 1, {T(4)}")
            e(f"v_cndmask_b32 {T(1)}, {T(1)}, {T(5)}, vcc")
            e(f"v_cndmask_b32 {T(2)}, {T(2)}, {T(4)}, vcc")
        e(f"v_lshlrev_b32 {T(0)}, 2, {T(0)}")
        e(f"v_lshlrev_b32 {T(1)}, 1, {T(1)}")
        e(f"v_lshlrev_b32 {T(2)}, 1, {T(2)}")

    def in_range(self, dst, x, limit, extra):
        """dst = extra, or the out-of-range bit (T[15], as decode leaves it) unless 0 <= x < limit (x a
        VGPR, limit an SGPR)."""
        self.e(f"v_cmp_gt_u32 vcc, {limit}, {x}")  # unsigned: also rejects -1
        self.e(f"v_cndmask_b32 {dst}, {self.vr('T', 15)}, {extra}, vcc")

    def patch_offsets(self):
        """VOFF: byte offsets of the 16 patch elements inside a channel; zero padding and columns that do
        not exist get the out-of-range bit, which no num_records reaches."""
        T = lambda i: self.vr("T", i)
        e = self.e
        for i in range(4):
            e(f"v_add_u32 {T(12)}, {i - 1}, {T(1)}")
            self.in_range(T(4 + i), T(12), self.sr("H"), T(3))
        for j in range(4):
            e(f"v_add_u32 {T(12)}, {j - 1}, {T(2)}")
            self.in_range(T(8 + j), T(12), self.sr("W"), T(14))
        # element (0, 0): ((2ty - 1) * W + 2tx - 1) * N * 4 + n * 4
        e(f"v_add_u32 {T(13)}, -1, {T(1)}")
        e(f"v_mul_lo_u32 {T(13)}, {T(13)}, {self.sr('RowStep')}")
        e(f"v_add_u32 {T(12)}, {T(0)}, {T(13)}")
        e(f"v_add_u32 {T(13)}, -1, {T(2)}")
        e(f"v_mul_lo_u32 {T(13)}, {T(13)}, {self.sr('ColStep')}")
        e(f"v_add_u32 {T(12)}, {T(12)}, {T(13)}")
        for i in range(4):
            e(f"v_mov_b32 {T(13)}, {T(12)}")
            for j in range(4):
                e(f"v_or3_b32 {self.vr('VOFF', i * 4 + j)}, {T(13)}, {T(4 + i)}, {T(8 + j)}")
                if j < 3:
                    e(f"v_add_u32 {T(13)}, {self.sr('ColStep')}, {T(13)}")
            if i < 3:
                e(f"v_add_u32 {T(12)}, {self.sr('RowStep')}, {T(12)}")

    def pack_store_offset(self):
        """EffP: byte offset of the lane's first output inside a filter's image (a multiple of four, below
        2^30), bit 0 / 1: the second output row / column does not exist, bit 31: nothing does."""
        T = lambda i: self.vr("T", i)
        e = self.e
        for d, (x, limit) in enumerate(((T(1), "H"), (T(2), "W"))):
            e(f"v_add_u32 {T(12)}, 1, {x}")
            e(f"v_cmp_gt_u32 vcc, {self.sr(limit)}, {T(12)}")
            e(f"v_cndmask_b32 {T(4 + d)}, {1 + d}, {T(14)}, vcc")
        e(f"v_mul_lo_u32 {T(13)}, {T(1)}, {self.sr('RowStep')}")
        e(f"v_mul_lo_u32 {T(12)}, {T(2)}, {self.sr('ColStep')}")
        e(f"v_add3_u32 {T(12)}, {T(0)}, {T(12)}, {T(13)}")
        e(f"v_or3_b32 {T(12)}, {T(12)}, {T(4)}, {T(5)}")
        e(f"v_or_b32 {self.vr('EffP')}, {T(12)}, {T(3)}")

    def store_offsets(self):
        """Eff[0..3]: byte offsets of the lane's four outputs, or out of range, from the packed one in Eff[0]."""
        e = self.e
        eff = lambda i: self.vr("Eff", i)
        e(f"v_lshlrev_b32 {eff(2)}, 31, {eff(0)}")               # no second row
        e(f"v_and_b32 {eff(1)}, 2, {eff(0)}")
        e(f"v_lshlrev_b32 {eff(1)}, 30, {eff(1)}")               # no second column
        e(f"v_and_b32 {eff(0)}, -4, {eff(0)}")
        e(f"v_add_u32 {eff(3)}, {self.sr('RowStep')}, {eff(0)}")
        e(f"v_add_u32 {eff(3)}, {self.sr('ColStep')}, {eff(3)}")
        e(f"v_or3_b32 {eff(3)}, {eff(3)}, {eff(2)}, {eff(1)}")
        e(f"v_add_u32 {self.vr('Tmp', 1)}, {self.sr('RowStep')}, {eff(0)}")
        e(f"v_or_b32 {eff(2)}, {self.vr('Tmp', 1)}, {eff(2)}")
        e(f"v_add_u32 {self.vr('Tmp', 1)}, {self.sr('ColStep')}, {eff(0)}")
        e(f"v_or_b32 {eff(1)}, {self.vr('Tmp', 1)}, {eff(1)}")

    # ------------------------------------------------------------------ loads
    def channel_descriptor(self):
        """RsrcX = channel 8 * Cp + wave; empty when the channel does not exist."""
        t, e, rx = self.t, self.e, self.S["RsrcX"]
        e(f"s_lshl_b32 {t(0)}, {self.sr('Cp')}, 3")
        e(f"s_add_u32 {t(0)}, {t(0)}, {self.sr('Wave')}")
        if self.ragged:
            e(f"s_cmp_lt_u32 {t(0)}, {self.sr('Creal')}")
            e(f"s_cselect_b32 {s(rx + 2)}, {self.sr('HWN4')}, 0")
        e(f"s_mul_hi_u32 {t(1)}, {t(0)}, {self.sr('HWN4')}")
        e(f"s_mul_i32 {t(0)}, {t(0)}, {self.sr('HWN4')}")
        e(f"s_add_u32 {s(rx)}, {s(self.S['X'])}, {t(0)}")
        e(f"s_addc_u32 {s(rx + 1)}, {s(self.S['X'] + 1)}, {t(1)}")

    def filter_offsets(self):
        """Uoff0 / Uoff1: byte offsets, in Ww, of the wave's positions of chunk Cq of the two filter groups
        of tile Tq (P's tile or the one before it)."""
        t, e = self.t, self.e
        e(f"s_cmp_eq_u32 {self.sr('Tq')}, {self.sr('Tp')}")
        e(f"s_cselect_b32 {t(0)}, {self.sr('Dkb')}, {self.sr('DkbPrev')}")
        e(f"s_lshl_b32 {t(0)}, {t(0)}, 1")
        e(f"s_mul_i32 {t(0)}, {t(0)}, {self.sr('Q')}")
        e(f"s_lshl_b32 {t(1)}, {self.sr('Cq')}, 1")
        e(f"s_add_u32 {t(0)}, {t(0)}, {t(1)}")
        e(f"s_lshl_b32 {t(2)}, {self.sr('Wave')}, 10")
        e(f"s_add_u32 {t(1)}, {t(0)}, {self.sr('Q')}")
        for kg in range(2):
            e(f"s_lshl_b32 {t(kg)}, {t(kg)}, 13")
            e(f"s_add_u32 {self.sr(f'Uoff{kg}')}, {t(kg)}, {t(2)}")

    def advance_p(self, ahead=2):
        """P cursor -> unit G + ahead when there is one; the tile switch lives out of line."""
        rare, back = self.newlabel("p_switch"), self.newlabel("p_back")
        t, e = self.t, self.e
        e(f"s_add_u32 {t(0)}, {self.sr('G')}, {ahead}")
        e(f"s_cmp_lt_u32 {t(0)}, {self.sr('Nunits')}")
        e(f"s_addc_u32 {self.sr('Cp')}, {self.sr('Cp')}, 0")
        e(f"s_cmp_eq_u32 {self.sr('Cp')}, {self.sr('Chunks')}")
        e(f"s_cbranch_scc1 {rare}")
        self.label(back)
        main, self.lines = self.lines, []
        self.label(rare)
        e(f"s_mov_b32 {self.sr('Cp')}, 0")
        e(f"s_add_u32 {self.sr('Tp')}, {self.sr('Tp')}, 1")
        e(f"s_mov_b32 {self.sr('DkbPrev')}, {self.sr('Dkb')}")
        e(f"v_mov_b32 {self.vr('EffPrev')}, {self.vr('EffP')}")
        self.p_tile()
        e(f"s_branch {back}")
        self.outofline.extend(self.lines)
        self.lines = main

    def p_tile(self):
        """What the lanes know about P's tile: VOFF, EffP and Dkb."""
        self.decode(self.sr("Tp"))
        self.patch_offsets()
        self.pack_store_offset()

    def advance_q(self):
        """Q cursor -> unit G + 1 when there is one."""
        t, e = self.t, self.e
        e(f"s_add_u32 {t(0)}, {self.sr('G')}, 1")
        e(f"s_cmp_lt_u32 {t(0)}, {self.sr('Nunits')}")
        e(f"s_addc_u32 {self.sr('Cq')}, {self.sr('Cq')}, 0")
        e(f"s_cmp_eq_u32 {self.sr('Cq')}, {self.sr('Chunks')}")
        e(f"s_cselect_b32 {self.sr('Cq')}, 0, {self.sr('Cq')}")
        e(f"s_addc_u32 {self.sr('Tq')}, {self.sr('Tq')}, 0")

    def u_load_items(self, kg):
        """The wave's two positions of filter group kg, 8 channels: two 16-byte loads."""
        load = lambda q, off: (f"buffer_load_dwordx4 {self.vr('U', kg * 8 + 4 * q, 4)}, {self.vr('Lane16')}, "
                               f"{self.sr('RsrcU', 4)}, {off} offen")
        return [("vm", f"U{kg}", load(0, self.sr(f"Uoff{kg}"))), f"s_add_u32 {self.sr('M')}, {self.sr(f'Uoff{kg}')}, 0x2000",
                ("vm", f"U{kg}", load(1, self.sr("M")))]

    def patch_load(self, dst, p):
        return f"buffer_load_dword {self.vr(dst, p)}, {self.vr('VOFF', p)}, {self.sr('RsrcX', 4)}, 0 offen"

    def patch_items(self, src):
        return [("vm", src, self.patch_load(src, p)) for p in range(16)]

    # ------------------------------------------------------------------ pieces of a chunk
    def split_operand(self, raw, kind, dst):
        """Instructions that turn four fp32 registers (channels of the lane half, in pairs) into bf16
        pieces: A = [l l h h m m], B = [h h m m h h l l] (two registers per piece).  A (filters) is scaled
        here (SPLIT_SCALES), B was in the transform."""
        x = lambda i: v(raw[i])
        t = lambda i: self.vr("S4", i)
        h, m, l = ((2, 4, 0) if kind == "A" else (0, 2, 6))
        scale = self.SPLIT_SCALES.get(kind)
        out = [f"v_mul_f32 {x(i)}, {self.sr(scale)}, {x(i)}" for i in range(4)] if scale else []
        for q in range(2):
            out.append(f"v_cvt_pk_bf16_f32 {v(dst + h + q)}, {x(2 * q)}, {x(2 * q + 1)}")
        for piece, nxt in ((h, m), (m, l)):
            for q in range(2):
                out.append(f"v_lshlrev_b32 {t(2 * q)}, 16, {v(dst + piece + q)}")
                out.append(f"v_and_b32 {t(2 * q + 1)}, {self.mask_hi()}, {v(dst + piece + q)}")
            for q in range(2):
                out.append(f"v_sub_f32 {x(2 * q)}, {x(2 * q)}, {t(2 * q)}")
                out.append(f"v_sub_f32 {x(2 * q + 1)}, {x(2 * q + 1)}, {t(2 * q + 1)}")
            for q in range(2):
                out.append(f"v_cvt_pk_bf16_f32 {v(dst + nxt + q)}, {x(2 * q)}, {x(2 * q + 1)}")
        if kind == "B":
            for q in range(2):
                out.append(f"v_mov_b32 {v(dst + 4 + q)}, {v(dst + q)}")
        return out

    def u_raw(self, e, kg):
        return [self.V["U"] + kg * 8 + (j >> 1) * 4 + e * 2 + (j & 1) for j in range(4)]

    def v_raw(self, e, cg):
        return [self.V["VR"] + (e * 2 + cg) * 4 + j for j in range(4)]

    def acc(self, e, kg, cg, i=0, n=1):
        return a(((e * 2 + kg) * 2 + cg) * 16 + i, n)

    def mfma(self, e, kg, cg, prod, fresh):
        """Product `prod` of the three; smallest terms first."""
        A, B = self.V[f"A{kg}"], self.V[f"B{cg}"]
        ar, br = ((A, B + 4), (A + 2, B + 2), (A + 2, B))[prod]
        c = "0" if fresh and prod == 0 else self.acc(e, kg, cg, 0, 16)
        return f"v_mfma_f32_32x32x16_bf16 {self.acc(e, kg, cg, 0, 16)}, {v(ar, 4)}, {v(br, 4)}, {c}"

    def transform_items(self, src, exact):
        """V = B^T d B of the patch in src (columns first, as Kernel.transform; the rows in place, v0 the
        one register more), and its way into the write buffer: two positions an instruction.  Unless exact,
        V comes out scaled, with the roundings of a transform that is not (a power of two): of every pair of terms
        one is scaled and the other meets the factor in an fma.  Rows 0 .. 2 are scaled in the column pass (one
        term serves all three), row 3 in the row pass (two terms serve its four): six multiplications a patch."""
        d = lambda i: self.vr(src, i)
        t = lambda i: self.vr("T", i)
        scale = self.sr("Scale")
        scaled = lambda x: f"v_mul_f32 {x}, {scale}, {x}"
        column, row = [], []
        for c in range(4):
            if exact:
                column += [f"v_sub_f32 {t(c)}, {d(c)}, {d(8 + c)}", f"v_add_f32 {t(4 + c)}, {d(4 + c)}, {d(8 + c)}",
                           f"v_sub_f32 {t(8 + c)}, {d(8 + c)}, {d(4 + c)}"]
            else:
                column += [scaled(d(8 + c)), f"v_fma_f32 {t(c)}, {d(c)}, {scale}, -{d(8 + c)}",
                           f"v_fma_f32 {t(4 + c)}, {d(4 + c)}, {scale}, {d(8 + c)}",
                           f"v_fma_f32 {t(8 + c)}, -{d(4 + c)}, {scale}, {d(8 + c)}"]
            column.append(f"v_sub_f32 {t(12 + c)}, {d(4 + c)}, {d(12 + c)}")
        for r in range(4):
            m = [t(4 * r + c) for c in range(4)]
            put = lambda p, x, y: ("lds", "write", f"ds_write2st64_b32 {self.vr('LdsWr')}, {x}, {y} offset0:{8 * p} offset1:{8 * p + 8}")
            if exact or r < 3:
                outer = [f"v_sub_f32 {m[0]}, {m[0]}, {m[2]}", f"v_sub_f32 {m[3]}, {m[1]}, {m[3]}"]
            else:
                row += [scaled(m[1]), scaled(m[2])]
                outer = [f"v_fma_f32 {m[0]}, {m[0]}, {scale}, -{m[2]}", f"v_fma_f32 {m[3]}, -{m[3]}, {scale}, {m[1]}"]
            row += [f"v_add_f32 v0, {m[1]}, {m[2]}", *outer, put(4 * r, m[0], "v0"),
                    f"v_sub_f32 {m[2]}, {m[2]}, {m[1]}", put(4 * r + 2, m[2], m[3])]
        return column, row

    def swap_buffers(self):
        self.e("s_waitcnt lgkmcnt(0)")
        self.e("s_barrier")
        for r in ("Lds0", "Lds1", "LdsWr"):
            self.e(f"v_xor_b32 {self.vr(r)}, 0x{BUFFER_SWAP:x}, {self.vr(r)}")
        self.e(f"s_xor_b32 {self.sr('Buf')}, {self.sr('Buf')}, 0x{BUFFER_SWAP:x}")

    # ------------------------------------------------------------------ one chunk
    # (filter group, column group) of the MFMAs, three each, for the wave's first and second position.  The
    # orders leave A0 and B0 early in the first half, A1 early in the second, so that the filter
    # registers are free, and loaded again, half a unit before their next split.
    ORDER = [[(0, 0), (0, 1), (1, 0), (1, 1)], [(0, 0), (1, 0), (0, 1), (1, 1)]]
    # What rides behind MFMA i, as (first slot, last slot + 1) per piece of work.  A split ends in front of
    # the first MFMA that reads it (3, 6, 12, 12, 15, 18; A0 and B0 of the next unit: the next chunk) and
    # starts behind the last one that reads the registers it overwrites.
    SLOTS = {"cursors": (0, 2), "column": (2, 6), "patch": (3, 11), "row": (6, 12),
             "B1": (0, 3), "A1": (3, 6), "A0'": (6, 9), "U0": (9, 10), "B0'": (9, 12), "A1'": (12, 15), "U1": (15, 16),
             "B1'": (15, 18), "swap": (14, 15), "read": (15, 16), "read'": (18, 19), "B0": (18, 21), "A0": (21, 24),
             "exchange": (17, 24)}

    def captured(self, *emitters):
        main, self.lines = self.lines, []
        for emit in emitters:
            emit()
        lines, self.lines = self.lines, main
        return lines

    def read_items(self):
        return [("lds", f"V{e}{cg}", f"ds_read2st64_b32 {v(self.v_raw(e, cg)[j], 2)}, {self.vr(f'Lds{cg}')} "
                 f"offset0:{e * 8 + 2 * j} offset1:{e * 8 + 2 * j + 2}") for e in range(2) for cg in range(2) for j in (0, 2)]

    def v_ready(self, cg):
        """Behind the reads of V: the values of column group cg are in their registers."""
        return [("lwait", f"V0{cg}"), ("lwait", f"V1{cg}")]

    def all_v_ready(self):
        return [("lwait", "V11")]

    def emit_chunk(self, seq, first):
        """Emits a chunk's items.  ("vm", tag, text) is a global load and ("wait", tag) the wait for the last
        load of that tag, issued in this chunk or in the chunk before it (the same sequence of loads); loads
        return in order, so the wait leaves as many in flight as were issued behind it.  In a first
        chunk the stores of an output transform lie between the two chunks.  ("lds", tag, text) and
        ("lwait", tag): the same for LDS; the reads of a chunk's V are the last LDS instructions of the chunk
        before it, or the first of its own."""
        loads = [x[1] for x in seq if x[0] == "vm"]
        reads = [] if first else [x[1] for x in self.read_items()]
        for item in seq:
            if item[0] == "vm":
                loads.append(item[1])
                self.e(item[2])
            elif item[0] == "lds":
                reads.append(item[1])
                self.e(item[2])
            elif item[0] == "wait":
                half = sum(1 for x in seq if x[0] == "vm")
                last = max(k for k, tag in enumerate(loads) if tag == item[1])
                n = len(loads) - 1 - last + (STORES if first and last < half else 0)
                self.e(f"s_waitcnt vmcnt({min(63, n)})")
            elif item[0] == "lwait":
                last = max(k for k, tag in enumerate(reads) if tag == item[1])
                self.e(f"s_waitcnt lgkmcnt({min(15, len(reads) - 1 - last)})")
            elif item.startswith((".L", "\t")):
                self.lines.append(item)
            else:
                self.e(item)

    def chunk(self, first, last):
        """Unit G: its MFMAs, the transform of unit G + 1's patch, the loads of unit G + 1's filters and of
        unit G + 2's patch, and, once every wave has written its share of V (the barrier in the chunk's second
        half), the reads of unit G + 1's V and its first two splits, so that the next chunk starts with
        MFMAs.  first: the first chunk of a segment, which does these two splits itself; last: the last
        one, which leaves them to it (the output transform needs the registers)."""
        self.comment(f"---- chunk{', first of a segment' if first else ''}{', last of a segment' if last else ''}")
        fill = [[] for _ in range(24)]

        def put(what, items):
            lo, hi = self.SLOTS[what]
            for k, item in enumerate(items):
                fill[lo + k * (hi - lo) // len(items)].append(item)
        split = self.split_operand
        a0 = lambda e: [("wait", "U0")] * (e == 0) + split(self.u_raw(e, 0), "A", self.V["A0"])
        b0 = lambda e: [("lwait", f"V{e}0")] + split(self.v_raw(e, 0), "B", self.V["B0"])
        b1 = lambda e: [("lwait", f"V{e}1")] + split(self.v_raw(e, 1), "B", self.V["B1"])
        column, row = self.transform_items("P", False)
        put("cursors", self.captured(self.advance_p, self.channel_descriptor, self.advance_q, self.filter_offsets))
        put("B1", b1(0))
        put("column", [("wait", "P")] + column)
        put("patch", [("vm", "P", self.patch_load("P", 4 * r + c)) for c in range(4) for r in range(4)])
        put("A1", [("wait", "U1")] + split(self.u_raw(0, 1), "A", self.V["A1"]))
        put("A0'", a0(1))
        put("U0", self.u_load_items(0))
        put("row", row)
        put("B0'", b0(1))
        put("B1'", b1(1))
        put("swap", self.captured(self.swap_buffers))
        put("A1'", split(self.u_raw(1, 1), "A", self.V["A1"]))
        put("U1", self.u_load_items(1))
        if not last:
            put("read", self.read_items()[:4])
            put("read'", self.read_items()[4:])
            put("A0", a0(0))
            put("B0", b0(0))
        else:
            # the accumulators of the wave's first position are final: their way to the other waves begins
            put("exchange", self.captured(self.exchange_address, lambda: self.exchange_write(0, 0)))
        seq = []
        if first:
            seq = self.read_items() + a0(0) + b0(0)
        i = 0
        for e in range(2):
            for kg, cg in self.ORDER[e]:
                for prod in range(3):
                    if i in (0, 3, 6, 12, 15, 18):
                        seq.append("s_nop 1")  # two wait states between a split and the MFMA that reads it
                    seq.append(self.mfma(e, kg, cg, prod, first))
                    seq += fill[i]
                    i += 1
        self.emit_chunk(seq, first)
        self.e(f"s_add_u32 {self.sr('G')}, {self.sr('G')}, 1")
        self.e(f"s_add_u32 {self.sr('Cm')}, {self.sr('Cm')}, 1")

    def exact_chunk(self, first):
        """Unit G on the fp32 MFMA, one piece of work after the other."""
        self.comment(f"---- exact chunk{', first of a segment' if first else ''}")
        column, row = self.transform_items("P", True)
        seq = self.read_items() + [("wait", "U1")] + self.all_v_ready()
        seq += self.captured(self.advance_p, self.channel_descriptor, self.advance_q, self.filter_offsets)
        for e in range(2):
            for kg in range(2):
                for cg in range(2):
                    for j in range(4):
                        c = "0" if first and j == 0 else self.acc(e, kg, cg, 0, 16)
                        seq.append(f"v_mfma_f32_32x32x2_f32 {self.acc(e, kg, cg, 0, 16)}, {v(self.u_raw(e, kg)[j])}, "
                                   f"{v(self.v_raw(e, cg)[j])}, {c}")
        seq += self.u_load_items(0) + self.u_load_items(1) + [("wait", "P")] + column + row
        seq += self.patch_items("P") + self.captured(self.swap_buffers)
        # (the loads come in another order than in the split chunks, the tags in the same)
        self.emit_chunk(seq, first)
        self.e(f"s_add_u32 {self.sr('G')}, {self.sr('G')}, 1")
        self.e(f"s_add_u32 {self.sr('Cm')}, {self.sr('Cm')}, 1")

    # ------------------------------------------------------------------ output transform
    def flag_address(self, previous):
        """Fl = &flags[((L - previous) * 8 + wave) * 2 + 1]."""
        t, fl = self.t, self.S["Fl"]
        self.e(f"s_sub_u32 {t(0)}, {self.sr('L')}, {1 if previous else 0}")
        self.e(f"s_lshl_b32 {t(0)}, {t(0)}, 3")
        self.e(f"s_add_u32 {t(0)}, {t(0)}, {self.sr('Wave')}")
        self.e(f"s_lshl_b32 {t(0)}, {t(0)}, 3")
        self.e(f"s_add_u32 {t(0)}, {t(0)}, 4")
        self.e(f"s_add_u32 {s(fl)}, {s(self.S['Sync'])}, {t(0)}")
        self.e(f"s_addc_u32 {s(fl + 1)}, {s(self.S['Sync'] + 1)}, 0")

    def store_flag(self, value_reg):
        self.e(f"v_mov_b32 {self.vr('Zero')}, 0")
        if value_reg == self.vr("One"):
            self.e(f"v_mov_b32 {value_reg}, 1")
        super().store_flag(value_reg)

    def wait_flag(self):
        """As Kernel.wait_flag; the 1 that a wave stores to the status word when it gives up is written
        into its register there."""
        n = len(self.outofline)
        self.e(f"v_mov_b32 {self.vr('Zero')}, 0")
        super().wait_flag()
        at = next(i for i in range(n, len(self.outofline)) if "_giveup_" in self.outofline[i]) + 1
        self.outofline.insert(at, f"\tv_mov_b32 {self.vr('One')}, 1")

    def row_descriptor(self, kg, b):
        """RsrcY = the image of filter row Dkb * 64 + kg * 32 + 4 * wave + b."""
        t, ry = self.t, self.S["RsrcY"]
        if b == 0:
            self.e(f"s_lshl_b32 {t(0)}, {self.sr('DkbM')}, 6")
            self.e(f"s_lshl_b32 {t(1)}, {self.sr('Wave')}, 2")
            self.e(f"s_add_u32 {t(2)}, {t(0)}, {t(1)}")
            if kg:
                self.e(f"s_add_u32 {t(2)}, {t(2)}, {32 * kg}")
            self.e(f"s_mul_hi_u32 {t(1)}, {t(2)}, {self.sr('HWN4')}")
            self.e(f"s_mul_i32 {t(0)}, {t(2)}, {self.sr('HWN4')}")
            self.e(f"s_add_u32 {s(ry)}, {s(self.S['Y'])}, {t(0)}")
            self.e(f"s_addc_u32 {s(ry + 1)}, {s(self.S['Y'] + 1)}, {t(1)}")
        else:
            self.e(f"s_add_u32 {s(ry)}, {s(ry)}, {self.sr('HWN4')}")
            self.e(f"s_addc_u32 {s(ry + 1)}, {s(ry + 1)}, 0")
            if self.ragged:
                self.e(f"s_add_u32 {t(2)}, {t(2)}, 1")
        if self.ragged:
            self.e(f"s_cmp_lt_u32 {t(2)}, {self.sr('Kreal')}")
            self.e(f"s_cselect_b32 {s(ry + 2)}, 0x{OOB:x}, 0")

    def exchange_address(self):
        """Tmp[0]: where the wave's first position goes in the exchange region (the 128 KB next to the live V
        buffer), [pos][8 groups of 4 rows][64 columns][4 rows]: wave * 16 KB + lane half * 1 KB + n * 16."""
        t, e = self.t, self.e
        e(f"s_cmp_eq_u32 {self.sr('Buf')}, 0")
        e(f"s_cselect_b32 {t(0)}, 0x8000, 0")
        e(f"s_lshl_b32 {t(1)}, {self.sr('Wave')}, 14")
        e(f"s_add_u32 {t(1)}, {t(0)}, {t(1)}")
        e(f"v_and_b32 {self.vr('Tmp', 1)}, 0x200, {self.vr('Lane16')}")
        e(f"v_add_u32 {self.vr('Tmp')}, {self.vr('Tmp', 1)}, {self.vr('Lane16')}")
        e(f"v_add_u32 {self.vr('Tmp')}, {t(1)}, {self.vr('Tmp')}")

    def exchange_write(self, kg, ee):
        for cg in range(2):
            for aa in range(4):
                self.e(f"ds_write_b128 {self.vr('Tmp')}, {self.acc(ee, kg, cg, 4 * aa, 4)} offset:{ee * 8192 + aa * 2048 + cg * 512}")

    def exchange_read(self):
        """EX: the 16 positions of row group = wave, column = lane: [pos][row group][column], 16 bytes each."""
        t, e = self.t, self.e
        ex, er = self.V["EX"], self.vr("Tmp", 1)
        e(f"s_lshl_b32 {t(2)}, {self.sr('Wave')}, 10")
        e(f"s_cmp_eq_u32 {self.sr('Buf')}, 0")
        e(f"s_cselect_b32 {t(0)}, 0x8000, 0")
        e(f"s_add_u32 {t(0)}, {t(0)}, {t(2)}")
        e(f"v_add_u32 {er}, {t(0)}, {self.vr('Lane16')}")
        for pos in range(8):
            e(f"ds_read_b128 {v(ex + 4 * pos, 4)}, {er} offset:{pos * 8192}")
        e(f"v_add_u32 {er}, 0x10000, {er}")
        for pos in range(8, 16):
            e(f"ds_read_b128 {v(ex + 4 * pos, 4)}, {er} offset:{(pos - 8) * 8192}")

    def mask_hi(self):
        return self.sr("MaskHi")

    def unscale(self):
        """Operand that takes the scale off a final output."""
        return self.sr("Unscale")

    def epilogue(self, exact):
        """Output transform of the tile.  Round kg: every wave writes its two positions of filter group
        kg, [pos][8 groups of 4 rows][64 columns][4 rows]; wave w reads the 16 positions of row group w
        (lane = column), transforms four rows and stores 16 values.  Kind, bit 0: the segment started
        inside the tile, its outputs are published (past the caches, then the flag); bit 1: it ended
        inside it, the part that the workgroup behind this one published is added."""
        t, e = self.t, self.e
        ex = self.V["EX"]
        m = lambda pos, b: v(ex + 4 * pos + b)
        self.comment("---- output transform")
        # the last MFMAs must have written the accumulators before they are read
        e("s_nop 15")
        e("s_nop 15")
        if exact:
            self.exchange_address()
            self.exchange_write(0, 0)
        self.exchange_write(0, 1)
        self.store_offsets()
        e(f"v_mov_b32 {self.vr('Sum')}, 0")
        for kg in range(2):
            e("s_waitcnt lgkmcnt(0)")
            e("s_barrier")
            self.exchange_read()
            e("s_waitcnt lgkmcnt(0)")
            e("s_barrier")
            if kg == 0:
                self.exchange_write(1, 0)
                self.exchange_write(1, 1)
            for b in range(4):
                for j in range(4):
                    e(f"v_add_f32 {m(j, b)}, {m(j, b)}, {m(4 + j, b)}")
                    e(f"v_sub_f32 {m(4 + j, b)}, {m(4 + j, b)}, {m(8 + j, b)}")
                for j in range(4):
                    e(f"v_add_f32 {m(j, b)}, {m(j, b)}, {m(8 + j, b)}")
                    e(f"v_sub_f32 {m(4 + j, b)}, {m(4 + j, b)}, {m(12 + j, b)}")
                for r in (0, 4):
                    e(f"v_add_f32 {m(r, b)}, {m(r, b)}, {m(r + 1, b)}")
                    e(f"v_sub_f32 {m(r + 1, b)}, {m(r + 1, b)}, {m(r + 2, b)}")
                for r in (0, 4):
                    e(f"v_add_f32 {m(r, b)}, {m(r, b)}, {m(r + 2, b)}")
                    e(f"v_sub_f32 {m(r + 1, b)}, {m(r + 1, b)}, {m(r + 3, b)}")
            out = lambda q, b: m((0, 1, 4, 5)[q], b)
            if exact:
                for b in range(4):
                    self.row_descriptor(kg, b)
                    for q in range(4):
                        e(f"buffer_store_dword {out(q, b)}, {self.vr('Eff', q)}, {self.sr('RsrcY', 4)}, 0 offen{self.final_policy()}")
                continue
            plain, stored, merges = self.newlabel("store"), self.newlabel("stored"), self.newlabel("merges")
            e(f"s_bitcmp1_b32 {self.sr('Kind')}, 1")
            e(f"s_cbranch_scc1 {merges}")
            for b in range(4):
                for q in range(4):
                    e(f"v_add_f32 {self.vr('Sum')}, {self.vr('Sum')}, |{out(q, b)}|")
            self.store_rows(kg, out, plain, stored)
            main, self.lines = self.lines, []
            self.label(merges)
            if kg == 0:
                for b in range(4):
                    for q in range(4):
                        e(f"v_mov_b32 {self.vr('VOFF', 4 * b + q)}, {out(q, b)}")
                e(f"s_branch {stored}")
            else:
                self.merge(out, stored)
            self.outofline.extend(self.lines)
            self.lines = main
        if exact:
            return
        # a lane whose sum is not finite (or close to it): the workgroup computes the tiles that it stores again.
        # A part that is published carries its infinities and NaNs to the workgroup that stores the tile.
        bad, bad_done, flag, done = (self.newlabel(x) for x in ("bad", "baddone", "flag", "nosplit"))
        e(f"s_mov_b32 {t(0)}, 0x{SUM_LARGE:x}")
        e(f"v_cmp_ngt_f32 vcc, {t(0)}, {self.vr('Sum')}")
        e(f"s_cbranch_vccnz {bad}")
        self.label(bad_done)
        e(f"s_bitcmp1_b32 {self.sr('Kind')}, 0")
        e(f"s_cbranch_scc1 {flag}")
        self.label(done)
        main, self.lines = self.lines, []
        self.label(flag)
        e("s_waitcnt vmcnt(0)")  # every write-through store acknowledged, then the flag
        self.flag_address(True)
        self.store_flag(self.vr("One"))
        e(f"s_branch {done}")
        self.label(bad)
        e(f"s_bitcmp1_b32 {self.sr('Kind')}, 0")
        e(f"s_cbranch_scc1 {bad_done}")
        e(f"s_mov_b32 {self.sr('Bad')}, 1")
        e(f"s_branch {bad_done}")
        self.outofline.extend(self.lines)
        self.lines = main

    def store_rows(self, kg, out, plain, stored):
        """The 16 outputs of filter group kg: published past the caches as they are (Kind bit 0), or final ones.
        (Those are unscaled in front of the stores: with every multiplication next to its store a tile took 0.5 ... 1 us
        longer, N=4 C=48 59x59 K=253 15.9 -> 16.9 us.)"""
        for final in (False, True):
            policy = self.final_policy() if final else " sc0 sc1"
            if final:
                self.label(plain)
                for b in range(4):
                    for q in range(4):
                        self.e(f"v_mul_f32 {out(q, b)}, {self.unscale()}, {out(q, b)}")
            else:
                self.e(f"s_bitcmp1_b32 {self.sr('Kind')}, 0")
                self.e(f"s_cbranch_scc0 {plain}")
            for b in range(4):
                self.row_descriptor(kg, b)
                for q in range(4):
                    self.e(f"buffer_store_dword {out(q, b)}, {self.vr('Eff', q)}, {self.sr('RsrcY', 4)}, 0 offen{policy}")
            if not final:
                self.e(f"s_branch {stored}")
        self.label(stored)

    def merge(self, out1, done):
        """A range that ends inside a tile: its last segment.  Both filter groups' outputs are there (those of
        group 0 in VOFF, which nothing reads any more) before the wait for the flag, so that between the flag
        of the workgroup behind and this one's there is one trip to memory and its acknowledgement: the
        partial tile lands in P and U, once their last prefetches have.  (With the two groups merged one after
        the other, a trip each, a hand-over took 1.7 us longer.)"""
        e = self.e
        out0 = lambda q, b: self.vr("VOFF", 4 * b + q)
        land = lambda kg, q, b: self.vr("P" if kg == 0 else "U", 4 * b + q)
        e("s_waitcnt vmcnt(0)")
        self.wait_flag()
        for kg in range(2):
            for b in range(4):
                self.row_descriptor(kg, b)
                for q in range(4):
                    e(f"buffer_load_dword {land(kg, q, b)}, {self.vr('Eff', q)}, {self.sr('RsrcY', 4)}, 0 offen sc0 sc1")
        for kg, out in ((0, out0), (1, out1)):
            e("s_waitcnt vmcnt(16)")  # the group's loads (behind them: the other group's, or 16 stores)
            for b in range(4):
                for q in range(4):
                    e(f"v_add_f32 {out(q, b)}, {out(q, b)}, {land(kg, q, b)}")
                    e(f"v_add_f32 {self.vr('Sum')}, {self.vr('Sum')}, |{out(q, b)}|")
            if kg == 1:
                self.store_flag(self.vr("Zero"))  # hand the flag back for the next launch
            self.store_rows(kg, out, self.newlabel("store"), self.newlabel("stored"))
        e(f"s_branch {done}")

    def stamp(self):
        """Timeline, as Kernel.stamp; the stamp count lives in a register of its own, and the temporaries in
        the registers that hold nothing between two segments."""
        begin, tmp, zero = self.S["Begin"], self.V["Tmp"], self.V["Zero"]
        self.S["Begin"], self.V["Tmp"], self.V["Zero"] = self.S["Stamps"], self.V["EX"], self.V["EX"] + 2
        n = len(self.lines)
        super().stamp()
        at = next(i for i in range(n, len(self.lines)) if "s_memrealtime" in self.lines[i])
        self.lines.insert(at, f"\tv_mov_b32 {self.vr('Zero')}, 0")
        self.S["Begin"], self.V["Tmp"], self.V["Zero"] = begin, tmp, zero

    # ------------------------------------------------------------------ whole kernel
    def body(self):
        e, t = self.e, self.t
        self.head()
        self.stamp()
        self.start()
        self.lds_addresses()
        self.prologue(False)
        self.stamp()
        self.segments(False)
        end = self.newlabel("end")
        # does any wave ask for the exact pass?  (the barrier: no wave still reads LDS)
        e("s_barrier")
        e(f"v_mov_b32 {self.vr('Tmp', 0)}, {self.sr('Bad')}")
        e(f"s_lshl_b32 {t(0)}, {self.sr('Wave')}, 2")
        e(f"v_mov_b32 {self.vr('Tmp', 1)}, {t(0)}")
        e(f"ds_write_b32 {self.vr('Tmp', 1)}, {self.vr('Tmp', 0)}")
        e("s_waitcnt lgkmcnt(0)")
        e("s_barrier")
        ex = self.V["EX"]
        e(f"v_mov_b32 {self.vr('Zero')}, 0")
        for i in range(2):
            e(f"ds_read_b128 {v(ex + 4 * i, 4)}, {self.vr('Zero')} offset:{16 * i}")
        e("s_waitcnt lgkmcnt(0)")
        for i in range(1, 8):
            e(f"v_or_b32 {v(ex)}, {v(ex)}, {v(ex + i)}")
        e(f"v_readfirstlane_b32 {self.sr('Bad')}, {v(ex)}")
        e("s_nop 4")
        e(f"s_cmp_eq_u32 {self.sr('Bad')}, 0")
        e(f"s_cbranch_scc1 {end}")
        # the tiles this workgroup stores are those whose first unit lies in its range
        e("s_waitcnt vmcnt(0)")
        e("s_barrier")  # everybody has read the words that the first transform overwrites
        for src, dst in ((self.sr("Begin"), t(0)), (t(3), t(1))):
            if dst == t(1):
                e(f"s_add_u32 {t(3)}, {self.sr('Begin')}, {self.sr('Nunits')}")
            e(f"s_add_u32 {t(2)}, {src}, {self.sr('Chunks')}")
            e(f"s_sub_u32 {t(2)}, {t(2)}, 1")
            # / Chunks by repeated use of the magic number: on the weighted line it divides by another number
            self.ceil_tiles(dst, t(2))
        e(f"s_sub_u32 {t(4)}, {t(1)}, {t(0)}")
        e(f"s_cmp_eq_u32 {t(4)}, 0")
        e(f"s_cbranch_scc1 {end}")
        e(f"s_mul_i32 {self.sr('Nunits')}, {t(4)}, {self.sr('Chunks')}")
        e(f"s_mov_b32 {self.sr('Tm')}, {t(0)}")
        e(f"s_mov_b32 {self.sr('Cm')}, 0")
        self.start()
        self.lds_addresses()
        self.prologue(True)
        self.segments(True)
        self.label(end)
        e("s_endpgm")
        self.lines.extend(self.outofline)

    def ceil_tiles(self, dst, x):
        """dst = x / Chunks by restoring division (31 steps): rare, and the magic number of the chunks may
        belong to the weighted line.  Uses T4..T7."""
        e, t = self.e, self.t
        loop, skip = self.newlabel("div"), self.newlabel("divskip")
        e(f"s_mov_b32 {t(4)}, 31")
        e(f"s_mov_b32 {t(5)}, 0")
        e(f"s_mov_b32 {dst}, 0")
        self.label(loop)
        e(f"s_sub_u32 {t(4)}, {t(4)}, 1")
        e(f"s_lshr_b32 {t(6)}, {x}, {t(4)}")
        e(f"s_and_b32 {t(6)}, {t(6)}, 1")
        e(f"s_lshl_b32 {t(5)}, {t(5)}, 1")
        e(f"s_or_b32 {t(5)}, {t(5)}, {t(6)}")
        e(f"s_lshl_b32 {dst}, {dst}, 1")
        e(f"s_cmp_lt_u32 {t(5)}, {self.sr('Chunks')}")
        e(f"s_cbranch_scc1 {skip}")
        e(f"s_sub_u32 {t(5)}, {t(5)}, {self.sr('Chunks')}")
        e(f"s_or_b32 {dst}, {dst}, 1")
        self.label(skip)
        e(f"s_cmp_lg_u32 {t(4)}, 0")
        e(f"s_cbranch_scc1 {loop}")

    def start(self):
        """Cursors at the first unit (Tm, Cm)."""
        e = self.e
        for n in ("Tp", "Tq"):
            e(f"s_mov_b32 {self.sr(n)}, {self.sr('Tm')}")
        for n in ("Cp", "Cq"):
            e(f"s_mov_b32 {self.sr(n)}, {self.sr('Cm')}")

    def head(self):
        S, t, e = self.S, self.t, self.e
        e(f"s_load_dwordx8 {s(8, 8)}, s[0:1], 0x0")
        e(f"s_load_dwordx16 {s(16, 16)}, s[0:1], 0x20")
        e(f"s_load_dwordx8 {s(32, 8)}, s[0:1], 0x60")
        e(f"s_load_dwordx2 {s(40, 2)}, s[0:1], 0x80")
        e(f"s_load_dwordx2 {s(S['Status'], 2)}, s[0:1], 0x88")
        e(f"s_load_dword {self.sr('SpinLimit')}, s[0:1], 0x90")
        e(f"v_and_b32 {self.vr('Tmp', 1)}, 0x3ff, v0")
        e(f"v_lshrrev_b32 {self.vr('Tmp')}, 6, {self.vr('Tmp', 1)}")
        e(f"v_and_b32 {self.vr('Lane16')}, 63, {self.vr('Tmp', 1)}")
        e(f"v_lshlrev_b32 {self.vr('Lane16')}, 4, {self.vr('Lane16')}")
        e("s_waitcnt lgkmcnt(0)")
        # only now: a vector instruction that writes an SGPR while scalar loads are still
        # outstanding came back with a corrupted value on this part
        e(f"v_readfirstlane_b32 {self.sr('Wave')}, {self.vr('Tmp')}")
        e("s_nop 4")
        e(f"s_and_b32 {t(0)}, s2, 7")
        e(f"s_mul_i32 {t(0)}, {t(0)}, {self.sr('GridPerXcd')}")
        e(f"s_lshr_b32 {t(1)}, s2, 3")
        e(f"s_add_u32 {t(0)}, {t(0)}, {t(1)}")
        e(f"s_cmp_eq_u32 {self.sr('GridPerXcd')}, 0")
        e(f"s_cselect_b32 {self.sr('L')}, s2, {t(0)}")
        self.unit_range(self.sr("L"))
        e(f"s_load_dword {self.sr('PlaceM')}, s[0:1], 0x94")
        e(f"s_load_dword {self.sr('PlaceS')}, s[0:1], 0x98")
        e(f"s_load_dword {self.sr('PlaceG')}, s[0:1], 0x9c")
        e(f"s_load_dword {self.sr('PlaceTn')}, s[0:1], 0xa0")
        e("s_waitcnt lgkmcnt(0)")
        e(f"s_lshl_b32 {self.sr('ColStep')}, {self.sr('N')}, 2")
        e(f"s_mul_i32 {self.sr('RowStep')}, {self.sr('ColStep')}, {self.sr('W')}")
        self.constants()
        e(f"s_mov_b32 {self.sr('Stamps')}, 0")
        e(f"s_mov_b32 {self.sr('Bad')}, 0")
        e(f"s_mov_b32 {s(S['RsrcX'] + 2)}, {self.sr('HWN4')}")
        e(f"s_mov_b32 {s(S['RsrcX'] + 3)}, 0x{FLAGS:x}")
        e(f"s_mov_b32 {s(S['RsrcU'])}, {s(S['U'])}")
        e(f"s_mov_b32 {s(S['RsrcU'] + 1)}, {s(S['U'] + 1)}")
        e(f"s_mov_b32 {s(S['RsrcU'] + 2)}, {self.sr('UswBytes')}")
        e(f"s_mov_b32 {s(S['RsrcU'] + 3)}, 0x{FLAGS:x}")
        e(f"s_mov_b32 {s(S['RsrcY'] + 2)}, 0x{OOB:x}")
        e(f"s_mov_b32 {s(S['RsrcY'] + 3)}, 0x{FLAGS:x}")

    def constants(self):
        self.e(f"s_mov_b32 {self.sr('MaskHi')}, 0xffff0000")
        self.e(f"s_mov_b32 {self.sr('Scale')}, 0x{SCALE:x}")
        self.e(f"s_mov_b32 {self.sr('Unscale')}, 0x{UNSCALE:x}")

    def lds_addresses(self):
        """V[pos][channel][column]: element at pos * 2048 + channel * 256 + (column ^ 32 * (channel & 1)) * 4.
        Lds0 / Lds1: the wave's first position, channel = lane half, column group 0 / 1, in the read
        buffer; LdsWr: channel = wave, column = lane, in the write buffer.  The prologue writes
        buffer 0, which the swap in end_of_chunk then makes the read buffer."""
        t, e = self.t, self.e
        tmp = lambda i: self.vr("Tmp", i)
        e(f"s_mov_b32 {self.sr('Buf')}, 0x{BUFFER_SWAP:x}")
        e(f"v_lshrrev_b32 {tmp(0)}, 2, {self.vr('Lane16')}")
        e(f"v_and_b32 {tmp(0)}, 0x7c, {tmp(0)}")                        # n * 4
        e(f"v_lshrrev_b32 {tmp(1)}, 9, {self.vr('Lane16')}")            # lane half
        e(f"s_lshl_b32 {t(0)}, {self.sr('Wave')}, 12")
        e(f"s_add_u32 {t(0)}, {t(0)}, 0x{BUFFER_SWAP:x}")
        e(f"v_mul_u32_u24 {self.vr('Lds0')}, 0x180, {tmp(1)}")          # 256 + the swapped half
        e(f"v_add3_u32 {self.vr('Lds0')}, {self.vr('Lds0')}, {tmp(0)}, {t(0)}")
        e(f"v_xor_b32 {self.vr('Lds1')}, 0x80, {self.vr('Lds0')}")
        e(f"s_and_b32 {t(1)}, {self.sr('Wave')}, 1")
        e(f"s_lshl_b32 {t(1)}, {t(1)}, 7")
        e(f"s_lshl_b32 {t(0)}, {self.sr('Wave')}, 8")
        e(f"v_lshrrev_b32 {self.vr('LdsWr')}, 2, {self.vr('Lane16')}")
        e(f"v_xor_b32 {self.vr('LdsWr')}, {t(1)}, {self.vr('LdsWr')}")
        e(f"v_add_u32 {self.vr('LdsWr')}, {t(0)}, {self.vr('LdsWr')}")

    def prologue(self, exact):
        """Unit 0 into V buffer 0, its filters into U, the patch of unit 1 into P; unit 0's patch lands in
        VR, so that all loads leave together."""
        e = self.e
        self.p_tile()
        self.filter_offsets()
        self.channel_descriptor()
        first = self.patch_items("VR")
        for item in first:
            e(item[2])
        loads = self.u_load_items(0) + self.u_load_items(1)
        for item in loads:
            e(item if isinstance(item, str) else item[2])
        e(f"s_mov_b32 {self.sr('G')}, -1")
        self.advance_p()  # G + 2 = 1: on to unit 1 when there is one
        self.channel_descriptor()
        for item in self.patch_items("P"):
            e(item[2])
        e(f"s_mov_b32 {self.sr('G')}, 0")
        self.behind_first_loads(exact)
        e(f"s_waitcnt vmcnt({4 + len(first)})")
        self.first_transform(exact)
        e("s_waitcnt vmcnt(0)")  # the first chunk counts on a queue without surprises
        self.swap_buffers()

    def behind_first_loads(self, exact):
        pass

    def first_transform(self, exact):
        column, row = self.transform_items("VR", exact)
        for item in column + row:
            self.e(item if isinstance(item, str) else item[2])

    def units(self, epi):
        """The chunks of a segment, the last one of which is SegEnd - 1, then on to the label epi."""
        e = self.e
        only, final, regular = self.newlabel("only"), self.newlabel("final"), self.newlabel("regular")
        e(f"s_cmp_lt_u32 {self.sr('Cm')}, {self.sr('SegEnd')}")
        e(f"s_cbranch_scc0 {only}")
        self.chunk(True, False)
        e(f"s_cmp_lt_u32 {self.sr('Cm')}, {self.sr('SegEnd')}")
        e(f"s_cbranch_scc0 {final}")
        self.label(regular)
        self.chunk(False, False)
        e(f"s_cmp_lt_u32 {self.sr('Cm')}, {self.sr('SegEnd')}")
        e(f"s_cbranch_scc1 {regular}")
        self.label(final)
        self.chunk(False, True)
        e(f"s_branch {epi}")
        self.label(only)
        self.chunk(True, True)

    def segments(self, exact):
        t, e = self.t, self.e
        seg_loop, regular, epi, done = (self.newlabel(x) for x in ("seg", "regular", "epi", "done"))
        self.label(seg_loop)
        # P is in this tile, or (tiles of one chunk) in the next one
        e(f"s_cmp_eq_u32 {self.sr('Tm')}, {self.sr('Tp')}")
        e(f"s_cselect_b32 {self.sr('DkbM')}, {self.sr('Dkb')}, {self.sr('DkbPrev')}")
        e(f"s_cselect_b64 vcc, -1, 0")
        e(f"v_cndmask_b32 {self.vr('Eff')}, {self.vr('EffPrev')}, {self.vr('EffP')}, vcc")
        # chunks Cm .. SegEnd-1 of tile Tm; Kind bit 0: starts inside the tile, bit 1: ends inside it
        e(f"s_sub_u32 {t(0)}, {self.sr('Nunits')}, {self.sr('G')}")
        e(f"s_sub_u32 {t(1)}, {self.sr('Chunks')}, {self.sr('Cm')}")
        e(f"s_min_u32 {t(0)}, {t(0)}, {t(1)}")
        e(f"s_add_u32 {self.sr('SegEnd')}, {self.sr('Cm')}, {t(0)}")
        e(f"s_cmp_lg_u32 {self.sr('Cm')}, 0")
        e(f"s_cselect_b32 {self.sr('Kind')}, 1, 0")
        e(f"s_cmp_lt_u32 {self.sr('SegEnd')}, {self.sr('Chunks')}")
        e(f"s_cselect_b32 {t(0)}, 2, 0")
        e(f"s_or_b32 {self.sr('Kind')}, {self.sr('Kind')}, {t(0)}")
        if exact:
            self.exact_chunk(True)
            e(f"s_cmp_lt_u32 {self.sr('Cm')}, {self.sr('SegEnd')}")
            e(f"s_cbranch_scc0 {epi}")
            self.label(regular)
            self.exact_chunk(False)
            e(f"s_cmp_lt_u32 {self.sr('Cm')}, {self.sr('SegEnd')}")
            e(f"s_cbranch_scc1 {regular}")
        else:
            e(f"s_sub_u32 {self.sr('SegEnd')}, {self.sr('SegEnd')}, 1")  # the last chunk of the segment
            self.units(epi)
        self.label(epi)
        self.stamp()
        self.epilogue(exact)
        self.stamp()
        e(f"s_add_u32 {self.sr('Tm')}, {self.sr('Tm')}, 1")
        e(f"s_mov_b32 {self.sr('Cm')}, 0")
        e(f"s_cmp_lt_u32 {self.sr('G')}, {self.sr('Nunits')}")
        e(f"s_cbranch_scc1 {seg_loop}")
        self.label(done)

    def emit(self, out):
        """The base class's kernel descriptor with this kernel's registers and LDS."""
        super().emit(out)
        out[-1] = (out[-1].replace("group_segment_fixed_size 0", f"group_segment_fixed_size {LDS_BYTES}")
                   .replace("next_free_vgpr 512", "next_free_vgpr 256").replace("accum_offset 256", "accum_offset 128"))

    def metadata(self):
        return (super().metadata().replace(".agpr_count:     256", ".agpr_count:     128")
                .replace(".group_segment_fixed_size: 0", f".group_segment_fixed_size: {LDS_BYTES}")
                .replace(".max_flat_workgroup_size: 256", ".max_flat_workgroup_size: 512")
                .replace(".vgpr_count:     512", ".vgpr_count:     256"))


def all_forms(kernel):
    """The kernels of a class: whole tiles, _ragged and _packed, for one filter block and for pairs; then the _cached ones."""
    forms = lambda: [kernel(kw, ragged, packed) for ragged, packed in ((False, False), (True, False), (True, True))
                     for kw in (2, 4)]
    return forms() + cached_forms(forms())


def write_kernels(kernels, stream):
    out = ['\t.amdgcn_target "amdgcn-amd-amdhsa--gfx950"', "\t.amdhsa_code_object_version 6"]
    for k in kernels:
        k.emit(out)
    out.append("\t.amdgpu_metadata\n---\namdhsa.kernels:")
    out.extend(k.metadata() for k in kernels)
    out.append("amdhsa.target:   amdgcn-amd-amdhsa--gfx950\namdhsa.version:\n  - 1\n  - 2\n...\n\t.end_amdgpu_metadata")
    stream.write("\n".join(out) + "\n")


if __name__ == "__main__":
    write_kernels(all_forms(KernelSplit), sys.stdout)
