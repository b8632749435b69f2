"""Dense "uvw" tensor products with shared weights in fp32 on the bf16 matrix cores (same problem and weight order as
:mod:`.uvw`; reference: the register-tiled CUDA-core matmul of openequivariance/templates/wmm.cuh:1-88).

Every fp32 operand of a contraction is split into three bf16 numbers, ``x = h + m + l``, each the rounding of what the ones
before it leave: together they hold all 24 bits of ``x``, denormal numbers included (``SCALE``), and of the nine products of
two such numbers the three below 2^-26 of the largest (m l, l m, l l) are left out.  The other six are v_mfma_f32_16x16x32_bf16 steps into one fp32
accumulator: 6 x 16 cycles per 16 x 16 x 32 block where v_mfma_f32_16x16x4_f32 takes 8 x 32, and a block of 32 channels
meets the accumulator with 6 roundings where the fp32 instruction has 8 to 32.

A split costs 5.5 vector instructions per number, so what is split is read often and split once: the contraction comes
*before* the Clebsch-Gordan part, on X (forward) or dZ (backward) as they lie in memory,

    U_t[b, w, i] = sum_u W_t[u, w] x[b, u, i],      Z[b, w, k]  += sum_i M_t[b, i, k] U_t[b, w, i]
    V_t[b, u, k] = sum_w W_t[u, w] dz[b, w, k],     dX[b, u, i] += sum_k M_t[b, i, k] V_t[b, u, k]

with M_t = sum_j C_ijk y_j.  A workgroup splits the rows of its 16-row tiles into LDS (6 bytes a number) and every wavefront
owns 16 output channels of a tile, for all paths: A = weights, split by the preparation kernel, [channel][K]; B = rows of X
or dZ from LDS, [K][row]; an accumulator holds four adjacent channels of one row, so that the Clebsch-Gordan part has its
row's M in registers and results leave as contiguous runs.  A row fragment read from LDS serves all paths of a chunk
(``_chunks``), a weight fragment all components of the row's records.

dW_t[u, w] = sum_bk T_t[b, u, k] dz[b, w, k] runs over the batch, in steps of 16 rows on v_mfma_f32_32x32x16_bf16: dZ of a tile
is split into LDS once per workgroup (two buffers), T is formed in the registers of the wavefront that multiplies it, from M
in LDS, split and used for all w, beside the matrix steps of the component before.

An infinity, a NaN or a number whose multiple overflows among the operands makes the residuals of its split NaN.  A wavefront
whose results are not all finite computes its part again with fp32 multiply-adds from the original operands, a dW wavefront the
groups of four channels concerned and until all of their sums are NaN.  64 channels, 100 000 rows, forward / backward in us: 180 /
550 without, one NaN in X 355 / 1550 (a row's whole batch share of dW cell by cell 8400), one in dZ 180 / 1480, dZ all NaN 180 /
3600, one infinite weight 2720 / 2010.

Measured, 64x0e+64x1o+64x2e with 1x0e+1x1o+1x2e, fp32 kernels / these: 100 000 rows forward 291 / 175 us, backward 575 / 440 us;
4097 rows 31 / 15 and 61 / 52; 100 channels, 50 000 rows 455 / 294 and 2048 / 690 (the fp32 dW walks the batch once per pass of
accumulators there).  Relative errors against fp64 (2-norm; Z, dX, dY, dW) at 100 000 rows: 2.9e-7 1.6e-7 2.0e-7 7.7e-7 / 1.1e-7
1.1e-7 1.6e-7 2.1e-7, and smaller than those of the kernels they replace on every problem of ``_pays``, 4097 and 50 000 rows, and on
64 to 512 channels with all operands of one sign (dY too, ``_apart``).

What bounds them: the matrix cores are busy for 47 % of the forward's time, 34 % of dX/dY's and 37 % of dW's (counters); the rest of
the first two is weight fragments through L1 (270 KB per tile: 70 us when every one hits it, as measured with all
loads at one address), and what a workgroup does before its first product - rows in, split, two barriers - beside one other
workgroup per compute unit (55 KB of LDS and 200 - 256 registers each).  Measured without gain: eight wavefronts per tile at
128 registers (206 / 201), two tiles a workgroup (241 / 233), three or four paths a chunk (216 / 217).
"""
from __future__ import annotations

import threading
from collections import OrderedDict
from dataclasses import dataclass
from functools import cached_property
from typing import List

import numpy as np

from ..problem import TPProblem
from .common import Emitter
from .uvw import UVWGenerator, WPath, _ceil

# Operands are split times 2^24, which is exact, and results taken back by 2^-48: the last bit of the smallest fp32 number,
# 2^-149, is then a normal bf16 number, and no part of a split falls below what bf16 (or a matrix step) holds.  Operands from 2^103
# on, and sums from 2^79, overflow on the way and are computed with fp32 multiply-adds like infinities and NaN.  (Without the
# factor: operands of 1e-36 lost 8 of their 24 bits, 2.7e-5 relative error of a result.)
SCALE, BACK = 2.0 ** 24, 2.0 ** -48
PRODUCTS = ((2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0))     # (split of A, split of B), smallest products first


@dataclass
class Shape:
    """How a workgroup's wavefronts share its 16-row tiles."""
    waves: int                   # of a tile, along its 16-wide tiles of output channels
    tiles: int                   # 16-row tiles of a workgroup
    units: int                   # LDS of a tile, split, in units of 16 bytes

    @property
    def threads(self) -> int:
        """At least four wavefronts, which all take part in moving the rows."""
        return 64 * max(4, self.waves * self.tiles)

    @property
    def helpers(self) -> bool:
        return self.threads > 64 * self.waves * self.tiles


class DWKind:
    """What one kind of workgroup of the dW kernel does: the output blocks (with ranges of 32-channel tiles) whose dZ it keeps
    in LDS, split, and the jobs of its wavefronts."""

    def __init__(self, g, blocks, bins=(), waves=()):
        self.g, self.blocks, self.bins, self.waves = g, list(blocks), list(bins), list(waves)
        self.offs, self.units = {}, 0
        for o, lo, hi in self.blocks:
            self.offs[o] = self.units
            self.units += 3 * g.out[o].D * 2 * 32 * (hi - lo)
        self.entries = {}        # (path, i, k) -> (entry of the M table, first y, coefficients)
        outs = {o for o, _, _ in self.blocks}
        mine = {sg[0].t for b, _ in [w for w in self.waves if w] for sg in self.bins[b]} if self.waves else None
        for p in g.paths:
            if p.o.idx not in outs or (mine is not None and p.t not in mine):
                continue
            terms = {}
            for (i, j), ks in p.pairs.items():
                for k, val in ks:
                    terms.setdefault((i, k), {})[j] = val
            for (i, k), c in sorted(terms.items()):
                self.entries[p.t, i, k] = (len(self.entries), p.b.off, [c.get(j, 0.0) for j in range(p.b.D)])
        self.width = max([len(c) for _, _, c in self.entries.values()] + [1])

    @staticmethod
    def cost(segs) -> int:
        return sum(p.o.D * (hi - lo) for p, lo, hi in segs)

    @property
    def lds_units(self) -> int:
        """LDS in units of 16 bytes: Y, split dZ and M of two tiles each, one behind the other."""
        return 2 * (4 * self.g.D2 + self.units + 4 * len(self.entries))

    def lds_bytes(self) -> int:
        return 16 * self.lds_units


class UVWSplitGenerator(UVWGenerator):
    LDS_BYTES = 160 * 1024
    ACC_BUDGET = 48              # accumulator registers of the paths of a chunk
    PATHS = 2                    # paths of a chunk at most
    AHEAD = 60                   # matrix steps between the request of a weight fragment and its use, where there are as many
    BESIDE = 2                   # statements of the Clebsch-Gordan part beside a matrix step
    KEEP_BUDGET = 72             # registers that outlive the chunks: Z of the output blocks, X and dX of the in1 blocks

    def __init__(self, problem: TPProblem):
        super().__init__(problem)
        if self.T != "float":
            raise NotImplementedError("the split kernels are for fp32")
        self.kind = "uvw"
        shape = lambda which, blocks, tiles: self._shape(which, blocks, max(tiles(p) for p in self.paths))
        self.fwd_shape = shape(self.used_in1, self.in1, lambda p: p.NTW)
        self.bwd_shape = shape(self.used_out, self.out, lambda p: p.NTU)
        # cycles of the fp32 instruction over those of the split one
        forward = sum(p.o.D * p.SU * p.NTW * 32 for p in self.paths) / sum(p.a.D * self.kblocks(p.mu) * p.NTW * 96 for p in self.paths)
        backward = sum(p.o.D * p.SW * p.NTU * 32 for p in self.paths) / sum(p.o.D * self.kblocks(p.mw) * p.NTU * 96 for p in self.paths)
        self.split_forward = self._pays(self.fwd_shape, forward, 1.5, 0, 7 if self._single(self.used_in1) else 5)
        self.split_dx = self._pays(self.bwd_shape, backward, 1.3, 64 * max(1, self.D2), 5)
        # packed copies, in words: forward, then backward
        self.FWD_WORDS = self._place("wb", 0, self.split_forward, lambda p: p.NTW * self.kblocks(p.mu) * 192, lambda p: p.SU * 64 * p.NTW)
        self.WA_END = self._place("wa", self.FWD_WORDS, self.split_dx, lambda p: p.NTU * self.kblocks(p.mw) * 192,
                                  lambda p: p.NTU * _ceil(p.SW, self.VW) * 64 * self.VW)
        least = self.ws_elems                                   # (what the kernels for few rows may use)
        self.PART_OFF = _ceil(self.WA_END, 64) * 64
        self.ws_elems = max(least, self.PART_OFF + self.DW_WORKGROUPS * self.WN)

    def _place(self, name: str, pos: int, split: bool, units, words) -> int:
        """Offsets of a direction's packed copies (in units of 16 bytes where split): returns the end in words."""
        pos = _ceil(pos, 4) * 4
        for p in self.paths:
            setattr(p, name, pos // 4 if split else pos)
            pos += 4 * units(p) if split else words(p)
        return pos

    # ------------------------------------------------------------------ shape
    @staticmethod
    def kblocks(mul: int) -> int:
        return _ceil(mul, 32)

    def _tile_units(self, blocks, which) -> int:
        """LDS of one 16-row tile of the blocks ``which``, split, in units of 16 bytes."""
        return sum(3 * blocks[b].D * 4 * self.kblocks(blocks[b].mul) * 16 for b in which)

    def _shape(self, which, blocks, channel_tiles: int) -> Shape:
        """A wavefront per 16 output channels, at most eight (beyond, they take several in turn); tiles of few wavefronts share
        a workgroup while four wavefronts and half the LDS allow."""
        waves, units = min(8, channel_tiles), self._tile_units(blocks, which)
        tiles = max(1, 4 // waves)
        while tiles > 1 and 16 * units * tiles > self.LDS_BYTES // 2:
            tiles //= 2
        return Shape(waves, tiles, units)

    def _lds_units(self, shape: Shape, *dims) -> int:
        """The split tiles, or rows of the widths ``dims`` as they lie in memory (these take turns)."""
        return max([shape.units * shape.tiles] + [_ceil(16 * shape.tiles * self._row_pitch(d), 4) + 16 for d in dims])

    @staticmethod
    def _row_pitch(d: int) -> int:
        """Words from one row to the next of outputs in LDS: a multiple of four that is 4 mod 64 banks, so that the 16 rows
        a wavefront writes at the same column fall on different banks."""
        return d + (4 - d) % 64

    def _single(self, blocks) -> bool:
        """Whether at most one path reads each block on average: its split rows serve one contraction only."""
        return len(self.paths) <= len(blocks)

    def _pays(self, shape: Shape, gain: float, least: float, extra: int, resident: int) -> bool:
        """Whether the split kernel of a direction is the faster one: its tiles fit LDS, three wavefronts or more of a workgroup
        have a tile of output channels, and the padding to 32 (K) leaves enough of the 2.67 times shorter matrix steps.
        40 000 rows, l <= 2 with second operand l <= 2, gain, fp32 / split kernel in us:

            channels        forward                dX, dY
            64           2.67  129.8 /  69.9    2.67  140.2 /  97.0
            100          2.33  389.2 / 239.9    2.08  375.2 / 282.0
            48           2.00   79.9 /  60.2    2.00   96.2 /  76.1
            32           2.67   46.5 /  29.1    2.67   66.3 /  41.4
            20 -> 72     2.67  116.5 /  80.0    2.00  115.8 / 261.6   (two wavefronts)
            16           1.33   18.8 /  21.3    1.33   38.5 /  28.7
            9 -> 95      1.33   91.0 /  91.7    2.67  227.4 / 257.2   (one wavefront)
            96 -> 9      2.67   83.1 / 245.0    1.00  185.8 / 120.1   (one wavefront forward)

        And as many wavefronts as ``resident`` in the workgroups that LDS lets a compute unit hold, for they wait for one another at
        both ends of a tile: five, of the forward seven where split rows serve one path each.  40 000 rows, wavefronts, whole
        forward and backward calls (the dX of both on the same dW), fp32 / split, us:

            64, l <= 3, in2 l <= 1            4   175 / 256    316 / 408
            50, l <= 3, in2 l <= 2            4   299 / 393    408 / 649
            50, both parities, l <= 2, 1x0e   4   108 / 175    248 / 325
            33, both parities, in2 l <= 2     3   219 / 476    494 / 840
            65, l <= 2, in2 l <= 2            5   244 / 178    472 / 462
            96, l <= 2, in2 l <= 1            6   236 / 136    375 / 341
            65, l <= 2, 1x0e                  5    81 /  99    221 / 224   (72, l <= 3, 1x0e: 193 / 166, 369 / 360)
            33 | 48, l <= 2, 1x0e (65 536)    6    45 /  54     50 /  56   (forward of each)
            100, l <= 2, 1x0e                 7   151 / 121    278 / 270
            64, l <= 2, 1x0e (65 536)         8   100 /  74
            150 | 200, l <= 1, in2 l <= 1     8   197 / 132, 423 / 218;  422 / 345, 590 / 485"""
        lds = 16 * self._lds_units(shape, self.D1, self.D3) + extra * shape.waves * shape.tiles
        waves = shape.waves * shape.tiles
        return waves >= 3 and gain >= least and self.LDS_BYTES // lds * waves >= resident

    @classmethod
    def create(cls, problem: TPProblem):
        """The generator, or None where the fp32 kernels serve every direction: also where no multiplicity exceeds 16 and half of
        every matrix step is padding (16 channels, l <= 2, 4097 rows: 26 / 29 us backward; 40 000 rows 108 / 76)."""
        if problem.irrep_dtype != np.float32 or not problem.shared_weights:
            return None
        g = cls(problem)
        if max(max(p.mu, p.mw) for p in g.paths) <= 16:
            return None
        return g if g.split_forward or g.split_dx or g.dw_kinds else None

    def few_rows(self, limits):
        """Largest batches of the kernels for few rows (``limits``: beside the fp32 kernels) that these leave them.

        Forward: every 16-row tile has a workgroup whose wavefronts share its output channels, so next to nothing.  Only rows that
        serve one path each and whose channels are no multiple of eight, which are split number by number: few rows / split, 500
        and 2048 rows, us: 50 channels of both parities, l <= 1, 8.6 / 9.9 and 9.6 / 10.2, 20 -> 64 l <= 2 7.3 / 8.9 and 8.6 / 9.3,
        100 12.1 / 14.0 and 15.8 / 14.8 (1000 rows 13.4 / 14.9); 64 9.0 / 8.7 and 10.3 / 9.1, 128 l <= 1 11.8 / 8.8.

        Backward: the dW workgroups are later to start, with a chain of 32 channels and more for each path.  us:

            channels                       500 rows      2048          4096          4097
            64, l <= 2                  29.5 / 32.0   37.7 / 42.2   51.3 / 49.2   60.5 / 54.3
            32, l <= 2                  20.2 / 22.5   23.8 / 25.9   29.4 / 33.8   35.6 / 34.0
            48, l <= 2                                            42.0 / 48.2   49.4 / 52.3
            25, l <= 1                  14.5 / 16.7   18.7 / 19.5   19.8 / 24.2   20.9 / 24.2
            64, both parities, l <= 1   23.4 / 25.6   28.0 / 35.8   34.3 / 41.0   40.8 / 43.0
            65, l <= 2                  45.2 / 40.0   63.5 / 54.7   84.0 / 67.8
            128, l <= 1                 31.0 / 25.4   37.8 / 36.7   46.8 / 39.3
            one path a block:
            64, l <= 1                  15.2 / 15.2   22.6 / 18.7   27.9 / 24.2   (1000 rows 18.1 / 18.0)
            64, l <= 2                  19.2 / 19.8   28.1 / 24.1   34.2 / 31.8   (22.4 / 22.9)
            50, both parities, l <= 1   17.4 / 20.5   23.6 / 25.0   26.7 / 32.5   (8192 rows 36.5 / 37.1, 20 480 64.0 / 60.9)

        Up to 16 channels half of a matrix step is padding: 17 / 22 at 1000 and 26 / 29 at 4097 rows."""
        forward, backward = limits
        widest = max(max(p.mu, p.mw) for p in self.paths)
        if self.split_forward:
            odd = self._single(self.used_in1) and any(self.in1[a].mul % 8 for a in self.used_in1)
            forward = min(forward, 0 if not odd else 2048 if widest <= 64 else 1024)
        if self.split_dx and self.dw_kinds and max(p.mw for p in self.paths) > 16:
            if max(p.mw for p in self.paths) > 64:
                most = 0
            elif self._single(self.used_out):
                most = 8192 if len(self.used_in1) >= 4 else 1024
            elif max(self.in1[a].D for a in self.used_in1) <= 3:
                most = 5120
            else:
                most = 4096 if widest < 64 else 2048
            backward = min(backward, most)
        return forward, backward

    def _chunks(self, paths: List[WPath], comps, tiles) -> List[List[WPath]]:
        """Paths that read the same rows (one in1 block forward, one output block backward), as many together as
        ACC_BUDGET allows, at most PATHS."""
        out: List[List[WPath]] = []
        for p in paths:
            if out and len(out[-1]) < self.PATHS and tiles(out[-1][0]) == tiles(p) and 4 * comps(p) * (len(out[-1]) + 1) <= self.ACC_BUDGET:
                out[-1].append(p)
            else:
                out.append([p])
        return out

    def _passes(self, blocks, which, per: int):
        """Blocks whose registers (``per`` per component) are held together."""
        passes = [[]]
        for b in which:
            if passes[-1] and per * (sum(blocks[q].D for q in passes[-1]) + blocks[b].D) > self.KEEP_BUDGET:
                passes.append([])
            passes[-1].append(b)
        return passes

    # ================================================================== prep
    def _pack(self, E: Emitter, backward: bool) -> None:
        E("const int q = blockIdx.x * 256 + threadIdx.x;")
        E("U4* __restrict__ wsp = (U4*)ws;")
        first = 0
        for p in self.paths:
            kb = self.kblocks(p.mw if backward else p.mu)
            units = (p.NTU if backward else p.NTW) * kb * 64
            base = p.wa if backward else p.wb
            row, k = ("u", "w") if backward else ("w", "u")
            E(f"if (q >= {first} && q < {first + units}) {{   // path {p.t}: [{row} tile][{k} block][split][lane]")
            E.level += 1
            E(f"const int e = q - {first}, ln = e & 63, kb = (e >> 6) % {kb}, {row} = 16 * (e / {64 * kb}) + (ln & 15), k0 = 32 * kb + 8 * (ln >> 4);")
            E("T v[8];")
            E(f"for (int j = 0; j < 8; ++j) {{ const int {k} = k0 + j; v[j] = (u < {p.mu} && w < {p.mw}) ? {self.lit(SCALE)} * W[{self.oeq_index(p, 'u', 'w')}] : (T)0; }}")
            E("U4 h, m, l;")
            E("oeq_split8(v, h, m, l);")
            E(f"U4* __restrict__ d = wsp + {base} + (e >> 6) * 192 + ln;")
            E("d[0] = h; d[64] = m; d[128] = l;")
            E.level -= 1
            E("}")
            first += units

    def prep_body(self) -> str:
        E = Emitter()
        if self.split_forward:
            self._pack(E, False)
        else:
            E("const int q = blockIdx.x * 256 + threadIdx.x;")
            E("T* __restrict__ wsT = (T*)ws;")
            for p in self.paths:
                self._pack_forward_copy(E, p)
        return E.text()

    def prep_backward_body(self) -> str:
        E = Emitter()
        if self.split_dx:
            self._pack(E, True)
        else:
            E(f"const int q = {self.FWD_WORDS // 256 * 256} + blockIdx.x * 256 + threadIdx.x;")
            E("T* __restrict__ wsT = (T*)ws;")
            for p in self.paths:
                self._pack_backward_copy(E, p)
        return E.text()

    @property
    def prep_blocks(self) -> int:
        return _ceil(self.FWD_WORDS // 12 if self.split_forward else self.FWD_WORDS, 256)

    @property
    def prep_backward_blocks(self) -> int:
        return _ceil((self.WA_END - self.FWD_WORDS) // 12, 256) if self.split_dx else _ceil(self.WA_END - self.FWD_WORDS // 256 * 256, 256)

    # ---------------------------------------------------------------- helpers
    def _prologue(self, E: Emitter, shape: Shape, *dims) -> None:
        waves, tiles, units = shape.waves, shape.tiles, shape.units
        E("const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;")
        E("const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));")
        E(f"const int sub = {f'wv / {waves}' if tiles > 1 else '0'}, wave = {f'wv % {waves}' if tiles > 1 else 'wv'};")
        E(f"const u64 base0 = (u64)blockIdx.x * {16 * tiles}, row0 = base0 + 16 * sub;")
        E("if (base0 >= n) return;")
        E("oeq_priority(3);")
        E("const u64 rowB = min(row0 + (u64)c, n - 1);")
        E("const bool bvalid = row0 + c < n;")
        E("const U4* __restrict__ wsp = (const U4*)ws;")
        E(f"__shared__ U4 xs[{self._lds_units(shape, *dims)}];")
        E("T* __restrict__ raw = (T*)xs;")
        # a row of the tile in LDS: component i of octet 4 kb + g of a block is 16 bytes at ((split * D + i) * octets + octet) * 16
        # + (c ^ 2 octet % 16).  Reads of a fragment and writes of a task (adjacent octets of a row) both meet every bank once
        E(f"const U4* __restrict__ xrow0 = xs + {f'sub * {units} + ' if tiles > 1 else ''}g * 16 + (c ^ (2 * g));")
        E(f"const U4* __restrict__ xrow1 = xs + {f'sub * {units} + ' if tiles > 1 else ''}g * 16 + (c ^ (2 * g) ^ 8);")

    MOVES = 12                   # 16-byte pieces of a row in flight per thread

    def _rows_in(self, E: Emitter, src: str, d: int, shape, tag: str):
        """Statements that bring the workgroup's rows of ``src`` (d words each, one run of memory) to ``raw``: lists of
        (requests, LDS writes), adjacent threads at adjacent 16 bytes; rows past the end are zeros."""
        NT, tiles = shape.threads, shape.tiles
        pieces = 4 * tiles * d
        E(f"const T* __restrict__ {tag}_ = {src} + base0 * {d} + 4 * threadIdx.x;")
        E(f"const bool {tag}all = base0 + {16 * tiles} <= n;")
        E(f"const i64 {tag}left = (i64)((n - base0) * {d}) - 4 * (int)threadIdx.x;")
        out = []
        for q0 in range(0, _ceil(pieces, NT), self.MOVES):
            turns = range(q0, min(_ceil(pieces, NT), q0 + self.MOVES))
            guard = {q: "" if NT * (q + 1) <= pieces else f"if ((int)threadIdx.x < {pieces - NT * q}) " for q in turns}
            req = ["VTU " + ", ".join(f"{tag}{q}" for q in turns) + ";", f"if ({tag}all) {{"]
            req += [f"    {guard[q]}{tag}{q} = *(const VTU*)({tag}_ + {4 * NT * q});" for q in turns]
            req += ["} else {"]
            req += [f"    {guard[q]}for (int e = 0; e < 4; ++e) {tag}{q}[e] = {4 * NT * q} + e < {tag}left ? {tag}_[{4 * NT * q} + e] : (T)0;" for q in turns]
            req += ["}"]
            out.append((req, [f"{guard[q]}*(VT*)(raw + 4 * ((int)threadIdx.x + {NT * q})) = {tag}{q};" for q in turns]))
        return out

    def _tasks(self, blocks, which, shape):
        """Splitting work: (block, turn, index expression, guard) with a task = eight adjacent channels of a row.  Blocks of fewer
        tasks than threads go to the wavefronts that have the least to do."""
        waves, tiles = shape.threads // 64, shape.tiles
        load = [0] * waves
        for b in sorted(which, key=lambda b: -blocks[b].D):
            left = 16 * tiles * 4 * self.kblocks(blocks[b].mul)
            q = 0
            while left > 0:
                width = min(waves, _ceil(left, 64))
                first = min(range(waves - width + 1), key=lambda w: max(load[w:w + width]))
                for w in range(first, first + width):
                    load[w] += blocks[b].D
                idx = f"((int)threadIdx.x + {64 * (-first)})" if first else "(int)threadIdx.x"
                done = 16 * tiles * 4 * self.kblocks(blocks[b].mul) - left
                conds = ([f"wv >= {first}"] if first else []) + ([f"wv < {first + width}"] if first + width < waves else [])
                if left < 64 * width:
                    conds.append(f"{idx} < {left}")
                yield b, q, f"({idx} + {done})" if done else f"({idx})", f"if ({' && '.join(conds)}) " if conds else ""
                left -= 64 * width
                q += 1

    def _split_rows(self, E: Emitter, d: int, blocks, which, shape) -> dict:
        """Rows of d words at ``raw`` -> split tiles at ``xs`` (the same memory: everything is read before anything is
        written).  Returns the blocks' offsets within a tile."""
        units = shape.units
        offs, pos = {}, 0
        for b in which:
            offs[b] = pos
            pos += 3 * blocks[b].D * 4 * self.kblocks(blocks[b].mul) * 16
        assert pos == units
        for b, q, idx, guard in self._tasks(blocks, which, shape):
            o, noct, tag = blocks[b], 4 * self.kblocks(blocks[b].mul), f"{b}_{q}"
            E(f"const int r{tag} = {idx} / {noct}, o{tag} = {idx} % {noct};")
            E(f"T v{tag}[{8 * o.D}];")
            E(f"{guard}{{ const T* __restrict__ s_ = raw + r{tag} * {d} + {o.off} + 8 * o{tag} * {o.D};")
            if o.mul % 8 == 0:
                E(f"    if (8 * o{tag} < {o.mul}) {{")
                wide = d % 4 == 0 and o.off % 4 == 0
                for i in range(2 * o.D):
                    if wide:
                        E(f"        {{ const VT t_ = *(const VT*)(s_ + {4 * i}); " + " ".join(f"v{tag}[{4 * i + e}] = t_[{e}];" for e in range(4)) + " }")
                    else:
                        E("        " + " ".join(f"v{tag}[{4 * i + e}] = s_[{4 * i + e}];" for e in range(4)))
                E("    } else { " + " ".join(f"v{tag}[{e}] = (T)0;" for e in range(8 * o.D)) + " }")
            else:
                for j in range(8):
                    E(f"    if (8 * o{tag} + {j} < {o.mul}) {{ " + " ".join(f"v{tag}[{j * o.D + i}] = s_[{j * o.D + i}];" for i in range(o.D))
                      + " } else { " + " ".join(f"v{tag}[{j * o.D + i}] = (T)0;" for i in range(o.D)) + " }")
            E("}")
        E("oeq_block_sync();")
        for b, q, idx, guard in self._tasks(blocks, which, shape):
            o, noct, tag = blocks[b], 4 * self.kblocks(blocks[b].mul), f"{b}_{q}"
            E(f"{guard}{{ U4* __restrict__ d = xs + (r{tag} >> 4) * {units} + {offs[b]} + o{tag} * 16 + ((r{tag} ^ (2 * o{tag})) & 15);")
            for i in range(o.D):
                E(f"    {{ const T e[8] = {{{', '.join(f'{self.lit(SCALE)} * v{tag}[{j * o.D + i}]' for j in range(8))}}}; U4 h, m, l;")
                E("      oeq_split8(e, h, m, l);")
                E("      " + " ".join(f"d[{(s * o.D + i) * noct * 16}] = {nm};" for s, nm in enumerate("hml")) + " }")
            E("}")
        E("oeq_block_sync();")
        E("oeq_priority(0);")
        return offs

    def _rows_out(self, E: Emitter, dst: str, d: int, blocks, used, shape: Shape) -> None:
        """The workgroup's finished rows from LDS (row pitch ``_row_pitch``) to memory, adjacent threads at adjacent 16 bytes."""
        NT, pitch = shape.threads, self._row_pitch(d)
        pieces = 4 * shape.tiles * d
        for o in blocks:
            if o.dim and o.idx not in used:
                E(f"for (int q = threadIdx.x; q < {16 * shape.tiles * o.dim}; q += {NT}) raw[(q / {o.dim}) * {pitch} + {o.off} + q % {o.dim}] = (T)0;")
        E("oeq_block_sync();")
        E("#pragma unroll")
        E(f"for (int q = 0; q < {_ceil(pieces, NT)}; ++q) {{")
        E(f"    const int idx = (int)threadIdx.x + {NT} * q, r_ = idx / {d // 4}, col = idx - r_ * {d // 4};")
        E(f"    if (idx < {pieces} && base0 + r_ < n) *(VTU*)({dst} + (base0 + r_) * {d} + 4 * col) = *(const VT*)(raw + r_ * {pitch} + 4 * col);")
        E("}")

    def _products(self, E: Emitter, chunks, offs, blocks, row_block, tile: str, base, tiles_of, apply, apart=lambda p: False) -> None:
        """The contractions of ``chunks``, one after the other, as slots of one product (a matrix step per path) with the
        loads of later slots and the Clebsch-Gordan part of finished paths (``apply``: a list of statements) spread
        between them: a wavefront issues in order, and a burst of loads or vector instructions is time its matrix core idles.
        ``apart``: paths whose five smaller products have an accumulator of their own."""
        KB = lambda ch: self.kblocks(blocks[row_block(ch[0])].mul)
        D = lambda ch: blocks[row_block(ch[0])].D
        steps = [(ci, kb) for ci, ch in enumerate(chunks) for kb in range(KB(ch))]
        matrix = [len(PRODUCTS) * D(chunks[ci]) * len(chunks[ci]) for ci, _ in steps]
        widest = max(tiles_of(q) for ch in chunks for q in ch)

        def fragments(n):
            """Loads of the weight fragments of step n."""
            ci, kb = steps[n]
            for p in chunks[ci]:
                nt = tiles_of(p)
                t_ = tile if nt == widest else f"min({tile}, {nt - 1})"
                for s in range(3):
                    yield f"const U4 a{n}_{p.t}_{s} = (wsp + ({base(p) + 64 * s + 192 * kb} + ({t_}) * {192 * KB(chunks[ci])}))[lane];"

        def rows(n, i):
            """LDS reads of component i of step n's rows."""
            ci, kb = steps[n]
            d, noct = D(chunks[ci]), 4 * KB(chunks[ci])
            at = offs[row_block(chunks[ci][0])] + (i * noct + 4 * kb) * 16
            return [f"const U4 b{n}_{i}_{s} = xrow{kb & 1}[{at + s * d * noct * 16}];" for s in range(3)]

        parts = [(n, i) for n, (ci, _) in enumerate(steps) for i in range(D(chunks[ci]))]
        E.extend(list(fragments(0)) + rows(0, 0))
        loaded, loads, after = 0, [], []
        for at, (n, i) in enumerate(parts):
            ci, kb = steps[n]
            ch = chunks[ci]
            if i == 0:
                # weight fragments one step ahead, further where the steps are short
                while loaded + 1 < len(steps) and (loaded == n or sum(matrix[n:loaded + 1]) < self.AHEAD):
                    loaded += 1
                    loads += list(fragments(loaded))
                per = _ceil(len(loads), len(PRODUCTS) * D(ch)) if loads else 0
            reads = rows(*parts[at + 1]) if at + 1 < len(parts) else []
            if kb == 0 and i == 0:
                E(f"// paths {[p.t for p in ch]}")
                for p in ch:
                    E("V4 " + ", ".join(f"{nm}{p.t}_{q} = {{0, 0, 0, 0}}" for nm in ("us" if apart(p) else "u") for q in range(D(ch))) + ";")
            for sa, sb in PRODUCTS:
                acc = [f"{'s' if sa + sb and apart(p) else 'u'}{p.t}_{i}" for p in ch]
                E(" ".join(f"{u} = oeq_mfma_bf16(a{n}_{p.t}_{sa}, b{n}_{i}_{sb}, {u}); OEQ_PIN({u});" for p, u in zip(ch, acc)))
                for _ in range(per):
                    if loads:
                        E(loads.pop(0))
                if reads:
                    E(reads.pop(0))
                for _ in range(self.BESIDE * len(ch)):
                    if after:
                        E(after.pop(0))
                E("oeq_sched_fence();")
            if kb + 1 == KB(ch) and i + 1 == D(ch):
                for p in ch:
                    if apart(p):
                        after += [f"u{p.t}_{q}[{r}] += s{p.t}_{q}[{r}];" for q in range(D(ch)) for r in range(4)]
                    after += apply(p)
        E.extend(after)

    # =============================================================== forward
    @property
    def forward_threads(self) -> int:
        return self.fwd_shape.threads if self.split_forward else 64

    def forward_attr(self) -> str:
        return " __attribute__((amdgpu_waves_per_eu(2)))" if self.split_forward else super().forward_attr()

    def _inside(self, shape: Shape, tile: str, count: int) -> str:
        return f"{tile} < {count}" + (f" && wv < {shape.waves * shape.tiles}" if shape.helpers else "")

    def forward_body(self) -> str:
        if not self.split_forward:
            return super().forward_body()
        E = Emitter()
        shape = self.fwd_shape
        NTW = max(p.NTW for p in self.paths)
        self._prologue(E, shape, self.D1, self.D3)
        for f in self.used_y:
            E(f"const T y{f} = Y[rowB * {self.D2} + {f}];")
        for req, put in self._rows_in(E, "X", self.D1, shape, "in"):
            E.extend(req + put)
        E("oeq_block_sync();")
        offs = self._split_rows(E, self.D1, self.in1, self.used_in1, shape)
        passes = self._passes(self.out, self.used_out, 4)
        through = len(passes) == 1 and NTW <= shape.waves and self.D3 % 4 == 0     # Z leaves through LDS
        E(f"if (const int wt = wave; {self._inside(shape, 'wt', NTW)}) {{" if NTW <= shape.waves
          else f"for (int wt = wave; {self._inside(shape, 'wt', NTW)}; wt += {shape.waves}) {{")
        E.level += 1
        for outs in passes:
            self._forward_pass(E, outs, offs, NTW)
            if through:
                E("oeq_priority(3);")
                E("oeq_block_sync();")
            for oi in outs:
                if through:
                    self._to_rows(E, self.D3, self.out[oi], "wt", lambda r, k, oi=oi: f"z{oi}_{k}[{r}]")
                else:
                    self._store_records(E, f"Z + (row0 + c) * {self.D3}", "bvalid", self.out[oi], "wt", lambda r, k, oi=oi: f"z{oi}_{k}[{r}]")
            E.level -= 1
            E("}")
        E.level -= 1
        E("}")
        if through:
            E("else oeq_block_sync();")
            self._rows_out(E, "Z", self.D3, self.out, self.used_out, shape)
        else:
            self._zero_blocks(E, "Z", self.D3, self.out, self.used_out)
        return E.text()

    def _forward_pass(self, E: Emitter, outs, offs, NTW: int) -> None:
        """Z of the output blocks ``outs`` in registers z{block}_{k} (leaves a block open)."""
        E(f"{{ // output blocks {outs}")
        E.level += 1
        for oi in outs:
            E("V4 " + ", ".join(f"z{oi}_{k} = {{0, 0, 0, 0}}" for k in range(self.out[oi].D)) + ";")

        def apply(p):
            terms, lines = {}, []
            for (i, j), ks in p.pairs.items():
                for k, val in ks:
                    terms.setdefault((i, k), []).append((j, val))
            for (i, k), lst in sorted(terms.items()):
                expr = " + ".join(f"{self.lit(val)} * y{p.b.off + j}" for j, val in sorted(lst))
                lines.append(f"const T m{p.t}_{i}_{k} = {expr};")
                lines += [f"z{p.o.idx}_{k}[{r}] = oeq_fma(m{p.t}_{i}_{k}, u{p.t}_{i}[{r}], z{p.o.idx}_{k}[{r}]);" for r in range(4)]
            return lines
        for nt in sorted({p.NTW for p in self.paths if p.o.idx in outs}):
            paths = [p for a in self.used_in1 for p in self.paths_from(a) if p.o.idx in outs and p.NTW == nt]
            chunks = [ch for a in sorted(self.used_in1, key=lambda a: -self.in1[a].D)
                      for ch in self._chunks([p for p in paths if p.a.idx == a], lambda p: p.a.D, lambda p: p.NTW)]
            E(f"if (wt < {nt}) {{" if nt < NTW else "{")
            E.level += 1
            self._products(E, chunks, offs, self.in1, lambda p: p.a.idx, "wt", lambda p: p.wb, lambda p: p.NTW, apply)
            E.level -= 1
            E("}")
        names = [f"z{oi}_{k}" for oi in outs for k in range(self.out[oi].D)]
        E("T fin = (T)0;")
        for nm in names:
            E(" ".join(f"fin = oeq_fma({nm}[{r}], (T)0, fin);" for r in range(4)))
        E(f"T back = {self.lit(BACK)};")
        E("if (oeq_any(!(fin == (T)0))) {   // infinities or NaN: again with fp32 multiply-adds")
        E.level += 1
        E("back = (T)1;")
        E(f"const T* __restrict__ Xr = X + rowB * {self.D1};")
        for nm in names:
            E(f"{nm} = V4{{0, 0, 0, 0}};")
        for oi in outs:
            for p in self.paths_into(oi):
                E("{")
                E.level += 1
                self.emit_cg_matrix(E, p, "y", "m")
                E("#pragma unroll 1")
                E(f"for (int u = 0; u < {p.mu}; ++u) {{")
                E.level += 1
                E("const T " + ", ".join(f"x{i} = Xr[{p.a.off + i} + u * {p.a.D}]" for i in range(p.a.D)) + ";")
                self.emit_cg_apply(E, p, "x", "m", "t")
                for r in range(4):
                    E(f"{{ const int w = min(16 * wt + 4 * g + {r}, {p.mw - 1}); const T wv_ = W[{self.oeq_index(p, 'u', 'w')}]; "
                      + " ".join(f"z{oi}_{k}[{r}] = oeq_fma(t{k}, wv_, z{oi}_{k}[{r}]);" for k in range(p.o.D)) + " }")
                E.level -= 1
                E("}")
                E.level -= 1
                E("}")
        E.level -= 1
        E("}")
        for nm in names:
            E(" ".join(f"{nm}[{r}] *= back;" for r in range(4)))

    def _zero_blocks(self, E: Emitter, dst: str, d: int, blocks, used) -> None:
        for o in blocks:
            if o.dim and o.idx not in used:
                E(f"if (wave == 0 && bvalid) for (int q = g; q < {o.dim}; q += 4) {dst}[(row0 + c) * {d} + {o.off} + q] = (T)0;")

    def _to_rows(self, E: Emitter, d: int, o, tile: str, val) -> None:
        self._store_records(E, f"raw + (16 * sub + c) * {self._row_pitch(d)}", "true", o, tile, val, d % 4 == 0 and o.off % 4 == 0)

    def _store_records(self, E: Emitter, row: str, valid: str, o, tile: str, val, wide: bool = True) -> None:
        """The four adjacent records of a lane (channels 16 tile + 4 g ..) of block ``o`` to the row at ``row``."""
        flat = [val(r, k) for r in range(4) for k in range(o.D)]
        E(f"if ({valid}) {{ const int ch = 16 * {tile} + 4 * g; T* __restrict__ zp = {row} + {o.off} + ch * {o.D};")
        E(f"    if (ch + 4 <= {o.mul}) {{")
        for i in range(o.D):
            if wide:
                E(f"        {{ VTU t_; " + " ".join(f"t_[{e}] = {flat[4 * i + e]};" for e in range(4)) + f" *({'VT' if row.startswith('raw') else 'VTU'}*)(zp + {4 * i}) = t_; }}")
            else:
                E("        " + " ".join(f"zp[{4 * i + e}] = {flat[4 * i + e]};" for e in range(4)))
        E("    }")
        if o.mul % 4:
            E("    else {")
            for r in range(3):
                E(f"        if (ch + {r} < {o.mul}) {{ " + " ".join(f"zp[{r * o.D + k}] = {val(r, k)};" for k in range(o.D)) + " }")
            E("    }")
        E("}")

    # ====================================================== backward: dX, dY
    def _apart(self, p) -> bool:
        """Whether V of a path sums its five smaller products apart from the largest.  An accumulator is a multiple of its last bit,
        so what a small addend loses to it is a matter of the addend alone, and of operands of one sign that is much the same for
all channels of a row: dY adds it up.  All operands in 0.5 .. 1.5, 4100 rows, relative error of dY against fp64, fp32
        kernel / together / apart: 200 channels (l <= 1) 4.9e-8 / 4.3e-8, 256 scalars 4.7 / 5.6 / 4.3, 384 5.5 / 6.9 / 4.7, 512
        5.4 / 8.2 / 4.2 (operands of mean zero 4.2e-7 / 3.4e-7 / 1.6e-7, dX 4.1e-7 / 3.4e-7 / 1.3e-7).  In time no difference: 256
        scalars, 40 000 rows, backward 117 / 116 us, 256 channels, l <= 1, 20 000 rows 195 / 195."""
        return self.kblocks(p.mw) >= 8

    @property
    def backward_threads(self) -> int:
        return self.bwd_shape.threads if self.split_dx else 256

    def backward_attr(self) -> str:
        return " __attribute__((amdgpu_waves_per_eu(2)))" if self.split_dx else super().backward_attr()

    def _records_in(self, E: Emitter, row: str, a, names, vector: str) -> None:
        """The four adjacent records of a lane (channels 16 ut + 4 g ..) of in1 block ``a`` into ``names``."""
        if a.mul % 4 == 0 and vector:
            E(f"{{ const T* __restrict__ xp = {row} + {a.off} + min(16 * ut + 4 * g, {a.mul - 4}) * {a.D};")
            for i in range(a.D):
                E(f"  {{ const {vector} t_ = *(const {vector}*)(xp + {4 * i}); " + " ".join(f"{names[4 * i + e]} = t_[{e}];" for e in range(4)) + " }")
            E("}")
        else:
            for r in range(4):
                E(f"{{ const T* __restrict__ xp = {row} + {a.off} + min(16 * ut + 4 * g + {r}, {a.mul - 1}) * {a.D}; "
                  + " ".join(f"{names[r * a.D + i]} = xp[{i}];" for i in range(a.D)) + " }")

    def backward_body(self) -> str:
        if not self.split_dx:
            return super().backward_body()
        E = Emitter()
        shape = self.bwd_shape
        NTU = max(p.NTU for p in self.paths)
        self._prologue(E, shape, self.D1, self.D3)
        E(f"__shared__ T dyl[{shape.waves * shape.tiles * 16 * max(1, self.D2)}];")
        E(f"const T* __restrict__ Xr = X + rowB * {self.D1};")
        for f in self.used_y:
            E(f"const T y{f} = Y[rowB * {self.D2} + {f}];")
            E(f"T dy{f} = (T)0;")
        passes = self._passes(self.in1, self.used_in1, 8)
        # X comes and dX leaves through LDS, as whole rows
        through = len(passes) == 1 and NTU <= shape.waves and self.D1 % 4 == 0
        rows = self._rows_in(E, "G", self.D3, shape, "gr")
        slot = {}
        if through:
            E(f"T xr[{4 * sum(self.in1[a].D for a in self.used_in1)}];")
            xin = self._rows_in(E, "X", self.D1, shape, "xr")
            for req, put in xin[:-1]:
                E.extend(req + put)
            E.extend(xin[-1][0] + rows[0][0] + xin[-1][1])       # the first dZ rows are on their way while X is dealt out
            E("oeq_block_sync();")
            E(f"if (const int ut = wave; {self._inside(shape, 'ut', NTU)}) {{")
            pos = 0
            for ai in self.used_in1:
                a, slot[ai] = self.in1[ai], pos
                self._records_in(E, f"raw + (16 * sub + c) * {self.D1}", a, [f"xr[{pos + q}]" for q in range(4 * a.D)],
                                 "VT" if a.off % 4 == 0 else "")
                pos += 4 * a.D
            E("}")
            E("oeq_block_sync();")
            E.extend(rows[0][1])
        else:
            E.extend(rows[0][0] + rows[0][1])
        for req, put in rows[1:]:
            E.extend(req + put)
        E("oeq_block_sync();")
        offs = self._split_rows(E, self.D3, self.out, self.used_out, shape)
        E(f"if (const int ut = wave; {self._inside(shape, 'ut', NTU)}) {{" if NTU <= shape.waves
          else f"for (int ut = wave; {self._inside(shape, 'ut', NTU)}; ut += {shape.waves}) {{")
        E.level += 1
        for ins in passes:
            self._backward_pass(E, ins, offs, NTU, slot)
            if through:
                E("oeq_priority(3);")
                E("oeq_block_sync();")
            for ai in ins:
                val = lambda r, i, ai=ai: f"dx{ai}_{r}_{i}"
                if through:
                    self._to_rows(E, self.D1, self.in1[ai], "ut", val)
                else:
                    self._store_records(E, f"Xg + (row0 + c) * {self.D1}", "bvalid", self.in1[ai], "ut", val)
            E.level -= 1
            E("}")
        E.level -= 1
        E("}")
        if through:
            E("else oeq_block_sync();")
            self._rows_out(E, "Xg", self.D1, self.in1, self.used_in1, shape)
        else:
            self._zero_blocks(E, "Xg", self.D1, self.in1, self.used_in1)
        waves, tiles = shape.waves, shape.tiles
        # ---- dY: sum over the 4 lane groups (channels), then over the tile's wavefronts, in pairs: eight sums of one sign one
        # after the other round at the size of the whole four times and more (512 channels, all operands positive: relative error
        # against fp64 9.0e-8, in pairs 8.2e-8; 128 channels, l <= 1, 5.8e-8 and 4.4e-8, the fp32 kernel's four 5.3e-8)
        for f in self.used_y:
            E(f"dy{f} += oeq_shfl_xor(dy{f}, 16);")
            E(f"dy{f} += oeq_shfl_xor(dy{f}, 32);")
        E(f"if (g == 0 && wv < {waves * tiles}) {{")
        for f in range(self.D2):
            E(f"    dyl[(wv * 16 + c) * {self.D2} + {f}] = " + (f"dy{f};" if f in self.used_y else "(T)0;"))
        E("}")
        E("oeq_block_sync();")
        E(f"for (int q = threadIdx.x; q < {16 * tiles * self.D2}; q += {self.backward_threads}) {{")
        E(f"    const int r_ = q / {self.D2}, f = q - r_ * {self.D2};")
        E(f"    const T* __restrict__ s_ = dyl + ((r_ >> 4) * {16 * waves} + (r_ & 15)) * {self.D2} + f;")
        terms = [f"s_[{w * 16 * self.D2}]" for w in range(waves)]
        while len(terms) > 1:
            terms = [f"({' + '.join(terms[q:q + 2])})" for q in range(0, len(terms), 2)]
        E(f"    if (base0 + r_ < n) Yg[(base0 + r_) * {self.D2} + f] = {terms[0]};")
        E("}")
        return E.text()

    def _backward_pass(self, E: Emitter, ins, offs, NTU: int, slot: dict) -> None:
        """dX of the in1 blocks ``ins`` in registers dx{block}_{r}_{i}, their share of dY added to dy (leaves a block open).
        ``slot``: where the blocks' X records are among the registers xr, empty if they are still to be loaded."""
        E(f"{{ // in1 blocks {ins}")
        E.level += 1
        E("const int ch = 16 * ut + 4 * g;     // this lane's four channels")
        for ai in ins:
            a = self.in1[ai]
            names = [f"x{ai}_{r}_{i}" for r in range(4) for i in range(a.D)]
            if slot:
                E("const T " + ", ".join(f"{nm} = xr[{slot[ai] + q}]" for q, nm in enumerate(names)) + ";")
            else:
                E("T " + ", ".join(names) + ";")
                self._records_in(E, "Xr", a, names, "VTU")
            E("T " + ", ".join(f"d{nm} = (T)0" for nm in names) + ";")
        sums = [f"dy{f}" for f in self.used_y]
        E("const T " + ", ".join(f"was_{nm} = {nm}" for nm in sums) + ";")
        E(" ".join(f"{nm} = (T)0;" for nm in sums))

        def apply(p):
            lines = []
            for r in range(4):
                for (i, j), ks in p.ordered_pairs():
                    s = f"{self.lit(ks[0][1])} * u{p.t}_{ks[0][0]}[{r}]"
                    for k, val in ks[1:]:
                        s = f"oeq_fma({self.lit(val)}, u{p.t}_{k}[{r}], {s})"
                    lines.append(f"const T s{p.t}_{r}_{i}_{j} = {s};")
                    lines.append(f"dx{p.a.idx}_{r}_{i} = oeq_fma(s{p.t}_{r}_{i}_{j}, y{p.b.off + j}, dx{p.a.idx}_{r}_{i});")
                    lines.append(f"dy{p.b.off + j} = oeq_fma(s{p.t}_{r}_{i}_{j}, x{p.a.idx}_{r}_{i}, dy{p.b.off + j});")
            return lines
        for nt in sorted({p.NTU for p in self.paths if p.a.idx in ins}):
            paths = [p for p in self.paths if p.a.idx in ins and p.NTU == nt]
            chunks = [ch for o in sorted(self.used_out, key=lambda o: -self.out[o].D)
                      for ch in self._chunks([p for p in paths if p.o.idx == o], lambda p: p.o.D * (2 if self._apart(p) else 1), lambda p: p.NTU)]
            E(f"if (ut < {nt}) {{" if nt < NTU else "{")
            E.level += 1
            self._products(E, chunks, offs, self.out, lambda p: p.o.idx, "ut", lambda p: p.wa, lambda p: p.NTU, apply, self._apart)
            E.level -= 1
            E("}")
        names = [f"dx{ai}_{r}_{i}" for ai in ins for r in range(4) for i in range(self.in1[ai].D)]
        E("T fin = (T)0;")
        for nm in names + sums:
            E(f"fin = oeq_fma({nm}, (T)0, fin);")
        E(f"T back = {self.lit(BACK)};")
        E("if (oeq_any(!(fin == (T)0))) {   // infinities or NaN: again with fp32 multiply-adds")
        E.level += 1
        E("back = (T)1;")
        E(f"const T* __restrict__ Gr = G + rowB * {self.D3};")
        for nm in names + sums:
            E(f"{nm} = (T)0;")
        for ai in ins:
            for p in self.paths_from(ai):
                E("{")
                E.level += 1
                E("T " + ", ".join(f"dt{r}_{k} = (T)0" for r in range(4) for k in range(p.o.D)) + ";")
                E("#pragma unroll 1")
                E(f"for (int w = 0; w < {p.mw}; ++w) {{")
                E.level += 1
                E("const T " + ", ".join(f"g{k} = Gr[{p.o.off + k} + w * {p.o.D}]" for k in range(p.o.D)) + ";")
                for r in range(4):
                    E(f"{{ const int u = min(ch + {r}, {p.mu - 1}); const T wv_ = W[{self.oeq_index(p, 'u', 'w')}]; "
                      + " ".join(f"dt{r}_{k} = oeq_fma(wv_, g{k}, dt{r}_{k});" for k in range(p.o.D)) + " }")
                E.level -= 1
                E("}")
                for r in range(4):
                    E(f"if (ch + {r} < {p.mu}) {{")
                    E.level += 1
                    self.emit_cg_backward(E, p, f"dt{r}_", f"x{ai}_{r}_", "y", f"dx{ai}_{r}_", "dy")
                    E.level -= 1
                    E("}")
                E.level -= 1
                E("}")
        E.level -= 1
        E("}")
        for nm in names:
            E(f"{nm} *= back;")
        for nm in sums:
            E(f"{nm} = oeq_fma({nm}, back, was_{nm});")

    # ============================================================ backward: dW
    DW_REGISTERS = 160           # accumulators and X records of a wavefront
    DW_LDS = 160 * 1024

    @cached_property
    def dw_kinds(self):
        """Workgroup kinds of the dW kernel, a list of DWKind, or None where the fp32 kernel serves the problem.  A kind stages at
        most 64 channels of its output blocks; its jobs are bins of paths (with a range of w tiles) from one in1 block times
        32-channel tiles of u, one per wavefront.

        Not where T, split for a single w tile that is half padding, is most of the work (from three u tiles on within
        2 % of the fp32 kernel), nor where each kind of workgroup, which
        fetches and splits rows for itself, has one path for each and pads to 32 besides.  40 000 rows, backward on the fp32 dX
        with the fp32 / split dW kernel, us (gain as in ``_pays``):

            in1 -> out, l <= 2            in2 l <= 2                1x0e
            64 -> 8                   1.33   125 /  132
            96 -> 9                   1.33   268 /  274
            100 -> 12                 1.17   335 /  334      (100 -> 8)  1.17   149 /  142
            32 -> 16                  1.33   123 /   99      (64 -> 16)  1.33    94 /   91
            8 -> 100                  1.17   440 /  236
            9 -> 33                   1.00   178 /  126
            64 | 65, 4 kinds of 65    2.67   268 /  238                  1.85   206 /  221
            100, 4 kinds              2.04  1590 /  640                  2.04   311 /  278
            40 | 64 both, 3 kinds                                 1.50 201 / 208, 2.67 279 / 280
            33 | 96 both, 4 | 6 kinds 1.50   708 /  494                  2.67  1105 /  630
            128, 4 kinds              2.67  2449 /  757
            200, 15 kinds             2.30  8036 / 3136"""
        tiles = lambda o: _ceil(self.out[o].mul, 32)
        if max(p.mw for p in self.paths) <= 16 and 32 < max(p.mu for p in self.paths) <= 64 and len(self.paths) > 2 * len(self.used_in1):
            return None
        kinds: List[DWKind] = []
        for lo in range(0, max(tiles(o) for o in self.used_out), 2):
            blocks = [(o, lo, min(lo + 2, tiles(o))) for o in self.used_out if tiles(o) > lo]
            while blocks:                                     # as many output blocks as LDS holds, twice
                some = []
                while blocks and (not some or DWKind(self, some + blocks[:1]).lds_bytes() <= self.DW_LDS):
                    some.append(blocks.pop(0))
                base = DWKind(self, some)
                if base.lds_bytes() > self.DW_LDS:
                    return None
                bins = self._dw_bins(base)
                if bins is None:
                    return None
                jobs = sorted(((b, u) for b, m in enumerate(bins) for u in range(_ceil(m[0][0].mu, 32))),
                              key=lambda j: (-base.cost(bins[j[0]]), j))
                count, per = _ceil(len(jobs), 8), max(1, 8 // len(bins))
                # all bins of ``per`` tiles of u each, whose kinds share their code, where that takes no more kinds
                ranged = [[j for j in jobs if j[1] // per == q] for q in range(_ceil(1 + max(u for _, u in jobs), per))]
                dealt = ranged if len(bins) <= 8 and len(ranged) <= count else [jobs[q::count] for q in range(count)]
                for mine in dealt:
                    # wavefronts w and w + 4 share a SIMD: the most expensive jobs beside the cheapest
                    head, tail = mine[:4], mine[4:]
                    waves = head + [None] * (4 - len(head)) + ([None] * (4 - len(tail)) + tail[::-1])
                    kinds.append(DWKind(self, some, bins, waves))
        # cycles of the fp32 instruction over those of the split one
        gain = (sum(128 * p.NTU * p.NTW * p.o.D for p in self.paths)
                / sum(192 * _ceil(p.mu, 32) * _ceil(p.mw, 32) * p.o.D for p in self.paths))
        if len(kinds) >= 3 and self._single(self.used_out) and gain < 2:
            return None
        # (code and compile time grow with the column ranges: 64 channels 4 s where the fp32 kernels take 2, 100 channels 9 and 5,
        # 200 channels with four ranges 43 and 13)
        return kinds if len(kinds) <= 16 and len({tuple(k.blocks) for k in kinds}) <= 4 else None

    def _dw_bins(self, kind: "DWKind"):
        """The kind's paths in bins of one in1 block each, within DW_REGISTERS and of about an eighth of the work per bin."""
        segs = [(p, lo, hi) for p in self.paths for o, lo, hi in kind.blocks if p.o.idx == o]
        acc = lambda m: sum(16 * (hi - lo) for _, lo, hi in m)
        target = kind.cost(segs) / max(1, 8 // max(_ceil(p.mu, 32) for p, _, _ in segs))
        bins = []
        for a in self.used_in1:
            mine = sorted((sg for sg in segs if sg[0].a.idx == a), key=lambda sg: -kind.cost([sg]))
            if not mine:
                continue
            room = self.DW_REGISTERS - 8 * self.in1[a].D
            if max(acc([sg]) for sg in mine) > room:
                return None
            count = max(_ceil(acc(mine), room), round(kind.cost(mine) / target), 1)
            while True:
                parts = [[] for _ in range(count)]
                for sg in mine:
                    fits = [m for m in parts if acc(m + [sg]) <= room]
                    if not fits:
                        break
                    min(fits, key=kind.cost).append(sg)
                else:
                    break
                count += 1
            bins += [m for m in parts if m]
        return bins

    @property
    def dw_threads(self) -> int:
        return 512 if self.dw_kinds else super().dw_threads

    def dw_globals(self) -> str:
        if not self.dw_kinds:
            return ""
        out = []
        for q, kind in ((m[0], self.dw_kinds[m[0]]) for m in self._dw_programs()):
            coeff, first = [], []
            for _, y, c in sorted(kind.entries.values()):
                at = min(y, self.D2 - kind.width)            # every entry reads ``width`` values of Y, within the row
                first.append(at)
                coeff += [0.0] * (y - at) + c + [0.0] * (kind.width - (y - at) - len(c))
            out.append(f"__constant__ T oeq_m_coeff{q}[{len(coeff)}] = {{" + ", ".join(self.lit(v) for v in coeff) + "};")
            out.append(f"__constant__ int oeq_m_first{q}[{len(first)}] = {{" + ", ".join(map(str, first)) + "};")
        return "\n".join(out)

    def backward_dw_body(self) -> str:
        kinds = self.dw_kinds
        if not kinds:
            return super().backward_dw_body()
        D2 = self.D2
        E = Emitter()
        E("const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;")
        E("const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));")
        E("const u64 ntiles = (n + 15) / 16;")
        share = self.DW_WORKGROUPS // len(kinds)
        E(f"const int kind = blockIdx.x / {share}, first = blockIdx.x % {share};")
        E(f"const u64 step = {share};")
        E(f"if (kind >= {len(kinds)} || (u64)first >= ntiles) return;")
        # (one array, divided by each kind: the kind that stages most of dZ need not be the one with most entries of M)
        E(f"__shared__ U4 lds[{max(k.lds_units for k in kinds)}];")
        E("T* __restrict__ yl = (T*)lds;                                // Y of a tile: two buffers")
        E(f"T* __restrict__ part = (T*)ws + {self.PART_OFF} + (u64)first * {self.WN};")
        # Y of the first two tiles
        E(f"for (int q = threadIdx.x; q < {32 * D2}; q += 512) {{")
        E(f"    const u64 row = ((u64)first + (q >= {16 * D2} ? step : 0)) * 16 + (q % {16 * D2}) / {D2};")
        E(f"    yl[q] = row < n ? Y[row * {D2} + q % {D2}] : (T)0;      // rows past the end: M = 0, T = 0")
        E("}")
        for members in self._dw_programs():
            kind, q = kinds[members[0]], members[0]
            E(f"if ({' || '.join(f'kind == {m}' for m in members)}) {{   // output blocks (w tiles) {kind.blocks}")
            E.level += 1
            E(f"U4* __restrict__ gs = lds + {8 * D2};                      // dZ of a tile, split: two buffers")
            E(f"VT* __restrict__ mt = (VT*)(gs + {2 * kind.units});        // M of a tile, [entry][row]: two buffers")
            code = {}
            for w, job in enumerate(kind.waves):
                code.setdefault(job[0] if job else None, []).append(w)
            stage = self._dw_stage(kind, code)
            for at, (b, waves) in enumerate(code.items()):
                E(f"{'else ' if at else ''}if ({' || '.join(f'wv == {w}' for w in waves)}) {{")
                E.level += 1
                cases = [(m, w, kinds[m].waves[w][1] if kinds[m].waves[w] else 0) for m in members for w in waves]
                E("const int ut = " + "".join(f"kind == {m} && wv == {w} ? {u} : " for m, w, u in cases[:-1]) + f"{cases[-1][2]};")
                E("const int turn = " + "".join(f"wv == {w} ? {t} : " for t, w in enumerate(waves[:-1])) + f"{len(waves) - 1};")
                self._dw_bin(E, kind, q, kind.bins[b] if b is not None else [], stage[b], len(waves))
                E.level -= 1
                E("}")
            E.level -= 1
            E("}")
        return E.text()

    def _dw_programs(self):
        """Kinds (by number) that differ only in the 32-channel tiles of u of their wavefronts."""
        programs = {}
        for q, kind in enumerate(self.dw_kinds):
            key = tuple(kind.blocks), tuple(job and job[0] for job in kind.waves)
            programs.setdefault(key, []).append(q)
        return list(programs.values())

    def _dw_matrix(self, kind: "DWKind", q: int, buf: str, sign: str):
        """M of the tile whose Y is in yl[buf], times ``sign`` -> mt[buf]: a thread takes four rows of an entry."""
        n, D2 = len(kind.entries), self.D2
        yield f"for (int q = threadIdx.x; q < {4 * n}; q += 512) {{"
        yield f"    const int e = q >> 2, r = 4 * (q & 3); const T* __restrict__ yp = yl + ({buf}) * {16 * D2} + r * {D2} + oeq_m_first{q}[e];"
        yield "    VT m_; m_[0] = m_[1] = m_[2] = m_[3] = (T)0;"
        yield (f"    for (int j = 0; j < {kind.width}; ++j) {{ const T cf = oeq_m_coeff{q}[e * {kind.width} + j]; "
               + " ".join(f"m_[{r}] = oeq_fma(cf, yp[{r * D2} + j], m_[{r}]);" for r in range(4)) + " }")
        yield f"    mt[({buf}) * {4 * n} + q] = m_ * ({sign});"
        yield "}"

    @staticmethod
    def _dw_stage(kind: "DWKind", code) -> dict:
        """Output blocks whose dZ a bin's wavefronts split: dealt to the bins with registers to spare."""
        stage = {b: [] for b in code}
        need = {b: (sum(16 * (hi - lo) for _, lo, hi in kind.bins[b]) + 8 * kind.bins[b][0][0].a.D if b is not None else 0) for b in code}
        turns = lambda b, blk: _ceil(blk[2] - blk[1], len(code[b]))
        for blk in sorted(kind.blocks, key=lambda blk: -kind.g.out[blk[0]].D * (blk[2] - blk[1])):
            regs = lambda b: 8 * kind.g.out[blk[0]].D * turns(b, blk)
            b = min(code, key=lambda b: need[b] + regs(b))
            need[b] += regs(b)
            stage[b].append(blk)
        return stage

    def _dw_bin(self, E: Emitter, kind: "DWKind", at_kind: int, segs, stage, members: int) -> None:
        """The walk over the batch of the wavefronts that hold dW of ``segs`` (32 channels u) and split dZ of ``stage``."""
        a = segs[0][0].a if segs else None
        D2, entries = self.D2, len(kind.entries)
        cells = [(p, wt) for p, lo, hi in segs for wt in range(lo, hi)]
        for p, wt in cells:
            E("T " + ", ".join(f"acc{p.t}_{wt}_{r} = (T)0" for r in range(16)) + ";")
        tasks = [(blk, q) for blk in stage for q in range(_ceil(blk[2] - blk[1], members))]
        for (o, _, _), q in tasks:
            E("T " + ", ".join(f"g{o}_{q}_{j}_{k}" for j in range(8) for k in range(self.out[o].D)) + ";")
        if a:
            E("T " + ", ".join(f"x{j}_{i}" for j in range(8) for i in range(a.D)) + ";")
            E(f"const int ux = {a.off} + min(32 * ut + c, {a.mul - 1}) * {a.D};")

        def rows(tile):
            """First row of a tile and the last valid one in it."""
            E(f"const u64 r0 = ({tile}) * 16; const int lim = (int)min((u64)15, n - 1 - r0);")

        def x_loads():
            for j in range(8):
                yield (f"{{ const T* __restrict__ xp = X + r0 * {self.D1} + (min(8 * h + {j}, lim) * {self.D1} + ux); "
                       + " ".join(f"x{j}_{i} = xp[{i}];" for i in range(a.D)) + " }")

        def task(blk, q):
            """(width staged, statement that finds this lane's octet of rows hh and column w of task q of a block)."""
            np_ = 32 * (blk[2] - blk[1])
            return np_, f"const int ix = 64 * (turn + {members * q}) + lane, hh = ix / {np_}, w = ix % {np_};"

        def load_g():
            E(f"const T* __restrict__ Gt = G + r0 * {self.D3};")
            for blk, q in tasks:
                o, (np_, find) = self.out[blk[0]], task(blk, q)
                E("{ " + find)
                E("if (hh < 2) {")
                for j in range(8):
                    E(f"  {{ const T* __restrict__ gp = Gt + (min(8 * hh + {j}, lim) * {self.D3} + {o.off} + min({32 * blk[1]} + w, {o.mul - 1}) * {o.D}); "
                      + " ".join(f"g{o.idx}_{q}_{j}_{k} = gp[{k}];" for k in range(o.D)) + " }")
                E("} }")

        def split_g(buf):
            for blk, q in tasks:
                o, (np_, find) = self.out[blk[0]], task(blk, q)
                E("{ " + find)
                E(f"if (hh < 2) {{ U4* __restrict__ d = gs + ({buf}) * {kind.units} + {kind.offs[o.idx]} + hh * {np_} + w;")
                for k in range(o.D):
                    E(f"  {{ const T e[8] = {{{', '.join(f'{self.lit(SCALE)} * g{o.idx}_{q}_{j}_{k}' for j in range(8))}}}; U4 a_, b_, c_; oeq_split8(e, a_, b_, c_); "
                      + " ".join(f"d[{(s * o.D + k) * 2 * np_}] = {nm};" for s, nm in enumerate(("a_", "b_", "c_"))) + " }")
                E("} }")

        E("{")
        rows("(u64)first")
        load_g()
        if a:
            E.extend(x_loads())
        E("oeq_block_sync();                               // yl")
        E.extend(self._dw_matrix(kind, at_kind, "0", f"first & 1 ? {self.lit(-SCALE)} : {self.lit(SCALE)}"))
        split_g("0")
        E("}")
        E("oeq_block_sync();")
        E("int buf = 0;")
        E(f"T sign = first & 1 ? {self.lit(-SCALE)} : {self.lit(SCALE)};")
        E("for (u64 tile = first; tile < ntiles; tile += step) {")
        E.level += 1
        E(f"const U4* __restrict__ gb = gs + buf * {kind.units} + h * 32 + c;")
        E(f"const VT* __restrict__ mb = mt + buf * {4 * entries} + 2 * h;")
        E("const u64 next = tile + step, after = next + step;")
        E(f"const T back = sign * {self.lit(BACK / SCALE)};")
        # (the last tile fetches itself again rather than branch around the requests)
        rows("next < ntiles ? next : tile")
        load_g()
        turns = _ceil(16 * D2, 512)                          # Y of the tile after the next one
        for q in range(turns):
            E(f"T yn{q} = (T)0; {{ const int ix = (int)threadIdx.x + {512 * q}; const u64 row = after * 16 + ix / {D2}; "
              f"if (ix < {16 * D2} && row < n) yn{q} = Y[after * {16 * D2} + ix]; }}")
        # T of each (path, component) is formed and split beside the matrix steps of the one before it
        work = [(sg, k) for sg in segs for k in range(sg[0].o.D)]

        def operand(n):
            """Statements that leave T of ``work[n]`` split in t{n}_{split}."""
            (p, _, _), k = work[n]
            terms = [i for i in range(p.a.D) if (p.t, i, k) in kind.entries]
            out = [f"U4 t{n}_0, t{n}_1, t{n}_2;"]
            for half in range(2):
                for at, i in enumerate(terms):
                    out.append(f"const VT m{n}_{half}_{i} = mb[{4 * kind.entries[p.t, i, k][0] + half}];")
                    out += [(f"T v{n}_{4 * half + r} = " if at == 0 else f"v{n}_{4 * half + r} = ")
                            + (f"m{n}_{half}_{i}[{r}] * x{4 * half + r}_{i};" if at == 0
                               else f"oeq_fma(m{n}_{half}_{i}[{r}], x{4 * half + r}_{i}, v{n}_{4 * half + r});") for r in range(4)]
                if not terms:
                    out += [f"const T v{n}_{4 * half + r} = (T)0;" for r in range(4)]
                for q in (2 * half, 2 * half + 1):
                    out.append(f"{{ unsigned a_, b_, c_; oeq_split2(v{n}_{2 * q}, v{n}_{2 * q + 1}, a_, b_, c_); OEQ_PIN(a_); OEQ_PIN(b_); OEQ_PIN(c_); t{n}_0[{q}] = a_; t{n}_1[{q}] = b_; t{n}_2[{q}] = c_; }}")
            return out

        def columns(n, wt):
            (p, lo, hi), k = work[n]
            np_ = 32 * (hi - lo)
            at = kind.offs[p.o.idx] + k * 2 * np_ + 32 * (wt - lo)
            # (gb points 32 units further for the second octet of rows, np_ is what lies between the two)
            return [f"const U4 b{n}_{wt}_{s} = gb[{at + s * p.o.D * 2 * np_}{f' + h * {np_ - 32}' if np_ != 32 else ''}];" for s in range(3)]
        steps = [(n, wt) for n, ((_, lo, hi), _) in enumerate(work) for wt in range(lo, hi)]
        # The six products of a step are summed apart and added to the accumulators as a whole: a matrix step rounds at the size
        # of what it adds to, which is too often at the size of the sum over the batch; and it rounds downwards, so every other
        # tile, and workgroup, is summed negated (M carries the sign) and what that adds up to cancels
        sums = 2 if 16 * len(cells) <= 96 else 1
        if work:
            E.extend(operand(0) + columns(0, steps[0][1]))
            E("V16 " + ", ".join(f"s{q}" for q in range(sums)) + ";")
        adds = []
        for at, (n, wt) in enumerate(steps):
            (p, lo, hi), k = work[n]
            if wt == lo:
                beside = operand(n + 1) if n + 1 < len(work) else []
            if n + 1 == len(work) and wt == lo:              # the X records have been used for the last time
                E.extend(x_loads())
            reads = columns(*steps[at + 1]) if at + 1 < len(steps) else []
            left = len(PRODUCTS) * (hi - wt)
            for q, (sa, sb) in enumerate(PRODUCTS):
                if q == 0:
                    E(f"for (int r = 0; r < 16; ++r) s{at % sums}[r] = (T)0;")
                E(f"s{at % sums} = oeq_mfma32_bf16(t{n}_{sa}, b{n}_{wt}_{sb}, s{at % sums}); OEQ_PIN(s{at % sums});")
                for _ in range(_ceil(len(beside), left - q)):
                    E(beside.pop(0))
                for _ in range(_ceil(len(adds), len(PRODUCTS) - q)):
                    E(adds.pop(0))
                if reads:
                    E(reads.pop(0))
                E("oeq_sched_fence();")
            adds = [f"acc{p.t}_{wt}_{r} = oeq_fma(back, s{at % sums}[{r}], acc{p.t}_{wt}_{r}); OEQ_PIN(acc{p.t}_{wt}_{r});" for r in range(16)]
            if sums == 1 or at + 1 == len(steps):
                E.extend(adds)
                adds = []
        E("if (next < ntiles) {")
        E.level += 1
        split_g("1 - buf")
        E.extend(self._dw_matrix(kind, at_kind, "1 - buf", "-sign"))
        for q in range(turns):
            E(f"{{ const int ix = (int)threadIdx.x + {512 * q}; if (ix < {16 * D2}) yl[buf * {16 * D2} + ix] = yn{q}; }}")
        E.level -= 1
        E("}")
        E("buf = 1 - buf;")
        E("sign = -sign;")
        E("oeq_block_sync();")
        E.level -= 1
        E("}")
        for p, wt in cells:
            E(f"{{ // path {p.t}, w tile {wt}")
            E.level += 1
            for r in range(16):
                E(f"{{ const int u = 32 * ut + {8 * (r // 4) + r % 4} + 4 * h, w = {32 * wt} + c; if (u < {p.mu} && w < {p.mw}) part[{p.poff} + u * {p.mw} + w] = acc{p.t}_{wt}_{r}; }}")
            for q in range(4):
                E(f"T fin{q} = (T)0; " + " ".join(f"fin{q} = oeq_fma(acc{p.t}_{wt}_{4 * q + r}, (T)0, fin{q});" for r in range(4)))
            E("const int again = " + " | ".join(f"(oeq_any(!(fin{q} == (T)0)) ? {1 << q} : 0)" for q in range(4)) + ";")
            # infinities or NaN: the four channels u of a lane with some again with fp32 multiply-adds, until all sums are NaN
            E("#pragma unroll 1")
            E("for (int q = 0; q < 4; ++q) {")
            E.level += 1
            E("if (!(again >> q & 1)) continue;")
            E(f"const int u = 32 * ut + 8 * q + 4 * h, w = {32 * wt} + c;")
            E("T " + ", ".join(f"sum{r} = (T)0" for r in range(4)) + "; bool open = true;")
            E("for (u64 tile = first; open && tile < ntiles; tile += step) {")
            E.level += 1
            E("#pragma unroll 1")
            E("for (u64 row = tile * 16; row < min(n, tile * 16 + 16); ++row) {")
            E.level += 1
            for f in sorted({p.b.off + j for (_, j) in p.pairs}):
                E(f"const T y{f} = Y[row * {self.D2} + {f}];")
            E(f"const T* __restrict__ gp = G + row * {self.D3} + {p.o.off} + min(w, {p.mw - 1}) * {p.o.D};")
            E("const T " + ", ".join(f"g{k} = gp[{k}]" for k in range(p.o.D)) + ";")
            self.emit_cg_matrix(E, p, "y", "m")
            for r in range(4):
                E(f"{{ const T* __restrict__ xp = X + row * {self.D1} + {p.a.off} + min(u + {r}, {p.mu - 1}) * {p.a.D};")
                E.level += 1
                E("const T " + ", ".join(f"x{i} = xp[{i}]" for i in range(p.a.D)) + ";")
                self.emit_cg_apply(E, p, "x", "m", "t")
                E(" ".join(f"sum{r} = oeq_fma(t{k}, g{k}, sum{r});" for k in range(p.o.D)) + " }")
                E.level -= 1
            E.level -= 1
            E("}")
            E("open = oeq_any(sum0 == sum0 || sum1 == sum1 || sum2 == sum2 || sum3 == sum3);")
            E.level -= 1
            E("}")
            for r in range(4):
                E(f"if (u + {r} < {p.mu} && w < {p.mw}) part[{p.poff} + (u + {r}) * {p.mw} + w] = sum{r};")
            E.level -= 1
            E("}")
            E.level -= 1
            E("}")

    def reduce_body(self) -> str:
        if not self.dw_kinds:
            return super().reduce_body()
        E = Emitter()
        # 64 weights a workgroup, its four wavefronts take every fourth partial row
        E("const int q = blockIdx.x * 64 + (threadIdx.x & 63), sl = threadIdx.x >> 6;")
        E("__shared__ T sums[192];")
        E(f"const int live = (int)min((u64){self.DW_WORKGROUPS // len(self.dw_kinds)}, (n + 15) / 16);")
        E(f"const T* __restrict__ part = (const T*)ws + {self.PART_OFF} + min(q, {self.WN - 1});")
        # (eight sums side by side: loads in flight, and short chains of roundings)
        E("T a[8]; for (int j = 0; j < 8; ++j) a[j] = (T)0;")
        E("int b = sl;")
        E(f"for (; b + 28 < live; b += 32) for (int j = 0; j < 8; ++j) a[j] += part[(u64)(b + 4 * j) * {self.WN}];")
        E(f"for (int j = 0; j < 8; ++j) if (b + 4 * j < live) a[j] += part[(u64)(b + 4 * j) * {self.WN}];")
        E("const T acc = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));")
        E("if (sl > 0) sums[(sl - 1) * 64 + (threadIdx.x & 63)] = acc;")
        E("oeq_block_sync();")
        E("int dst = q;")
        for p in self.paths:
            E(f"if (q >= {p.poff} && q < {p.poff + p.mu * p.mw}) {{ const int e = q - {p.poff}; const int u = e / {p.mw}; const int w = e - u * {p.mw}; dst = {self.oeq_index(p, 'u', 'w')}; }}")
        E(f"if (sl == 0 && q < {self.WN}) Wg[dst] = ((acc + sums[threadIdx.x]) + sums[64 + threadIdx.x]) + sums[128 + threadIdx.x];")
        return E.text()

    # ---------------------------------------------------------------- rendering
    # Sources by problem, as writing one takes longer than all else a built operator does (64 channels, 11 paths, 780 KB: 15 ms,
    # the fp32 kernels' 7): the layers of a model share it.  Bounded: the least recently asked for goes.
    _SOURCES: "OrderedDict[tuple, str]" = OrderedDict()
    _SOURCES_MAX = 16
    _sources_lock = threading.Lock()

    def render(self, prelude: str = None) -> str:
        if prelude is not None:
            return super().render(prelude)
        key = self.problem.signature()
        with self._sources_lock:
            source = self._SOURCES.get(key)
            if source is not None:
                self._SOURCES.move_to_end(key)
                return source
        source = super().render()
        with self._sources_lock:
            self._SOURCES[key] = source
            while len(self._SOURCES) > self._SOURCES_MAX:
                self._SOURCES.popitem(last=False)
        return source

    def describe(self) -> str:
        return super().describe().replace("mfma=16x16x4", "mfma=16x16x32 bf16 split in three")

    def plan(self):
        fwd, bwd, ws = super().plan()
        if self.split_forward:
            fwd[1].update(num_threads=self.forward_threads, work_per_block=16 * self.fwd_shape.tiles, grid_y=1)
        bwd[0]["num_blocks"] = self.prep_backward_blocks
        if self.split_dx:
            bwd[1]["work_per_block"] = 16 * self.bwd_shape.tiles
        if self.dw_kinds:
            bwd[3]["num_blocks"] = _ceil(self.WN, 64)
        return fwd, bwd, ws
