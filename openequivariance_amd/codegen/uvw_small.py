"""Dense "uvw" tensor products with shared weights on batches of few rows (same contraction and packing as
:mod:`.uvw`; reference: templates/loop_unroll_tp.cuh:74-78, :184, :209).

The kernels of :mod:`.uvw` give a 16-row tile to one workgroup and a whole output block to one wavefront, and let every
dW workgroup walk all paths.  With fewer tiles than the chip has places for them, the longest of those serial chains is
the time of a launch.  Here the same work is cut finer:

* forward: output blocks in ranges of w tiles of at most ``FWD_ACC_LIMIT`` accumulators per work item;
* backward dX/dY: the in1 blocks of a tile are dealt to two or four groups of four wavefronts, which share the dZ tile;
* backward dW: a workgroup holds ONE path (or a range of its w tiles) and walks a share of the batch given by the path's
  cost; its 16 wavefronts are u-subtiles x phases of the batch, combined through LDS, so that the launch leaves 15 to 80
  partial rows of a path instead of 256 of all paths.  It comes first and packs the weights that dX reads.

Bound: latency of the operand loads, four wavefronts per SIMD hide what one did not.  50x0e+50x1o+50x1e+50x2o+50x2e with
one scalar, fp64, 4097 rows (kernel times, us): dX/dY 41 -> 30, dW 35 -> 19, reduction 16.7 -> 4.6; fp32 backward of that
product as a whole 65 -> 46.  64x0e+64x1o+64x2e, 500 rows: forward 29 -> 20 and backward 57 -> 29 in fp32, 44 -> 30 and
81 -> 44 in fp64.
"""
from __future__ import annotations

from typing import List

from ..problem import TPProblem
from .common import Emitter
from .uvw import UVWGenerator, _ceil


class UVWSmallGenerator(UVWGenerator):
    FWD_ACC_LIMIT = 40           # accumulator tiles x 4 of one forward work item (two w tiles of an l = 2 block)
    BWD_LDS_LIMIT = 144 * 1024   # the dZ tile may fill a compute unit: there is one workgroup for each at most
    LDS_BYTES = 160 * 1024       # of a compute unit: what a kernel's arrays together may take (see lds_bytes)
    FWD_PIPELINE = {4: (4, 2), 8: (1, 4)}
    FWD_NO_MULTIPLE = {4: 0, 8: 0}
    DW_WAVES = 16
    DW_REGISTERS = 88            # of 128 a lane has with 16 wavefronts: accumulators, operands and one T of a dW unit

    def __init__(self, problem: TPProblem):
        super().__init__(problem)
        words = self.itemsize // 4
        # in1 blocks of the backward by group of wavefronts, balanced by matrix-core steps.  fp64 takes 256 registers a
        # lane (two groups), fp32 about 120 (four)
        cost = {a: sum(p.o.D * p.SW * p.NTU for p in self.paths_from(a)) for a in self.used_in1}
        groups: List[List[int]] = [[] for _ in range(min(4 if words == 1 else 2, len(cost)))]
        if self.bwd_lds:
            for a in sorted(cost, key=lambda k: -cost[k]):
                min(groups, key=lambda m: sum(cost[k] for k in m)).append(a)
            self.bwd_groups = [sorted(m) for m in groups]
            loads = [sum(cost[a] for a in m) for m in self.bwd_groups]
            self.balance = sum(loads) / len(loads) / max(loads)
        # dW units: (path, first w tile, end w tile, wavefronts along u)
        self.units = []
        for p in self.paths:
            uw = 4 if p.NTU >= 3 else p.NTU
            q = _ceil(p.NTU, uw)
            fixed = words * (q * p.a.D + p.o.D + 9)
            per_w = words * (4 * q + p.o.D)
            step = max(1, min(p.NTW, (self.DW_REGISTERS - fixed) // per_w, 16 // (q * words)))
            step = _ceil(p.NTW, _ceil(p.NTW, step))
            self.units += [(p, lo, min(p.NTW, lo + step), uw) for lo in range(0, p.NTW, step)]
            self.dw_fits = getattr(self, "dw_fits", True) and fixed + step * per_w <= self.DW_REGISTERS + 24
        # workgroups per unit, by its time on a compute unit: matrix-core cycles plus what a step costs beside them
        cyc = 32 if words == 1 else 64
        load = [uw * (_ceil(p.NTU, uw) * (hi - lo) * p.o.D * cyc + 100) for p, lo, hi, uw in self.units]
        share = [max(1, int(self.DW_WORKGROUPS * l / sum(load))) for l in load]
        for k in sorted(range(len(load)), key=lambda k: -load[k] / share[k])[:max(0, self.DW_WORKGROUPS - sum(share))]:
            share[k] = min(self.DW_WORKGROUPS, share[k] + 1)
        self.chunks = share
        self.unit_off, pos = [], self.PART_OFF
        for (p, lo, hi, _), ch in zip(self.units, share):
            self.unit_off.append(pos)
            pos += ch * p.mu * self._width(p, lo, hi)
        assert pos <= self.ws_elems, "the partial rows of few workgroups per path outgrow those of all paths"

    @classmethod
    def row_limits(cls, g: UVWGenerator):
        """Largest batch (forward, backward) these kernels take from ``g``'s.

        Forward: none where the longest work item is not cut here (fp64, 500 rows: 97 -> 13 channels l <= 2 25 against 32 us, 100
        -> 30 channels 43 / 48, 32 channels 15 / 17).  fp64 otherwise 64 channels 2000 rows 47 -> 34, 4097 rows 50 -> 53.  fp32
        where that item is halved: 64 channels 8192 rows 50 -> 42 us, 65 536 rows 194 -> 234; where it loses less, the further
        wavefronts cost as much from the size on at which they no longer have a SIMD each: 4096 / 5120 rows, 100 channels l <=
        1 21 -> 19 / 22 -> 26, 128 channels l <= 2 48 -> 42 / 50 -> 59.  Up to 16 channels likewise, a path is one batch of K
        steps with as much work around it, which every cut item repeats: 16 -> 100 channels 4096 / 8192 rows 19 -> 18 / 27 -> 29.

        Backward, where a block is read by several paths, each of which fetches it here (64 channels, 3.9 times): 4097 rows 73
        -> 60 us in fp32 and 118 -> 104 in fp64, 8192 rows 81 -> 84 and 131 -> 149.  Where every block has one path it depends
        on how evenly the blocks load the groups of wavefronts (their balance: mean over largest load), for a full chip waits
        for the slowest.  fp32, second operand 1x0e, general / these kernels, us:

            channels, blocks            balance     8192      20 480      65 536 rows
            64, l <= 1                    0.67     34 / 32    52 / 49    108 / 95
            50, both parities, l <= 2     0.85     76 / 65   147 / 129   512 / 458
            20 -> 64, l <= 2              0.60     41 / 33    64 / 54    153 / 127     (general: two wavefronts of four)
            64, l <= 2                    0.60     48 / 46    79 / 84    223 / 261
            80, l <= 2                    0.60     66 / 62   113 / 124   327 / 385
            64, l <= 3                    0.57     67 / 71   122 / 139   371 / 453     (5120 rows 59 / 58)

        fp64, where the general kernel holds one wavefront per SIMD: 50 channels of both parities 65 536 rows 802 / 620, 80
        channels l <= 2 960 / 685; only where that kernel's four wavefronts have whole tiles and these are uneven 64 channels
        l <= 2 (0.90) 16 384 rows 109 / 111, 65 536 rows 433 / 464, against 64 channels l <= 3 (1.00) 964 / 810."""
        own = cls(g.problem)
        longest = lambda h: max((hi - lo) * sum(p.o.D * p.SU for p in h.paths_into(o.idx)) for o, lo, hi in h.fwd_order)
        if g.fwd_order[0] in own.fwd_order:
            forward = 0
        elif g.itemsize == 8:
            forward = 2048
        else:
            forward = 8192 if longest(own) <= 0.6 * longest(g) and max(p.mu for p in g.paths) > 16 else 4096
        fetched = sum(p.a.dim + p.o.dim for p in g.paths)
        once = sum(g.in1[a].dim for a in g.used_in1) + sum(g.out[o].dim for o in g.used_out)
        muls = [g.in1[a].mul for a in g.used_in1]
        if fetched > 1.25 * once or not own.bwd_lds:
            backward = 5120
        elif g.itemsize == 8:
            backward = 16384 if own.balance < 1 and all(m % 64 == 0 for m in muls) else 65536
        else:
            backward = 65536 if own.balance >= 0.65 or max(muls) <= 48 else 8192 if own.balance >= 0.595 else 5120
        return forward, backward

    @staticmethod
    def _width(p, lo, hi) -> int:
        return min(p.mw, 16 * hi) - 16 * lo

    @classmethod
    def create(cls, problem: TPProblem):
        """The generator, or None where a dW unit does not fit its registers, a kernel's arrays do not fit LDS together or
        no launch would be cut finer."""
        try:
            g = cls(problem)
        except NotImplementedError:
            return None
        return g if g.dw_fits and g.bwd_lds and g.lds_bytes() <= cls.LDS_BYTES else None

    def lds_bytes(self) -> int:
        """LDS of the largest kernel: the backward's dZ tile beside a dY patch per wavefront (1 KB per word of the second
        operand with 16 wavefronts: from 17 words on a tile within BWD_LDS_LIMIT can be too much), or the dW phases."""
        patches = self.backward_threads // 64 * 16 * max(1, self.D2)
        return max(16 * self.bwd_rs + patches, self._phase_elems()) * self.itemsize

    def _phase_elems(self) -> int:
        """What the dW phases of a workgroup hand over to each other, of the largest unit."""
        return max(uw * (self.DW_WAVES // uw // 2) * _ceil(p.NTU, uw) * (hi - lo) * 256 for p, lo, hi, uw in self.units)

    forward_from = None          # the generator whose forward is this set's, in place of its own

    def take_forward(self, g: UVWGenerator) -> None:
        self.forward_from, self.has_forward = g, True
        self.forward_body, self.forward_attr, self.prep_body = g.forward_body, g.forward_attr, g.prep_body

    def forward_attr(self) -> str:
        return " __attribute__((amdgpu_waves_per_eu(2)))"

    def backward_attr(self) -> str:
        return ""

    @property
    def backward_threads(self) -> int:
        return 256 * len(self.bwd_groups)

    @property
    def dw_threads(self) -> int:
        return 64 * self.DW_WAVES

    # ============================================================ backward: dW
    separate_prep = False

    def _emit_packing(self, E: Emitter) -> None:
        """The backward's packed weights, which dW does not read: 64 of every 16 384 elements a workgroup, one wavefront after
        the other.  Whole backward with a launch for them / here, us: 50 channels of both parities, fp64, 500 rows 26.9 / 24.9,
        4097 54.1 / 52.4; 64 channels l <= 2 of either operand, fp32, 500 rows 28.7 / 26.2, 4097 59.3 / 57.2; 20 -> 40 channels, 500
        rows 17.2 / 15.0."""
        waves, blocks = self.DW_WAVES, sum(self.chunks)
        lo, hi = min(p.wa for p in self.paths), self.WA_END
        E("T* __restrict__ wsT = (T*)ws;")
        E(f"for (int q = {lo} + (wv * {blocks} + (int)blockIdx.x) * 64 + lane; q < {hi}; q += {64 * waves * blocks}) {{")
        E.level += 1
        for p in self.paths:
            self._pack_backward_copy(E, p)
        E.level -= 1
        E("}")

    def _live_chunks(self, k: int) -> str:
        """Workgroups of unit k that have rows to walk (the rest leave no partial row)."""
        per = 4 * (self.DW_WAVES // self.units[k][3])
        return f"(int)min((u64){self.chunks[k]}, (n + {per - 1}) / {per})"

    def backward_dw_body(self) -> str:
        E = Emitter()
        PH = lambda uw: self.DW_WAVES // uw
        E("const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;")
        E(f"__shared__ T comb[{max(1, self._phase_elems())}];")
        self._emit_packing(E)
        first = 0
        for k, (p, lo, hi, uw) in enumerate(self.units):
            Q, ph, D = _ceil(p.NTU, uw), PH(uw), p.o.D
            cells = [(q, nt) for q in range(Q) for nt in range(lo, hi)]
            E(f"{'else ' if k else ''}if (blockIdx.x < {first + self.chunks[k]}) {{ // path {p.t}, w tiles {lo} .. {hi - 1} of {p.NTW}")
            E.level += 1
            E(f"const int chunk = blockIdx.x - {first}, live = {self._live_chunks(k)};")
            E("if (chunk >= live) return;")
            E(f"const int uwv = wv % {uw}, ph = wv / {uw};")
            for q, nt in cells:
                E(f"V4 acc{q}_{nt} = {{0, 0, 0, 0}};")
            E("#pragma unroll 1")
            E(f"for (u64 s = (u64)(chunk * {ph} + ph); s < (n + 3) / 4; s += (u64)(live * {ph})) {{")
            E.level += 1
            E("const u64 b = 4 * s + g;          // batch row of this lane for both operands")
            E("const bool bv = b < n;")
            E("const u64 bc = bv ? b : n - 1;")
            for f in sorted({p.b.off + j for (_, j) in p.pairs}):
                E(f"T y{f} = Y[bc * {self.D2} + {f}];")
            E(f"const T* __restrict__ Xr = X + bc * {self.D1} + {p.a.off};")
            E(f"const T* __restrict__ Gr = G + bc * {self.D3} + {p.o.off};")
            for q in range(Q):
                uexp = f"16 * (uwv + {uw * q}) + c"
                ucl = uexp if p.mu % (16 * uw) == 0 else f"min({uexp}, {p.mu - 1})"
                E("T " + ", ".join(f"x{q}_{i}" for i in range(p.a.D)) + ";")
                E(f"{{ const T* __restrict__ xp = Xr + ({ucl}) * {p.a.D}; " + " ".join(f"x{q}_{i} = xp[{i}];" for i in range(p.a.D)) + " }")
            for nt in range(lo, hi):
                wexp = f"{16 * nt} + c"
                wcl = wexp if p.mw % 16 == 0 else f"min({wexp}, {p.mw - 1})"
                E("T " + ", ".join(f"g{nt}_{k_}" for k_ in range(D)) + ";")
                E(f"{{ const T* __restrict__ gp = Gr + ({wcl}) * {D}; " + " ".join(f"g{nt}_{k_} = gp[{k_}];" for k_ in range(D)) + " }")
            E("if (!bv) { " + " ".join(f"y{f} = (T)0;" for f in sorted({p.b.off + j for (_, j) in p.pairs})) + " }     // rows past the end: T = 0 there")
            for q in range(Q):
                if p.mu % (16 * uw) != 0:
                    E(f"if (16 * (uwv + {uw * q}) + c >= {p.mu}) {{ " + " ".join(f"x{q}_{i} = (T)0;" for i in range(p.a.D)) + " }")
                E("{")
                E.level += 1
                self.emit_cg_forward(E, p, f"x{q}_", "y", "t")
                for nt in range(lo, hi):
                    for k_ in range(D):
                        E(f"acc{q}_{nt} = oeq_mfma(t{k_}, g{nt}_{k_}, acc{q}_{nt});")
                E.level -= 1
                E("}")
            E.level -= 1
            E("}")
            # phases of the batch, summed pairwise in a fixed order
            half = ph // 2
            while half >= 1:
                E(f"if (ph >= {half} && ph < {2 * half}) {{ T* __restrict__ d_ = comb + ((ph - {half}) * {uw} + uwv) * {len(cells) * 256} + lane;")
                for i, (q, nt) in enumerate(cells):
                    E("    " + " ".join(f"d_[{256 * i + 64 * r}] = acc{q}_{nt}[{r}];" for r in range(4)))
                E("}")
                E("oeq_block_sync();")
                E(f"if (ph < {half}) {{ const T* __restrict__ d_ = comb + (ph * {uw} + uwv) * {len(cells) * 256} + lane;")
                for i, (q, nt) in enumerate(cells):
                    E("    " + " ".join(f"acc{q}_{nt}[{r}] += d_[{256 * i + 64 * r}];" for r in range(4)))
                E("}")
                if half > 1:
                    E("oeq_block_sync();")
                half //= 2
            width = self._width(p, lo, hi)
            E(f"if (ph == 0) {{ T* __restrict__ part = (T*)ws + {self.unit_off[k]} + (u64)chunk * {p.mu * width};")
            for q, nt in cells:
                for r in range(4):
                    E(f"    {{ const int u = 16 * (uwv + {uw * q}) + {self.row(r)}; const int w = {16 * (nt - lo)} + c;")
                    E(f"      if (u < {p.mu} && w < {width}) part[u * {width} + w] = acc{q}_{nt}[{r}]; }}")
            E("}")
            E.level -= 1
            E("}")
            first += self.chunks[k]
        return E.text()

    def reduce_body(self) -> str:
        E = Emitter()
        # 64 weights a workgroup, its four wavefronts take every fourth partial row
        E("const int q = blockIdx.x * 64 + (threadIdx.x & 63), sl = threadIdx.x >> 6;")
        E("__shared__ T sums[192];")
        E("const T* __restrict__ part = (const T*)ws;")
        E("int live = 0, size = 0, dst = 0;")
        pos = 0
        for k, (p, lo, hi, _) in enumerate(self.units):
            width = self._width(p, lo, hi)
            size = p.mu * width
            E(f"{'else ' if k else ''}if (q < {pos + size}) {{ const int e = q - {pos}; const int u = e / {width}; const int w = {16 * lo} + e - u * {width};")
            E(f"    live = {self._live_chunks(k)}; size = {size}; part += {self.unit_off[k]} + e; dst = {self.oeq_index(p, 'u', 'w')}; }}")
            pos += size
        E("T acc = (T)0;")
        E("for (int b = sl; b < live; b += 4) acc += part[(u64)b * size];")
        E("if (sl > 0) sums[(sl - 1) * 64 + (threadIdx.x & 63)] = acc;")
        E("oeq_block_sync();")
        E(f"if (sl == 0 && q < {pos}) Wg[dst] = ((acc + sums[threadIdx.x]) + sums[64 + threadIdx.x]) + sums[128 + threadIdx.x];")
        return E.text()

    def plan(self):
        fwd, bwd, ws = super().plan()
        _, dx, dw, reduce = bwd
        dw["num_blocks"] = sum(self.chunks)
        reduce["num_blocks"] = _ceil(self.WN, 64)
        if self.forward_from is not None:
            fwd = self.forward_from.plan()[0]
        return fwd, [dw, dx, reduce], ws               # (dW packs the weights that dX reads)
