"""uvu batch product with one weight vector for all rows (``shared_weights=True``).

The forward is the register-direct kernel of ``uvu_direct.py`` with the weight row fixed.  The backward differs from it
in dW, a sum over the whole batch: a wavefront walks many rows with its channels' weights and dW sums in registers, the
wavefronts of a workgroup add their sums through LDS, and every workgroup leaves one partial row of dW that
``backward_reduce`` adds up in a fixed order (reproducible; the reference accumulates shared weights with racy adds).

What bounds it is HBM: X, Y and dZ in, dX and dY out.  The LDS-staged schedule of ``uvu.py`` (loads through LDS, a fence
per block, one wavefront per SIMD) ran 64 channels, 11 paths, 30 001 rows in 608 us (+ 39 us for a reduction whose
threads each added 1024 partial rows one after the other, + 71 us forward); this one: the backward takes
91 us (4.5 TB/s), the reduction 4 us and the forward 62 us (5.5 TB/s; a large copy moves 4.7, an add 5.9 TB/s).

Multiplicities above 64 take one wavefront per 64-channel chunk of a row, all in one workgroup, which adds the chunks'
dY through LDS once per tile of rows.  Problems with a run-time loop over the copies of the second operand (more than 8)
keep the schedule of ``uvu.py``: their dW sums do not fit registers.  The row's own X, dZ and dX come on top of what the
rule counts, so long rows spill: 128 channels l <= 4, 42 paths, 2.7 KB per lane, 256 channels l <= 3 in fp64 1.4 KB.  The
staged schedule spills more there and is slower at every size tried: backward of 19 531 rows 15.5 -> 4.5 ms, of 15 258
rows 14.8 -> 3.3 ms.
"""
from __future__ import annotations

from ..problem import TPProblem
from .common import WAVE, Emitter, jinja_env
from .uvu_direct import UVUDirectGenerator


class UVUSharedGenerator(UVUDirectGenerator):
    _allow_shared = True
    MAX_WORKGROUPS = None     # workgroups of the largest launch (= partial rows of dW); None: by the rule below
    FOLD_PATHS = 8            # dW sums of a workgroup's wavefronts are added through LDS this many paths at a time
    TILE_ROWS = 4             # rows per wavefront between two barriers when several wavefronts share a row
    # registers (32-bit) of dW sums and weights a wavefront may hold across its rows
    HELD_REGISTERS = 128
    LDS_BYTES = 160 * 1024    # of a compute unit: what the backward's arrays together may take (see lds_bytes)

    @classmethod
    def suits(cls, problem: TPProblem) -> bool:
        """A channel's dW sums and weights leave room in the registers (a long row may spill beside them, which still is the
        faster schedule), and a row's chunks fit one workgroup and its LDS."""
        muls = [problem.irreps_in2[i.i_in2].mul for i in problem.instructions]
        words = 2 * sum(muls) * (2 if problem.irrep_dtype().itemsize == 8 else 1)
        widest = max(mul for mul, _ in list(problem.irreps_in1) + list(problem.irreps_out))
        return (max(muls) <= 8 and words <= cls.HELD_REGISTERS and widest <= 16 * WAVE
                and cls(problem).lds_bytes() <= cls.LDS_BYTES)

    def __init__(self, problem: TPProblem, vector_stores: bool = True):
        super().__init__(problem, "tp", vector_stores=vector_stores)
        assert self.shared and not self.NLY
        self.slots = max(1, 4 // self.NCH)            # rows (R > 1: groups of R rows) in flight per workgroup
        self.waves = self.slots * self.NCH
        self.rows_per_block = self.R * self.slots * (self.TILE_ROWS if self.NCH > 1 else 1)
        # Measured backward in us at 256 / 512 / 768 / 1024 workgroups, 30 000 rows, l <= 2, 11 paths: 64 channels fp32
        # 94 / 91 / 96 / 98, 128 channels 153 / 154 / 161 / 161, 37 channels (27 of 64 lanes idle) 99 / 67 / 56 / 68,
        # 64 channels fp64 211 / 236 / 236 / 242; 2000 rows 9.9 at each
        full = all(self.full(b) for b in self.in1 + self.out if b.dim)
        self.max_workgroups = self.MAX_WORKGROUPS or (256 if self.T == "double" else 512 if full else 768)
        self.bwd_slot = any(self.dx_through_slot(self.in1[i]) for i in self.used_in1)

    def lds_bytes(self) -> int:
        """LDS of the backward: the wavefronts' dX slots, the chunks' dY (which a row of 1024 channels in fp64 fills with 160
        words of the second operand, used or not) and the fold of the dW sums."""
        elems = self.waves * self.lds_elems if self.bwd_slot else 0
        if self.NCH > 1:
            elems += 2 * self.slots * self.TILE_ROWS * self.NCH * self.D2
        if self.slots > 1:
            elems += min(self.FOLD_PATHS, sum(p.mv for p in self.paths)) * self.waves * WAVE
        return elems * self.itemsize

    def describe(self) -> str:
        return super().describe() + " shared weights"

    def render(self, prelude: str = None) -> str:
        env = jinja_env()
        if prelude is None:
            prelude = env.get_template("prelude.hip.jinja").render(T=self.T)
        return env.get_template("tp_uvu_shared.hip.jinja").render(g=self, prelude=prelude)

    def plan(self):
        ROW, FIXED = 1, 0
        fwd = [dict(kernel="forward", num_threads=64, grid_kind=ROW, work_per_block=self.R)]
        bwd = [dict(kernel="backward", num_threads=64 * self.waves, grid_kind=ROW, work_per_block=self.rows_per_block,
                    num_blocks=self.max_workgroups),
               dict(kernel="backward_reduce", num_threads=1024, grid_kind=FIXED, num_blocks=(self.WN + 15) // 16)]
        return fwd, bwd, (lambda nnz=0, nodes=0: self.max_workgroups * self.WN * self.itemsize)

    # =================================================================== backward
    def tp_backward_body(self) -> str:
        E = Emitter()
        R, P, NCH = self.R, self.P, self.NCH
        self.nt_load, self.nt_store = False, "bs" in self._nt_modes
        E("const int lane = threadIdx.x & 63, wv = (int)oeq_uniform_u64((u64)(threadIdx.x >> 6));")
        E(f"const int sub = lane >> {self.LOGP}, ul = lane & {P - 1};")
        E(f"const int c = wv % {NCH}, slot = wv / {NCH}, u = c * {P} + ul; (void)slot;" if NCH > 1
          else "const int c = 0, u = ul; (void)c;")
        if self.bwd_slot:
            E(f"__shared__ __attribute__((aligned(16))) T lds_all[{self.waves * self.lds_elems}];")
            E(f"T* __restrict__ lds = lds_all + wv * {self.lds_elems};")
        self._cur_c = "c"
        self._lazy = False
        self.emit_weight_preload(E, "c", wptr="W")
        self.nt_load = "bl" in self._nt_modes
        for p in self.paths:
            E("T " + ", ".join(f"dws{p.t}_{v} = (T)0" for v in range(p.mv)) + ";")
        if NCH == 1:
            E(f"const u64 items = (n + {R - 1}) / {R};")
            E(f"for (u64 it = (u64)blockIdx.x * {self.waves} + wv; it < items; it += (u64)gridDim.x * {self.waves}) {{")
            E.level += 1
            if self.uniform_rows:
                E("const u64 row = it;")
            else:
                E(f"const u64 row_ = it * {R} + sub;")
                E("const bool rv = row_ < n;")
                E("const u64 row = rv ? row_ : n - 1;         // lanes past the batch repeat its last row, without adding to dW")
            self._row(E)
            E(f"if ({'lane == 63' if P == WAVE else 'ul == 0'}) {{")
            E(f"    T* __restrict__ Ygr = Yg + row * {self.D2};")
            for f in range(self.D2):
                E(f"    Ygr[{f}] = " + (f"dy{f};" if f in self.used_y else "(T)0;"))
            E("}")
            E.level -= 1
            E("}")
        else:
            # the wavefronts of a row's chunks leave their dY in LDS; two buffers, so one barrier per tile
            S, K = self.slots, self.TILE_ROWS
            E(f"__shared__ T ybuf[{2 * S * K * NCH * self.D2}];")
            E("int parity = 0;")
            E(f"for (u64 tile = blockIdx.x; tile * {S * K} < n; tile += gridDim.x, parity ^= 1) {{")
            E.level += 1
            E(f"T* __restrict__ yb = ybuf + parity * {S * K * NCH * self.D2};")
            E("#pragma unroll 1")
            E(f"for (int k_ = 0; k_ < {K}; ++k_) {{")
            E.level += 1
            E(f"const u64 row = tile * {S * K} + (u64)(slot * {K} + k_);")
            E("if (row >= n) break;")
            self._row(E)
            E("if (lane == 63) {")
            E(f"    T* __restrict__ yr = yb + ((slot * {K} + k_) * {NCH} + c) * {self.D2};")
            for f in range(self.D2):
                E(f"    yr[{f}] = " + (f"dy{f};" if f in self.used_y else "(T)0;"))
            E("}")
            E.level -= 1
            E("}")
            E("oeq_block_sync();")
            E(f"for (int q = threadIdx.x; q < {S * K * self.D2}; q += {64 * self.waves}) {{")
            E(f"    const int r = q / {self.D2}, f = q - r * {self.D2};")
            E(f"    const u64 row = tile * {S * K} + r;")
            E(f"    if (row < n) {{ const T* __restrict__ yr = yb + r * {NCH * self.D2} + f; T s = yr[0];")
            E(f"        for (int k = 1; k < {NCH}; ++k) s += yr[k * {self.D2}];")
            E(f"        Yg[row * {self.D2} + f] = s; }}")
            E("}")
            E.level -= 1
            E("}")
        # dW: the lane groups of a wavefront, then the wavefronts of the workgroup that hold the same chunk
        sums = [(p, v) for p in self.paths for v in range(p.mv)]
        m = 32
        while m >= P:
            for p, v in sums:
                E(f"dws{p.t}_{v} += oeq_shfl_xor(dws{p.t}_{v}, {m});")
            m //= 2
        E(f"T* __restrict__ part = (T*)ws + (u64)blockIdx.x * {self.WN};")
        guard = lambda p: f"if (sub == 0 && u < {p.mu}) "
        if self.slots == 1:
            for p, v in sums:
                E(f"{guard(p)}part[{self.widx(p, 'u', v)}] = dws{p.t}_{v};")
            return E.text()
        F = min(self.FOLD_PATHS, len(sums))
        E(f"__shared__ T fold[{F * self.waves * WAVE}];")
        for b in range(0, len(sums), F):
            grp = sums[b:b + F]
            if b:
                E("oeq_block_sync();")
            for i, (p, v) in enumerate(grp):
                E(f"fold[{i * self.waves * WAVE} + threadIdx.x] = dws{p.t}_{v};")
            E("oeq_block_sync();")
            for i, (p, v) in enumerate(grp):
                # the wavefront of slot i % slots adds this path's sums (the chunk is the wavefront's own)
                own = f"wv == {i % self.slots}" if NCH == 1 else f"slot == {i % self.slots}"
                terms = " + ".join(f"fold[{i * self.waves * WAVE} + ({s * NCH} + c) * 64 + lane]" for s in range(self.slots))
                E(f"if ({own}) {{ const T s_ = {terms}; {guard(p)}part[{self.widx(p, 'u', v)}] = s_; }}")
        return E.text()

    def _row(self, E: Emitter) -> None:
        """One row of the wavefront's chunk: dX written, dy left in registers, dW sums added to."""
        E(f"const T* __restrict__ Yr = Y + row * {self.D2};")
        self.emit_y_load_direct(E)
        self.emit_x_preload(E, "c", "row")
        for oi in self.used_out:
            o = self.out[oi]
            self.emit_record_load(E, [f"G{oi}_{k}" for k in range(o.D)],
                                  f"G + (u64)row * {self.D3} + {o.off} + {self.uclamp(o, 'c')} * {o.D}", self.act(o), zero=True)
        self.emit_x_alias(E, "c")
        for f in self.used_y:
            E(f"T dy{f} = (T)0;")
        for i in self.used_in1:
            E("T " + ", ".join(f"dx{i}_{m} = (T)0" for m in range(self.in1[i].D)) + ";")
        for oi in self.used_out:
            o = self.out[oi]
            E("{")
            E.level += 1
            for k in range(o.D):
                E(f"const T g{k} = G{oi}_{k};")

            def sink(E, p, v, expr):
                E(f"  dws{p.t}_{v} += {expr};" if self.uniform_rows else f"  dws{p.t}_{v} += rv ? {expr} : (T)0;")
            self.emit_backward_block(E, o, "W", sink)
            E.level -= 1
            E("}")
        row_of = (lambda r: ("row", "true")) if self.R == 1 else (lambda r: (f"min(it * {self.R} + {r}, n - 1)", "true"))
        for a in self.in1:
            if a.dim == 0:
                continue
            if a.idx in self.used_in1:
                self.emit_block_store(E, a, [f"dx{a.idx}_{m}" for m in range(a.D)], "Xg", self.D1, "row", row_of, "store",
                                      via_lds=self.dx_through_slot(a))
            else:
                self.emit_record_store(E, ["(T)0"] * a.D, f"Xg + (u64)row * {self.D1} + {a.off} + u * {a.D}", self.act(a))
        if self.P == WAVE:
            for f in self.used_y:
                E(f"dy{f} = oeq_wave_sum63(dy{f});")
        else:
            self.emit_dy_reduce(E)

    def reduce_body(self) -> str:
        """dW = sum of the workgroups' partial rows: 16 weights per workgroup, 64 threads per weight take every 64th
        row, then the 64 sums are added in a fixed order."""
        E = Emitter()
        E("__shared__ T red[16 * 16];")
        E("const int q = blockIdx.x * 16 + (threadIdx.x & 15), wv = threadIdx.x >> 6;")
        E(f"const u64 want = (n + {self.rows_per_block - 1}) / {self.rows_per_block};")
        E(f"const int parts = (int)(want < {self.max_workgroups} ? want : {self.max_workgroups});     // workgroups of the backward launch")
        E(f"const T* __restrict__ p_ = (const T*)ws + min(q, {self.WN - 1});")
        E("T acc = (T)0;")
        E("#pragma unroll 4")
        E(f"for (int b = threadIdx.x >> 4; b < parts; b += 64) acc += p_[(u64)b * {self.WN}];")
        E("acc += oeq_shfl_xor(acc, 16);")
        E("acc += oeq_shfl_xor(acc, 32);")
        E("if ((threadIdx.x & 63) < 16) red[wv * 16 + (threadIdx.x & 15)] = acc;")
        E("oeq_block_sync();")
        E(f"if (threadIdx.x < 16 && q < {self.WN}) {{")
        E("    T s = (T)0;")
        E("    for (int w = 0; w < 16; ++w) s += red[w * 16 + threadIdx.x];")
        E("    Wg[q] = s;")
        E("}")
        return E.text()
