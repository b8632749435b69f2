"""uvw tensor products with per-row weights (``shared_weights=False``), e.g. the DiffDock layers
of the reference's benchmark set (openequivariance/benchmark/benchmark_configs.py:44-48).

    Z[b, w, k] = sum_t sum_u  W[b, t, u, w] * T_t[b, u, k]

With a separate weight matrix per row there is no operand reuse across the batch: the op is a
batched matrix-vector product that streams ``weight_numel`` words per row and is bound by HBM,
so it runs on the vector ALU, one wavefront per row (reference: loop_unroll_tp.cuh:56-78 streams
the same weights through shared memory into a CUDA-core matmul).  Both kernels read and write the
weights in the order they lie in memory - the external order keeps each 32 x 32 chunk [u][w] of a
path contiguous - so that a wavefront's access is one 256- or 512-byte run:

* forward: as for the backward, the weights pass through LDS in batches of 16-byte pieces where a row divides into such
  (forward_stream_body).  Otherwise lanes <-> channel u compute T_t[u, :] of every path into a group of output blocks and
  park it in LDS; then lanes <-> (output channel w, a slice of u) walk the chunks with the loads a
  fixed number of steps ahead of the multiplies, branch-free, T read from LDS; the slices are
  summed with lane exchanges at the end of an output block;
* backward: the weights go global -> registers -> LDS, lanes <-> (u, a slice of w) then read their row of a
  chunk, form dT (-> dX, dY through the CG transpose) against dZ in LDS and put dW = T (x) dZ back into
  the same LDS words, which leave in memory order again.  A row's weights pass in batches of whole chunks, 16 bytes
  per lane (backward_stream_body), or, where they do not divide into such, chunk by chunk.

The external (oeq) weight order is addressed in place by index arithmetic.
"""
from __future__ import annotations

import math

from ..problem import TPProblem
from .common import Emitter, jinja_env
from .uvw import UVWGenerator, _ceil


class UVWBatchedGenerator(UVWGenerator):
    _allow_batched = True

    def __init__(self, problem: TPProblem, pairs: bool = True, stream: bool = True):
        """``pairs``: fp32 weights move two words per lane where a chunk's offset and width are even (an 8-byte
        access sustains more of the HBM rate than a 4-byte one); needs W and dW at 8-byte aligned addresses.
        ``stream``: the backward's weights move in batches of 16 bytes per lane where a row divides into such; needs
        W and dW at 16-byte aligned addresses."""
        super().__init__(problem)
        self.pairs = bool(pairs) and self.T == "float" and self.WN % 2 == 0
        if self.shared:
            raise ValueError("UVWBatchedGenerator is for per-row weights")
        self.kind = "uvw_batched"
        self.t_lds = max([sum(p.mu * o.D for o in ph for p in self.paths_into(o.idx)) for ph in self.forward_phases()] + [0])
        self.ws_elems = 0
        self.batches = self._batches() if stream else None
        self.stream_forward = self.batches is not None and not self._first_operand_too_wide(forward=True)
        # the backward keeps its other walk where chunks are long and whole lines: 32 channels, 20 000 rows 112 us against 116.5, 48
        # channels 160 against 163, fp64, 24 channels, 6000 rows 117 against 120 (16 channels, chunks of 256 words: 81.9 / 79.8)
        self.stream_backward = self.batches is not None and self.WN <= self.STREAM_ROW[self.T] and not (
            self.WN >= 400 * sum(map(len, self.batches)) and all(
                ul * wl * self.itemsize % 128 == 0 for b in self.batches for _, _, ul, _, wl, _ in b)
        ) and not self._first_operand_too_wide(forward=False)
        self.stream = self.stream_forward or self.stream_backward
        self.rows_chunked = 0
        if self.stream_forward and self.WN * self.itemsize >= self.ROWS_CHUNKED_FROM:
            self.rows_chunked = next(rows for most, rows in self.ROWS_CHUNKED if self.WN * self.itemsize <= most)
        self.has_backward = True

    # Rows up to which the forward keeps the walk over chunks, as a kernel for few rows: a wavefront per SIMD, with nothing beside it to
    # hide a batch's way through LDS; half of them where a row is longer than 64 KB, none where the walk spills or a row is a batch or two.
    # Chunks / batches, us, 256, 1024 and 2048 rows: DiffDock's layer (28 KB) 5.0 / 5.9, 7.0 / 7.8 and 10.6 / 10.5, fp64 5.8 / 7.0,
    # 10.7 / 10.9 and 19.9 / 19.0; 10 channels to 50, l <= 2, 5.7 / 7.3, 7.5 / 8.7 and 10.7 / 10.3, fp64 5.5 / 8.8, 10.1 / 11.3 and 19.9 /
    # 17.6; 60 of both parities to 26, l <= 1, 6.5 / 10.5, 11.5 / 15.0 and 20.8 / 21.6.  256, 512 and 1024 rows: 80 channels to 34, l <= 2
    # (74 KB) 10.9 / 12.7, 12.1 / 16.4 and 17.0 / 19.8, 128 of both parities to 20, l <= 1 (100 KB) 11.1 / 17.8, 13.4 / 22.0 and 20.2 / 25.9, 34 to 100,
    # fp64 (106 KB) 7.0 / 11.0, 10.4 / 13.3 and 18.9 / 18.5, 128 to 18, fp64 (72 KB) 8.5 / 9.2, 10.2 / 11.4 and 15.3 / 13.9.
    # Below 16 KB, 34 channels, one scalar, 256, 1024 and 2048 rows 5.1 / 4.5, 6.4 / 5.9, 9.0 / 7.9.
    ROWS_CHUNKED_FROM, ROWS_CHUNKED = 16 << 10, ((64 << 10, 1024), (128 << 10, 512), (1 << 62, 0))

    def forward_of_few_rows(self) -> "UVWBatchedGenerator":
        few = UVWBatchedGenerator(self.problem, stream=False)
        few.has_backward = False
        return few

    # 32-bit words a lane holds of the first operand over a whole row, which the walks over chunks read block by block: in the forward
    # X (and few sums Z beside it: a narrow output), in the backward X and dX.  Beyond these the batches lose their wavefronts, then
    # their registers.  512 channels to 4, l <= 2, chunks / batches, us, 600 rows and 420 MB of weights: forward, fp32 (72 words) 15.1 /
    # 15.9 and 69 / 89, fp64 (144) 22.9 / 26.9 and 75 / 90; backward, fp32 (288) 41 / 26 and 146 / 154, fp64 (576) 56 / 84 and 154 / 289;
    # 2000x1o to 4, fp32 (378) 49 / 28 and 138 / 146, fp64 (756) 65 / 80 and 134 / 276.  256 channels, fp64: forward (72) 10.1 /
    # 9.9 and 60 / 62, backward (288) 30 / 21 and 141 / 135.
    FORWARD_WORDS, BACKWARD_WORDS = 64, 400

    def _first_operand_too_wide(self, forward: bool) -> bool:
        def held(blocks, lanes):
            return sum(_ceil(b.mul, lanes) * b.D for b in blocks if b.dim) * self.itemsize // 4
        if forward:
            return held(self.in1, 64) > max(self.FORWARD_WORDS, 4 * held(self.out, 32))
        return 2 * held(self.in1, 32) > self.BACKWARD_WORDS

    # Words of a row up to which the backward's weights move in batches.  A long row of few is bound by what one wavefront has in
    # flight, and the other walk has four chunks: fp32, batches / chunks, us, 46 channels, l <= 2 (23 276 words) 859 rows 41 / 44,
    # 6444 rows 264 / 278; 52 (29 744) 672 rows 55 / 47, 5043 rows 249 / 257; 100 (110 000) 500 rows 142 / 108, 1363 rows 256 / 271.
    # fp64, where that walk has two, does not lose: 38 880 words, 500 rows 82 / 83, 1929 rows 244 / 248.
    STREAM_ROW = {"float": 25000, "double": 1 << 62}
    STREAM_UNROLL = 4             # steps of a chunk's loop in flight in the forward
    STREAM_BYTES = 4096           # of a batch at most (a chunk of 32 x 32 words; 8192 in fp64)

    def _batches(self):
        """The row's weight chunks in the order they lie in memory, as batches of whole chunks that begin and end at multiples of
        16 bytes: [[(path, uc, ul, wc, wl, offset), ..], ..]; None where the row does not divide into such."""
        vw, most = 16 // self.itemsize, max(self.STREAM_BYTES, 1024 * self.itemsize) // self.itemsize
        jobs = sorted(((p, uc, ul, wc, wl, self.chunk_base(p, uc, wc)) for p in self.paths for uc, ul in self.chunks(p.mu)
                       for wc, wl in self.chunks(p.mw)), key=lambda job: job[-1])
        batches, begin, end = [], 0, 0
        todo = []                                    # chunks since the last multiple of 16 bytes
        for job in jobs:
            if job[-1] != end:
                return None
            end += job[2] * job[4]
            todo.append(job)
            if end % vw == 0:
                if not batches or end - begin > most:
                    begin = todo[0][-1]
                    batches.append([])
                batches[-1] += todo
                todo = []
                if end - begin > most:
                    return None
        if todo or end != self.WN or not batches:
            return None
        return batches

    def describe(self) -> str:
        return (f"uvw per-row weights T={self.T} paths={len(self.paths)} d1={self.D1} d2={self.D2} d3={self.D3} "
                f"wn={self.WN} (vector ALU, HBM bound)")

    def ld2(self, ptr: str) -> str:
        return f"oeq_ldnt2({ptr})" if self.NONTEMPORAL else f"*(const V2*)({ptr})"

    def st2(self, ptr: str, val: str) -> str:
        return f"oeq_stnt2({ptr}, {val});" if self.NONTEMPORAL else f"*(V2*)({ptr}) = {val};"

    def ld(self, ptr: str) -> str:
        return f"oeq_ldnt({ptr})" if self.NONTEMPORAL else f"*({ptr})"

    def st(self, ptr: str, val: str) -> str:
        return f"oeq_stnt({ptr}, {val});" if self.NONTEMPORAL else f"*({ptr}) = {val};"

    # ------------------------------------------------------------ weight order
    @staticmethod
    def chunks(mul: int):
        """(chunk number, width) of the 32-wide pieces of a multiplicity, as the external weight
        order cuts it (weight_order.py)."""
        return [(c, min(32, mul - 32 * c)) for c in range(_ceil(mul, 32))]

    def chunk_base(self, p, uc: int, wc: int) -> int:
        """Offset of the [u_local][w_local] slice (contiguous, ul * wl words) that holds chunk
        (uc, wc) of path ``p``'s copy of the second operand."""
        mu, mv, mw = p.mu, p.mv, p.mw
        vc, vl = divmod(p.v, 32)
        vlw = min(32, mv - 32 * vc)
        ul, wl = min(32, mu - 32 * uc), min(32, mw - 32 * wc)
        base = p.woff + uc * 32 * mv * mw + ul * (32 * vc * mw + vlw * (32 * wc) + vl * wl)
        assert base == eval(self.oeq_index(p, str(32 * uc), str(32 * wc)), {"min": min})
        return base

    @staticmethod
    def _split(width: int):
        """Lanes <-> (position in a chunk of ``width`` <= 32, slice): the power of two the positions
        are padded to, its log2, and the number of slices."""
        lp = 1
        while lp < width:
            lp *= 2
        return lp, lp.bit_length() - 1, 64 // lp

    # ----------------------------------------------------------------- forward
    FORWARD_AHEAD = 16    # weight loads in flight ahead of the one being multiplied
    T_LDS_WORDS = 4096    # T of the paths into the output blocks of one phase stays below this many words

    def forward_phases(self):
        """Output blocks grouped so that T of every path into a group fits the LDS budget together: a phase
        computes all its T first and then streams its weights as one pipeline."""
        phases, words = [[]], 0
        for o in self.out:
            if o.dim == 0:
                continue
            w = sum(p.mu * o.D for p in self.paths_into(o.idx))
            if phases[-1] and words + w > self.T_LDS_WORDS:
                phases.append([])
                words = 0
            phases[-1].append(o)
            words += w
        return [ph for ph in phases if ph]

    def forward_body(self) -> str:
        if self.stream_forward:
            return self.forward_stream_body()
        E = Emitter()
        E("const int lane = threadIdx.x;")
        E("const u64 row = blockIdx.x;")
        E("if (row >= n) return;")
        E(f"__shared__ T tl[{max(1, self.t_lds)}];")
        E(f"const T* __restrict__ Xr = X + row * {self.D1};")
        E(f"const T* __restrict__ Wr = W + row * {self.WN};")
        for f in self.used_y:
            E(f"const T y{f} = Y[row * {self.D2} + {f}];")
        for phase in self.forward_phases():
            # lanes <-> (V adjacent channels, a slice of u) within a chunk of output channels.  Lanes past the
            # chunk's width repeat its last columns: what they add up is never stored and never meets the other
            # lanes (the reduction over the slices keeps wq).  One step = one access of every lane: row
            # us + ns * j of a [ul][wl] slice; the last step of a slice whose rows do not divide re-reads the
            # last row with T = 0.
            toff, acc, groups, steps, lanes = {}, 0, [], [], []
            for o in phase:
                wcs = self.chunks(o.mul)
                into = self.paths_into(o.idx)
                width = {wc: 2 if self.pairs and wl % 2 == 0 and all(
                             self.chunk_base(p, uc, wc) % 2 == 0 for p in into for uc, _ in self.chunks(p.mu)) else 1
                         for wc, wl in wcs}
                for wc, wl in wcs:
                    lp, lg, _ = self._split(wl // width[wc])
                    lanes.append(f"const int wq{o.idx}_{wc} = min(lane & {lp - 1}, {wl // width[wc] - 1}), "
                                 f"us{o.idx}_{wc} = lane >> {lg};")
                for p in into:
                    toff[p.t] = acc
                    acc += p.mu * o.D
                per = max(1, 40 // (o.D * max(width.values())))
                for g0 in range(0, len(wcs), per):
                    grp = wcs[g0:g0 + per]
                    groups.append(dict(o=o, grp=grp, width=width, first=len(steps)))
                    for p in into:
                        for wc, wl in grp:
                            V = width[wc]
                            _, _, ns = self._split(wl // V)
                            for uc, ul in self.chunks(p.mu):
                                full, tail = divmod(ul, ns)
                                for j in range(full + (1 if tail else 0)):
                                    r = f"us{o.idx}_{wc} + {ns * j}"
                                    steps.append(dict(V=V, z=f"z{o.idx}_{wc}", wq=f"wq{o.idx}_{wc}", wl=wl, D=o.D,
                                                      base=self.chunk_base(p, uc, wc), t=toff[p.t] + 32 * uc * o.D,
                                                      row=r if j < full else f"min({r}, {ul - 1})",
                                                      ok=None if j < full else f"us{o.idx}_{wc} < {tail}"))
                    groups[-1]["last"] = len(steps)
            assert acc <= max(1, self.t_lds)

            def load(i):
                if i < len(steps):
                    st = steps[i]
                    addr = f"Wr + {st['base']} + {st['V']} * {st['wq']} + ({st['row']}) * {st['wl']}"
                    if st["V"] == 2:
                        E(f"const V2 wv{i} = {self.ld2(addr)};")
                    else:
                        E(f"const T wv{i}[1] = {{{self.ld(addr)}}};")

            def multiply(i):
                st = steps[i]
                for k in range(st["D"]):
                    t_ = f"tl[{st['t'] + k} + ({st['row']}) * {st['D']}]"
                    if st["ok"]:
                        t_ = f"({st['ok']}) ? {t_} : (T)0"
                    E(f"{{ const T t_ = {t_}; " + " ".join(
                        f"{st['z']}_{h}_{k} = oeq_fma(wv{i}[{h}], t_, {st['z']}_{h}_{k});" for h in range(st["V"])) + " }")

            E(f"{{ // output blocks {[o.idx for o in phase]}: T of every path into them, then their weights as one stream")
            E.level += 1
            for ln in lanes:
                E(ln)
            for i in range(self.FORWARD_AHEAD):
                load(i)
            paths = [p for o in phase for p in self.paths_into(o.idx)]
            for p in paths:
                for uc in range(_ceil(p.mu, 64)):
                    E(f"const T* __restrict__ xp{p.t}_{uc} = Xr + {p.a.off} + min({64 * uc} + lane, {p.mu - 1}) * {p.a.D};")
                    E("const T " + ", ".join(f"x{p.t}_{uc}_{i} = xp{p.t}_{uc}[{i}]" for i in range(p.a.D)) + ";")
            E("oeq_sync();")
            for p in paths:
                for uc in range(_ceil(p.mu, 64)):
                    E(f"{{ const int u = {64 * uc} + lane;   // path {p.t}")
                    E.level += 1
                    self.emit_cg_forward(E, p, f"x{p.t}_{uc}_", "y", "t")
                    E(f"if (u < {p.mu}) {{ " + " ".join(f"tl[{toff[p.t]} + u * {p.o.D} + {k}] = t{k};" for k in range(p.o.D)) + " }")
                    E.level -= 1
                    E("}")
            E("oeq_sync();")
            for gr in groups:
                o, width = gr["o"], gr["width"]
                E(f"// output block {o.idx}, channels {32 * gr['grp'][0][0]} ..")
                for wc, wl in gr["grp"]:
                    E("T " + ", ".join(f"z{o.idx}_{wc}_{h}_{k} = (T)0" for h in range(width[wc]) for k in range(o.D)) + ";")
                for i in range(gr["first"], gr["last"]):
                    load(i + self.FORWARD_AHEAD)
                    multiply(i)
                for wc, wl in gr["grp"]:
                    V = width[wc]
                    cols = wl // V
                    lp, lg, ns = self._split(cols)
                    z = f"z{o.idx}_{wc}"
                    s = lp
                    while s < 64:
                        E(" ".join(f"{z}_{h}_{k} += oeq_shfl_xor({z}_{h}_{k}, {s});" for h in range(V) for k in range(o.D)))
                        s *= 2
                    E(f"if (lane < {cols}) {{ T* __restrict__ zp = Z + row * {self.D3} + {o.off} + ({32 * wc} + {V} * lane) * {o.D}; "
                      + " ".join(f"zp[{h * o.D + k}] = {z}_{h}_{k};" for h in range(V) for k in range(o.D)) + " }")
            E.level -= 1
            E("}")
        return E.text()

    def _stream_header(self, E: Emitter, words) -> None:
        E("const int lane = threadIdx.x;")
        E("const u64 row = blockIdx.x;")
        E("if (row >= n) return;")
        E(f"__shared__ __attribute__((aligned(16))) T tile[{max(words)}];")
        E(f"const T* __restrict__ Xr = X + row * {self.D1};")
        E(f"const T* __restrict__ Wr = W + row * {self.WN};")

    def _vectors(self, words: int):
        """Positions of a lane's 16-byte pieces of a batch: lanes past its end repeat its last piece."""
        VW = 16 // self.itemsize
        return [f"{64 * VW * i} + {VW} * lane" if 64 * VW * (i + 1) <= words else f"min({64 * VW * i} + {VW} * lane, {words - VW})"
                for i in range(_ceil(words, 64 * VW))]

    def _stream(self, E: Emitter, words, work, store=None) -> None:
        """The row's batches through LDS, the next one in flight in registers while ``work(job, offset in the tile)`` is
        done on the chunks of one; ``store`` takes the tile back to memory."""
        def request(b):
            if b < len(words):
                E(f"// batch {b}: {words[b]} words at {self.batches[b][0][-1]}")
                for i, at in enumerate(self._vectors(words[b])):
                    E(f"const VT b{b}_{i} = oeq_ldnt16(Wr + {self.batches[b][0][-1]} + {at});")
        for b, batch in enumerate(self.batches):
            if b == 0:
                request(0)
                yield
            for i, at in enumerate(self._vectors(words[b])):
                E(f"*(VT*)(tile + {at}) = b{b}_{i};")
            E("oeq_sync();")
            request(b + 1)
            for job in batch:
                work(job, job[-1] - batch[0][-1])
            E("oeq_sync();")
            if store:
                for i, at in enumerate(self._vectors(words[b])):
                    E(f"oeq_stnt16({store} + {batch[0][-1]} + {at}, *(const VT*)(tile + {at}));")
                E("oeq_sync();")

    def forward_stream_body(self) -> str:
        """The forward over the same batches as backward_stream_body: T of a path goes to LDS when its weights come up (lanes <-> u),
        then lanes <-> (output channel, slice of u).  Against lanes that read the weights from memory chunk by chunk: DiffDock's
        layer, 50 000 rows 275 -> 252 us (5.9 TB/s), fp64, 20 000 rows 210 -> 197; 6 channels, 20 000 rows 26.5 -> 17.8, 12 31.7 ->
        26.4, 42, 10 000 rows 67.6 -> 60.2, 48, 4000 rows 65.8 -> 64.0 (eight steps at a time: 70.8), fp64, 2500 rows 141 -> 80
        (that walk spilled); 32 channels, 20 000 rows 53.8 and 54.0.

        Rows of no more than STREAM_UNROLL steps are no loop, and nothing waits for their sums before the row ends: left to itself the
        compiler keeps the operands of every chunk until then.  There a path's sums are taken when the next one begins.  8 channels
        to 36, both parities, l <= 2, 11 574 rows: chunks 89.7 us, sums left 122.6 (479 registers), taken 79.2 (120); fp64, 5787 rows
        93 / 409 (512 and 1972 bytes of scratch) / 81 (218); 4 to 34, fp64, l <= 1 91 / 88 / 85; 8 to 8, fp32 158 / 109 / 108."""
        E = Emitter()
        words = [sum(ul * wl for _, _, ul, _, wl, _ in b) for b in self.batches]
        self._stream_header(E, words)
        E(f"__shared__ T tl[{max(p.mu * p.o.D for p in self.paths)}];")
        for wl in sorted({wl for o in self.out for _, wl in self.chunks(o.mul)}):
            lp, lg, _ = self._split(wl)
            E(f"const int wq{wl} = min(lane & {lp - 1}, {wl - 1}), us{wl} = lane >> {lg};")
        outs = [(o, wc, wl) for o in self.out if o.dim for wc, wl in self.chunks(o.mul)]
        for o, wc, _ in outs:
            E("T " + ", ".join(f"z{o.idx}_{wc}_{k} = (T)0" for k in range(o.D)) + ";")
        held = [(a, h) for a in self.in1 if a.dim for h in range(_ceil(a.mul, 64))]
        now, put_off = [None], {}                     # the path whose T is in LDS; sums that the compiler may still put off

        def work(job, at):
            p, uc, ul, wc, wl, _ = job
            o = p.o
            if now[0] != p.t:
                now[0] = p.t
                self._take(E, put_off)
                E("oeq_sync();")
                for h in range(_ceil(p.mu, 64)):
                    E(f"{{ const int u = {64 * h} + lane;   // T of path {p.t}")
                    E.level += 1
                    self.emit_cg_forward(E, p, f"x{p.a.idx}_{h}_", "y", "t")
                    E(f"if (u < {p.mu}) {{ " + " ".join(f"tl[u * {o.D} + {k}] = t{k};" for k in range(o.D)) + " }")
                    E.level -= 1
                    E("}")
                E("oeq_sync();")
            _, _, ns = self._split(wl)
            full, tail = divmod(ul, ns)
            if full <= self.STREAM_UNROLL:
                put_off.update((f"z{o.idx}_{wc}_{k}", None) for k in range(o.D))
            E(f"{{ // weights [{ul}][{wl}] of path {p.t}")

            def step(u):
                E(f"  const int u_ = {u};")
                E(f"  const T wv = tile[{at} + u_ * {wl} + wq{wl}];")
                for k in range(o.D):
                    E(f"  z{o.idx}_{wc}_{k} = oeq_fma(wv, tl[({32 * uc} + u_) * {o.D} + {k}], z{o.idx}_{wc}_{k});")
            if full:
                E(f"#pragma unroll {self.STREAM_UNROLL}")
                E(f"for (int j = 0; j < {full}; ++j) {{")
                step(f"us{wl} + {ns} * j")
                E("}")
            if tail:
                E(f"if (us{wl} < {tail}) {{")
                step(f"us{wl} + {ns * full}")
                E("}")
            E("}")
        for _ in self._stream(E, words, work):           # (the first batch is on its way)
            for f in self.used_y:
                E(f"const T y{f} = Y[row * {self.D2} + {f}];")
            for a, h in held:
                E(f"const T* __restrict__ xp{a.idx}_{h} = Xr + {a.off} + min({64 * h} + lane, {a.mul - 1}) * {a.D};")
                E("const T " + ", ".join(f"x{a.idx}_{h}_{i} = xp{a.idx}_{h}[{i}]" for i in range(a.D)) + ";")
        for o, wc, wl in outs:
            lp, _, _ = self._split(wl)
            s = lp
            while s < 64:
                E(" ".join(f"z{o.idx}_{wc}_{k} += oeq_shfl_xor(z{o.idx}_{wc}_{k}, {s});" for k in range(o.D)))
                s *= 2
            E(f"if (lane < {wl}) {{ T* __restrict__ zp = Z + row * {self.D3} + {o.off} + ({32 * wc} + lane) * {o.D}; "
              + " ".join(f"zp[{k}] = z{o.idx}_{wc}_{k};" for k in range(o.D)) + " }")
        return E.text()

    # ---------------------------------------------------------------- backward
    # The walk over chunks: chunks whose loads are in flight ahead of the one being worked on, and steps of a chunk's row loop in
    # flight (all 16 at once would take 100 more registers).  fp32 words whose chunks are short or ragged: two of them ahead cover
    # less than a memory latency.  2 and 4 steps / 4 and 8, us, l <= 2, 0.6 GB of weights (20 000 rows at most) and 0.08: 17
    # channels 123 / 118 and 45 / 43, 31 267 / 258 and 42 / 42, 47 287 / 279 and 46 / 44; l <= 1, 17 45.0 / 43.2 and 40 / 38.  Chunks that
    # are 32 x 32 throughout, several to a block, are far enough ahead with two: 64 channels 241 / 254 and 43 / 45, of both parities
    # 254 / 253 and 109 / 119.  fp64, where a word is two registers, gains nothing (DiffDock's layer 465 / 463).
    AHEAD = {"float": (4, 8), "double": (2, 4)}
    AHEAD_WHOLE = 2, 4

    def _chunk_walk(self):
        """((chunks ahead, steps in flight), whether a path's sums are taken when it is done with).  Left to the compiler they go
        to the end of a block of the first operand (see PUT_OFF), which costs registers where its paths are many: fp32, 17 channels of
        both parities, l <= 2, 17 301 rows, 259 registers 486 us, taken 291; fp64, 20 channels to l = 3, 8152 rows 400, 309 and
        244, 48 of both parities, l <= 2, 1085 rows 313 and 272; and where a block is several chunks long: fp32, 80 channels, l <= 2,
        2130 rows 273 / 258, 65 channels 310 / 291.  Few sums are better left: 47 channels of both parities, l <= 1, 266 / 276."""
        muls = [b.mul for b in (*self.in1, *self.out) if b.dim]
        whole = all(m % 32 == 0 for m in muls) and max(muls) > 32
        sums = max(sum(p.o.D for p in self.paths_from(a.idx)) for a in self.in1 if a.dim)
        return self.AHEAD_WHOLE if whole else self.AHEAD[self.T], sums >= 20 or max(muls) > 64

    NONTEMPORAL = True    # the weights and their gradient are touched once
    def backward_body(self) -> str:
        if self.stream_backward:
            return self.backward_stream_body()
        E = Emitter()
        E("const int lane = threadIdx.x;")
        E("const u64 row = blockIdx.x;")
        E("if (row >= n) return;")
        E(f"__shared__ T gl[{max(1, self.D3)}];")
        E(f"__shared__ T tile[{32 * 33}];")
        E(f"const T* __restrict__ Xr = X + row * {self.D1};")
        E(f"const T* __restrict__ Wr = W + row * {self.WN};")
        E(f"T* __restrict__ Wgr = Wg + row * {self.WN};")
        # every [ul][wl] weight chunk of the row, in the order it is worked on
        jobs = []
        for a in self.in1:
            if a.dim == 0:
                continue
            for uc, ul in self.chunks(a.mul):
                for p in self.paths_from(a.idx):
                    for wc, wl in self.chunks(p.mw):
                        jobs.append((a.idx, uc, p.t, ul * wl, self.chunk_base(p, uc, wc)))

        def width(job):
            return 2 if self.pairs and job[3] % 2 == 0 and job[4] % 2 == 0 else 1

        def regs(job):
            return width(job) * _ceil(job[3], 64 * width(job))
        (ahead, unroll), take = self._chunk_walk()
        nbuf = ahead + 1
        for b in range(min(nbuf, len(jobs))):
            E(f"T r{b}_[{max(regs(job) for job in jobs[b::nbuf])}];")

        def request(n):
            if n < len(jobs):
                _, _, _, words, base = jobs[n]
                V = width(jobs[n])
                E(f"// chunk {n}: {words} words at {base}")
                for i in range(_ceil(words, 64 * V)):
                    guard = "" if 64 * V * (i + 1) <= words else f"if ({64 * V * i} + {V} * lane < {words}) "
                    if V == 2:
                        E(f"{guard}{{ const V2 v_ = {self.ld2(f'Wr + {base + 128 * i} + 2 * lane')}; "
                          f"r{n % nbuf}_[{2 * i}] = v_[0]; r{n % nbuf}_[{2 * i + 1}] = v_[1]; }}")
                    else:
                        E(f"{guard}r{n % nbuf}_[{i}] = {self.ld(f'Wr + {base + 64 * i} + lane')};")

        for n in range(ahead):
            request(n)
        E(f"for (int q = lane; q < {self.D3}; q += 64) gl[q] = G[row * {self.D3} + q];")
        E("oeq_sync();")
        for f in self.used_y:
            E(f"const T y{f} = Y[row * {self.D2} + {f}];")
            E(f"T dy{f} = (T)0;")
        n = 0
        for a in self.in1:
            if a.dim == 0:
                continue
            for uc, ul in self.chunks(a.mul):
                lp, lg, ns = self._split(ul)
                E(f"{{ // input block {a.idx}, channels {32 * uc} ..")
                E.level += 1
                E(f"const int uq = lane & {lp - 1}, ws = lane >> {lg};")
                E(f"const bool act = uq < {ul};")
                E(f"const int ur = min(uq, {ul - 1});")
                E(f"const T* __restrict__ xp = Xr + {a.off} + ({32 * uc} + ur) * {a.D};")
                E("const T " + ", ".join(f"x{i} = xp[{i}]" for i in range(a.D)) + ";")
                E("T " + ", ".join(f"dx{i} = (T)0" for i in range(a.D)) + ";")
                for p in self.paths_from(a.idx):
                    o = p.o
                    E(f"{{ // path {p.t}")
                    E.level += 1
                    self.emit_cg_forward(E, p, "x", "y", "t")
                    E("T " + ", ".join(f"dt{k} = (T)0" for k in range(o.D)) + ";")
                    for wc, wl in self.chunks(p.mw):
                        S = wl | 1
                        assert jobs[n][:3] == (a.idx, uc, p.t) and jobs[n][4] == self.chunk_base(p, uc, wc)
                        base, words = jobs[n][4], ul * wl

                        def pos(c):
                            return f"{c}" if S == wl else (f"{c} + (({c}) >> {wl.bit_length() - 1})" if wl & (wl - 1) == 0
                                                           else f"{c} + ({c}) / {wl}")
                        E(f"{{ // weights [{ul}][{wl}] at {base}: through LDS, one row per lane afterwards")
                        E.level += 1
                        V = width(jobs[n])
                        for i in range(_ceil(words, 64 * V)):
                            guard = "" if 64 * V * (i + 1) <= words else f"if ({64 * V * i} + {V} * lane < {words}) "
                            E(f"{guard}{{ " + " ".join(f"tile[{pos(f'{64 * V * i + h} + {V} * lane')}] = r{n % nbuf}_[{V * i + h}];"
                                                        for h in range(V)) + " }")
                        E("oeq_sync();")
                        request(n + ahead)
                        full, tail = divmod(wl, ns)

                        def step(wq):
                            E(f"  const T wv = tile[ur * {S} + {wq}];")
                            E("  const T " + ", ".join(f"g{k} = gl[{o.off + 32 * wc * o.D + k} + ({wq}) * {o.D}]"
                                                       for k in range(o.D)) + ";")
                            for k in range(o.D):
                                E(f"  dt{k} = oeq_fma(wv, g{k}, dt{k});")
                            E(("  if (act) " if lp != ul else "  ") + f"tile[ur * {S} + {wq}] = "
                              + " + ".join(f"t{k} * g{k}" for k in range(o.D)) + ";")
                        if full:
                            E(f"#pragma unroll {unroll}")
                            E(f"for (int j = 0; j < {full}; ++j) {{")
                            step(f"ws + {ns} * j")
                            E("}")
                        if tail:
                            E(f"if (ws < {tail}) {{")
                            step(f"ws + {ns * full}")
                            E("}")
                        E("oeq_sync();")
                        for i in range(_ceil(words, 64 * V)):
                            guard = "" if 64 * V * (i + 1) <= words else f"if ({64 * V * i} + {V} * lane < {words}) "
                            if V == 2:
                                E(f"{guard}{{ V2 v_; " + " ".join(f"v_[{h}] = tile[{pos(f'{128 * i + h} + 2 * lane')}];" for h in range(2))
                                  + " " + self.st2(f"Wgr + {base + 128 * i} + 2 * lane", "v_") + " }")
                            else:
                                E(guard + self.st(f"Wgr + {base + 64 * i} + lane", f"tile[{pos(f'{64 * i} + lane')}]"))
                        E("oeq_sync();")
                        E.level -= 1
                        E("}")
                        n += 1
                    s = lp
                    while s < 64:
                        E(" ".join(f"dt{k} += oeq_shfl_xor(dt{k}, {s});" for k in range(o.D)))
                        s *= 2
                    E("if (!act || ws != 0) { " + " ".join(f"dt{k} = (T)0;" for k in range(o.D)) + " }")
                    self.emit_cg_backward(E, p, "dt", "x", "y", "dx", "dy")
                    if take:
                        self._take_sums(E, [(p, "dx")])
                    E.level -= 1
                    E("}")
                E(f"if (act && ws == 0) {{ T* __restrict__ dp = Xg + row * {self.D1} + {a.off} + ({32 * uc} + uq) * {a.D}; "
                  + " ".join(f"dp[{i}] = dx{i};" for i in range(a.D)) + " }")
                E.level -= 1
                E("}")
        assert n == len(jobs)
        for f in self.used_y:
            E(f"dy{f} = oeq_wave_sum63(dy{f});")
        E("if (lane == 63) {")
        for f in range(self.D2):
            E(f"    Yg[row * {self.D2} + {f}] = " + (f"dy{f};" if f in self.used_y else "(T)0;"))
        E("}")
        return E.text()

    # A path's dT goes into dX and dY with products that nothing waits for before the row ends, and left to itself the compiler
    # keeps every dT until then: the registers grow with the paths.  Here they are taken after every four paths (of 32 channels;
    # fp64: eight), after every two where outputs reach l = 3.  Left / taken, registers (bytes of scratch) and us:
    #   fp32   44 channels of both parities, l <= 1, 7747 rows      512 (384) 367    248 240
    #          44 channels, l <= 2, 7043 rows                       264 251          245 238
    #          10 channels, l <= 3, 20 000 rows                     270 231          103 112
    #   fp64   17 channels of both parities, l <= 2, 8650 rows      454 308          236 261
    #          36 channels, l <= 3, 2516 rows                       512 (524) 323    324 268
    # Problems whose sums fit lose a little of what the order gave them, 38 channels, l <= 2, 9443 rows 265 / 271, and more where
    # they are taken after each path: DiffDock's layer, 20 000 rows 226 left, 227 after four, 231 after each.
    PUT_OFF, PUT_OFF_L3 = {"float": 4, "double": 8}, 2
    # A chunk whose rows are no longer than AHEAD's eight steps is one line to the compiler, together with those around it.  Where most
    # of a row is such chunks and some take more than STEP_WORDS words of dZ, four steps are in flight, a loop, and sums are taken every
    # two paths.  fp32, l <= 2, chunks / eight / four: 12 channels to 60 (190, 272 and 185 registers) 200 rows 16.2 / 14.8 / 16.7 us,
    # 2500 45.5 / 47.0 / 44.6, 18 939 234 / 311 / 230; 10 to 40 12.8 / 10.8 / 12.0, 20.8 / 25.1 / 19.9, 34 090 230 / 237 / 220.  Where
    # they are few, 42 channels, 7730 rows 263 / 252 / 257.
    STEP_WORDS, FEWER_STEPS = 32, 4

    def _stream_steps(self):
        """(steps in flight of a chunk's row with these words of dZ a step, paths after which sums are taken) of the backward over
        batches."""
        most, names = self.AHEAD[self.T][1], max(p.o.D for p in self.paths)
        put_off = self.PUT_OFF_L3 if names > 5 else self.PUT_OFF[self.T]
        line = [(ul * wl, wl // self._split(ul)[2] * p.o.D) for batch in self.batches for p, _, ul, _, wl, _ in batch
                if self.FEWER_STEPS < wl // self._split(ul)[2] <= most]
        if line and 2 * sum(words for words, _ in line) > self.WN and max(g for _, g in line) > self.STEP_WORDS:
            return (lambda words: self.FEWER_STEPS if most * words > self.STEP_WORDS else most), self.PUT_OFF_L3
        return (lambda words: most), put_off

    @staticmethod
    def _take(E: Emitter, names: dict) -> None:
        """The values are worked out here."""
        if names:
            E(" ".join(f"OEQ_OPAQUE({v});" for v in names))
            names.clear()

    def _take_sums(self, E: Emitter, put_off) -> None:
        """The dX (of these names) and dY of the paths are worked out here."""
        sums = dict.fromkeys([f"{dx}{i}" for p, dx in put_off for i in range(p.a.D)]
                             + [f"dy{p.b.off + j}" for p, _ in put_off for j in range(p.b.D) if p.b.off + j in self.used_y])
        self._take(E, sums)
        put_off.clear()

    def backward_stream_body(self) -> str:
        """The row's weights as batches of whole chunks, in memory order: a batch moves 16 bytes per lane and instruction, whole cache
        lines, and the next one is in flight in registers while this one is worked on in LDS.  Chunk by chunk, an access
        is as long as a chunk (400 bytes between two 10-channel blocks) and begins and ends inside a cache line.  All
        of the row's dX are live at once, as memory order takes the input blocks in turns.  DiffDock's layer, 50 000 rows
        595 -> 551 us (fp64, 20 000 rows, 465 -> 431); 8 channels, 20 000 rows 40.6 -> 38, 12, 61 -> 53, 42, 10 000 rows 150 -> 141, 36, 6000 rows
        144 -> 141.  Batches of 6 KB: 561; two or four steps of a row at a time: 568."""
        E = Emitter()
        words = [sum(ul * wl for _, _, ul, _, wl, _ in b) for b in self.batches]
        self._stream_header(E, words)
        E(f"__shared__ T gl[{max(1, self.D3)}];")
        E(f"T* __restrict__ Wgr = Wg + row * {self.WN};")
        now = [None]                                 # (path, uc, ul) whose t and dt the registers hold
        put_off = []                                 # paths whose sums the compiler may still put off
        names = max(p.o.D for p in self.paths)
        steps, put_off_most = self._stream_steps()

        def work(job, at):
            p, uc, ul = job[:3]
            if now[0] is None or (p.t, uc) != (now[0][0].t, now[0][1]):
                if now[0]:
                    finish(*now[0])
                now[0] = p, uc, ul
                E("{")
                self.emit_cg_forward(E, p, f"x{p.a.idx}_{uc}_", "y", "s")
                E(" ".join(f"t{k} = s{k}; dt{k} = (T)0;" for k in range(p.o.D)))
                E("}")
            chunk(job, at)
        stream = self._stream(E, words, work, "Wgr")
        next(stream)                                 # (the first batch is on its way)
        E(f"for (int q = lane; q < {self.D3}; q += 64) gl[q] = G[row * {self.D3} + q];")
        for f in self.used_y:
            E(f"const T y{f} = Y[row * {self.D2} + {f}];")
            E(f"T dy{f} = (T)0;")
        # lanes <-> (channel of a chunk, slice of its row), by the chunk's channels
        for ul in sorted({ul for a in self.in1 for _, ul in self.chunks(a.mul)}):
            lp, lg, _ = self._split(ul)
            E(f"const int uq{ul} = lane & {lp - 1}, ws{ul} = lane >> {lg}, ur{ul} = min(uq{ul}, {ul - 1}); const bool act{ul} = uq{ul} < {ul};")
        held = [(a, uc, ul) for a in self.in1 if a.dim for uc, ul in self.chunks(a.mul)]
        for a, uc, ul in held:
            E(f"const T* __restrict__ xp{a.idx}_{uc} = Xr + {a.off} + ({32 * uc} + ur{ul}) * {a.D};")
            E("const T " + ", ".join(f"x{a.idx}_{uc}_{i} = xp{a.idx}_{uc}[{i}]" for i in range(a.D)) + ";")
            E("T " + ", ".join(f"dx{a.idx}_{uc}_{i} = (T)0" for i in range(a.D)) + ";")
        banks = 128 // self.itemsize               # values side by side in LDS that lanes read without conflict

        def chunk(job, at):
            p, uc, ul, wc, wl, _ = job
            o = p.o
            lp, _, ns = self._split(ul)
            g = math.gcd(wl, banks)
            turn = banks // g <= banks // 4        # rows of four and more lanes would begin in one bank
            E(f"{{ // weights [{ul}][{wl}] of path {p.t}")
            E.level += 1
            if turn:
                E(f"const int turn_ = ur{ul} * {g} / {banks} % {wl};     // rows that begin in one bank are walked from another column each")
            full, tail = divmod(wl, ns)

            def step(wq):
                if turn:
                    E(f"  int c_ = {wq} + turn_; c_ -= c_ < {wl} ? 0 : {wl};")
                else:
                    E(f"  const int c_ = {wq};")
                E(f"  const T wv = tile[{at} + ur{ul} * {wl} + c_];")
                E("  const T " + ", ".join(f"g{k} = gl[{o.off + 32 * wc * o.D + k} + c_ * {o.D}]" for k in range(o.D)) + ";")
                for k in range(o.D):
                    E(f"  dt{k} = oeq_fma(wv, g{k}, dt{k});")
                E(("  if (act%d) " % ul if lp != ul else "  ") + f"tile[{at} + ur{ul} * {wl} + c_] = "
                  + " + ".join(f"t{k} * g{k}" for k in range(o.D)) + ";")
            if full:
                E(f"#pragma unroll {steps(o.D)}")
                E(f"for (int j = 0; j < {full}; ++j) {{")
                step(f"ws{ul} + {ns} * j")
                E("}")
            if tail:
                E(f"if (ws{ul} < {tail}) {{")
                step(f"ws{ul} + {ns * full}")
                E("}")
            E.level -= 1
            E("}")

        def finish(p, uc, ul):
            """dT of the channels is complete for the chunks worked on: slices summed, into dX and dY."""
            lp, _, _ = self._split(ul)
            s = lp
            while s < 64:
                E(" ".join(f"dt{k} += oeq_shfl_xor(dt{k}, {s});" for k in range(p.o.D)))
                s *= 2
            E(f"if (!act{ul} || ws{ul} != 0) {{ " + " ".join(f"dt{k} = (T)0;" for k in range(p.o.D)) + " }")
            self.emit_cg_backward(E, p, "dt", f"x{p.a.idx}_{uc}_", "y", f"dx{p.a.idx}_{uc}_", "dy")
            put_off.append((p, f"dx{p.a.idx}_{uc}_"))
            if len(put_off) == put_off_most:
                self._take_sums(E, put_off)
        E("T " + ", ".join(f"{v}{k} = (T)0" for v in ("t", "dt") for k in range(names)) + ";")
        for _ in stream:
            pass
        finish(*now[0])
        for a, uc, ul in held:
            E(f"if (act{ul} && ws{ul} == 0) {{ T* __restrict__ dp = Xg + row * {self.D1} + {a.off} + ({32 * uc} + uq{ul}) * {a.D}; "
              + " ".join(f"dp[{i}] = dx{a.idx}_{uc}_{i};" for i in range(a.D)) + " }")
        for f in self.used_y:
            E(f"dy{f} = oeq_wave_sum63(dy{f});")
        E("if (lane == 63) {")
        for f in range(self.D2):
            E(f"    Yg[row * {self.D2} + {f}] = " + (f"dy{f};" if f in self.used_y else "(T)0;"))
        E("}")
        return E.text()

    def render(self, prelude: str = None) -> str:
        env = jinja_env()
        if prelude is None:
            prelude = env.get_template("prelude.hip.jinja").render(T=self.T)
        return env.get_template("tp_uvw_batched.hip.jinja").render(g=self, prelude=prelude)

    def plan(self):
        fwd = [dict(kernel="forward", num_threads=64, grid_kind=1, work_per_block=1)]
        bwd = [dict(kernel="backward", num_threads=64, grid_kind=1, work_per_block=1)] if self.has_backward else []
        return fwd, bwd, (lambda nnz=0, nodes=0: 0)
