"""Double backward of the uvu batch product in one launch.

The product is trilinear in (x, y, w), so with cotangents (a, b, v) of (dx, dy, dw) the second derivatives are sums of
first-order terms with one operand replaced (reference: openequivariance/implementations/TensorProductBase.py:281-298
composes them from four backward and three forward calls, and so does ``autograd_glue.double_backward_terms``).  Per path
and channel, with s_ij = sum_k c_ijk g_k, t_i = sum_j s_ij y_j and t'_i = sum_j s_ij b_j:

    gx_i += w t'_i + v t_i                      gw  += sum_i a_i t_i + x_i t'_i
    gy_j += sum_i s_ij (w a_i + v x_i)          gg_k += sum_ij c_ijk ((w a_i + v x_i) y_j + w x_i b_j)

i.e. everything the seven launches compute from one read of the operands, about twice the arithmetic of one backward.

Bound: HBM.  Per row it reads x, y, w, their cotangents and dz and writes four gradients: 3 (d1 + d2 + wn) + 2 d3 words,
where the composition moved 4 backward + 3 forward calls and five elementwise sums: 7.0 times as much for the 8-path,
128-channel MACE problem.  On 20 011 rows of it: 782 us before,
160 us now (5.6 TB/s; an elementwise add of large tensors moves 5.9), forward + backward + double backward 1087 -> 320 us.

The schedule is the backward's of ``uvu_direct.py``: a wavefront per row (R rows for up to 32 channels), register-direct
loads, chunks of 64 channels in a loop; gg leaves through the LDS slot like the forward's Z.
"""
from __future__ import annotations

from ..problem import TPProblem
from .common import WAVE, Emitter, jinja_env
from .uvu import Block, Path
from .uvu_direct import UVUDirectGenerator


class DoubleArithmetic:
    """The arithmetic of one output block, shared by the batch product and the convolution."""

    def emit_double_block(self, E: Emitter, o: Block, zname: str, dw_sink, declare: bool = True) -> None:
        """Given g{k} = dZ[o][u, k], the weights ``w{t}_{v}`` and their cotangents ``ww{t}_{v}`` in registers: adds to
        dx{a}_{i}, dy{f} and {zname}{k}, and hands every second gradient of a weight to ``dw_sink``.  Without ``zname``
        only the former, without ``dw_sink`` only the sums {zname}{k} (no g{k} needed)."""
        if declare:
            E("T " + ", ".join(f"{zname}{k} = (T)0" for k in range(o.D)) + ";")
        for p in self.paths_into(o.idx):
            E(f"{{ // path {p.t}: l = {p.a.l} x {p.b.l} -> {p.o.l}")
            E.level += 1
            if dw_sink:
                self._emit_cg_products(E, p)
            for v in range(p.mv):
                E("{")
                E.level += 1
                self._emit_double_pairs(E, p, v, zname, bool(dw_sink))
                if dw_sink:
                    dw_sink(E, p, v, "dw")
                E.level -= 1
                E("}")
            E.level -= 1
            E("}")

    def emit_settle(self, E: Emitter, oi: int) -> None:
        """The sums an output block has added to are final here: the stores behind a block sit in branches, and the
        compiler otherwise moves the additions to dx and dy past them, with every operand alive until the end."""
        ps = self.paths_into(oi)
        names = [f"dx{i}_{m}" for i in sorted({p.a.idx for p in ps}) for m in range(self.in1[i].D)]
        names += [f"dy{f}" for f in sorted({p.b.off + v * p.b.D + j for p in ps for v in range(p.mv) for (_, j) in p.pairs})]
        E(" ".join(f"OEQ_OPAQUE({n});" for n in names))

    def _emit_double_pairs(self, E: Emitter, p: Path, v: int, zname: str, first: bool) -> None:
        """The (i, j) pairs of one path: with ``first`` the sums proportional to dZ (dw, dx, dy), with ``zname`` those
        of the gradient of dZ."""
        by_i = {}
        for (i, j), ks in sorted(p.pairs.items()):
            by_i.setdefault(i, []).append((j, ks))
        w, ww, X = f"w{p.t}_{v}", f"ww{p.t}_{v}", p.a.idx
        f = lambda j: p.b.off + v * p.b.D + j
        if first:
            E("T dw = (T)0;")
        for i, lst in sorted(by_i.items()):
            wx = f"wx = {w} * x{X}_{i}, " if zname else ""
            E(f"{{ const T {wx}pi = oeq_fma({w}, a{X}_{i}, {ww} * x{X}_{i});")
            E.level += 1
            if first:
                E("T t, tb;")
            for n_, (j, ks) in enumerate(lst):
                E("{")
                y, b = f"y{f(j)}", f"b{f(j)}"
                if first:
                    if len(ks) == 1:
                        E(f"  const T s = {'-' if ks[0][1] < 0 else ''}{self._cg_names[self._cg_key(*ks[0])]};")
                    else:
                        E(f"  T s = {self.lit(ks[0][1])} * g{ks[0][0]};")
                        for k, val in ks[1:]:
                            E(f"  s = oeq_fma({self.lit(val)}, g{k}, s);")
                    E(f"  t = s * {y}; tb = s * {b};" if n_ == 0 else f"  t = oeq_fma(s, {y}, t); tb = oeq_fma(s, {b}, tb);")
                    E(f"  dy{f(j)} = oeq_fma(s, pi, dy{f(j)});")
                if zname:
                    E(f"  const T q = oeq_fma(wx, {b}, pi * {y});")
                    E("  " + " ".join(f"{zname}{k} = oeq_fma({self.lit(val)}, q, {zname}{k});" for k, val in ks))
                E("}")
            if first:
                E(f"dw = oeq_fma(a{X}_{i}, t, dw); dw = oeq_fma(x{X}_{i}, tb, dw);")
                E(f"dx{X}_{i} = oeq_fma({w}, tb, dx{X}_{i}); dx{X}_{i} = oeq_fma({ww}, t, dx{X}_{i});")
            E.level -= 1
            E("}")


class UVUDoubleGenerator(DoubleArithmetic, UVUDirectGenerator):
    """One kernel: ``double_backward``."""

    @classmethod
    def suits(cls, problem: TPProblem) -> bool:
        """Per-row weights, at most 8 copies of a second-operand irrep (more are walked by a run-time loop elsewhere)."""
        return (not problem.shared_weights
                and max(problem.irreps_in2[i.i_in2].mul for i in problem.instructions) <= 8)

    def __init__(self, problem: TPProblem, vector_stores: bool = True):
        super().__init__(problem, "tp", vector_stores=vector_stores)
        assert not self.NLY

    def describe(self) -> str:
        return super().describe() + " double backward"

    def render(self, prelude: str = None) -> str:
        env = jinja_env()
        if prelude is None:
            prelude = env.get_template("prelude.hip.jinja").render(T=self.T)
        return env.get_template("tp_uvu_double.hip.jinja").render(g=self, prelude=prelude)

    def plan(self):
        """Launches of the double backward (the call takes no workspace)."""
        return [dict(kernel="double_backward", num_threads=64, grid_kind=1, work_per_block=self.R)]

    def body(self) -> str:
        E = Emitter()
        self.nt_load = self.nt_store = True       # as in the backward: every word is touched once
        self.emit_lane_direct(E, lds=True)
        _, _, rc = self._rows(E)
        E(f"const T* __restrict__ Br = B + {rc} * {self.D2};")
        E(f"const T* __restrict__ Vr = V + {rc} * {self.WN};")
        E(f"T* __restrict__ Wgr = Wg + {rc} * {self.WN};")
        for f in self.used_y:
            E(f"const T y{f} = Yr[{f}], b{f} = Br[{f}];")
            E(f"T dy{f} = (T)0;")
        if self.NCH == 1:
            E("{")
            E.level += 1
            E("const int c = 0, u = ul; (void)c;")
            self._chunk(E, 0, rc)
        else:
            E("#pragma unroll 1")
            E(f"for (int c = 0; c < {self.NCH}; ++c) {{")
            E.level += 1
            E(f"const int u = c * {self.P} + ul;")
            self._chunk(E, "c", rc)
        E.level -= 1
        E("}")
        for f in self.used_y:
            E(f"dy{f} = {'oeq_wave_sum63' if self.P == WAVE else f'oeq_group_sum<{self.P}>'}(dy{f});")
        E(f"if ({'lane == 63' if self.P == WAVE else 'ul == 0'}) {{")
        E(f"    T* __restrict__ Ygr = Yg + {rc} * {self.D2};")
        for f in range(self.D2):
            E(f"    Ygr[{f}] = " + (f"dy{f};" if f in self.used_y else "(T)0;"))
        E("}")
        return E.text()

    def _chunk(self, E: Emitter, c, rc: str) -> None:
        for i in self.used_in1:
            blk = self.in1[i]
            for src, name in (("X", "x"), ("A", "a")):
                self.emit_record_load(E, [f"{name}{i}_{m}" for m in range(blk.D)],
                                      f"{src} + (u64){rc} * {self.D1} + {blk.off} + {self.uclamp(blk, c)} * {blk.D}", self.act_c(blk, c))
            E("T " + ", ".join(f"dx{i}_{m} = (T)0" for m in range(blk.D)) + ";")

        def fetch(oi):
            o = self.out[oi]
            # everything a lane adds up across lanes (dy) is proportional to dZ: zero for idle lanes
            self.emit_record_load(E, [f"G{oi}_{k}" for k in range(o.D)],
                                  f"G + (u64){rc} * {self.D3} + {o.off} + {self.uclamp(o, c)} * {o.D}", self.act(o), zero=True)
            for p in self.paths_into(oi):
                for v in range(p.mv):
                    idx = self.widx(p, self.uclamp(p.a, c), v)
                    E(f"const T w{p.t}_{v} = oeq_ldnt(Wr + {idx}), ww{p.t}_{v} = oeq_ldnt(Vr + {idx});")
        lazy = self.one_block_ahead()
        for oi in (self.used_out[:1] if lazy else self.used_out):
            fetch(oi)
        for n_, oi in enumerate(self.used_out):
            o = self.out[oi]
            if lazy:
                E("oeq_sched_fence();")
                if n_ + 1 < len(self.used_out):
                    fetch(self.used_out[n_ + 1])
            E("{")
            E.level += 1
            E("const T " + ", ".join(f"g{k} = G{oi}_{k}" for k in range(o.D)) + ";")

            def sink(E, p, v, expr):
                act = self.act(p.a)
                E(("" if act == "true" else f"if ({act}) ") + f"oeq_stnt(Wgr + {self.widx(p, 'u', v)}, {expr});")
            self.emit_double_block(E, o, "z", sink)
            self.emit_settle(E, oi)
            self.emit_block_store(E, o, [f"z{k}" for k in range(o.D)], "Gg", self.D3, rc, self.zrow_of, "store", via_lds=True)
            E.level -= 1
            E("}")
        for o in self.out:
            if o.dim and o.idx not in self.used_out:
                self.emit_record_store(E, ["(T)0"] * o.D, f"Gg + (u64){rc} * {self.D3} + {o.off} + u * {o.D}", self.act(o))
        for a in self.in1:
            if a.dim == 0:
                continue
            if a.idx in self.used_in1:
                self.emit_block_store(E, a, [f"dx{a.idx}_{m}" for m in range(a.D)], "Xg", self.D1, rc, self.xrow_of, "store",
                                      via_lds=self.dx_through_slot(a))
            else:
                self.emit_record_store(E, ["(T)0"] * a.D, f"Xg + (u64){rc} * {self.D1} + {a.off} + u * {a.D}", self.act(a))

    ONE_BLOCK_AHEAD = None

    def one_block_ahead(self) -> bool:
        """dZ and the weights requested one output block ahead instead of all at the top of the row: fewer registers in
        flight (135 instead of 206 on the 17-path MACE problem), more waits.  Measured on MI355X, 20 000 rows in fp32,
        10 000 in fp64, us, ahead / at once:

            channels, paths, words       fp32             fp64
            128,  8,  42                 165.5 / 160.3    178.6 / 179.7
            128, 17, 105                 433.4 / 431.1    469.1 / 494.3
             32, 11,  57                  61.4 /  58.6     67.0 /  67.5
             64, 13,  69                 147.4 / 147.8    160.8 / 160.0
             32, 30, 162                 179.5 / 190.2    184.2 / 206.6
             37,  5,  25 (ragged)         41.5 /  34.8     35.5 /  33.7
            256, 13,  69                 613.7 / 616.9    651.1 / 681.4

        The rule takes it from 128 words (32-bit) per lane on."""
        if self.ONE_BLOCK_AHEAD is not None:
            return self.ONE_BLOCK_AHEAD
        words = sum(self.out[i].D for i in self.used_out) + 2 * sum(p.mv for p in self.paths)
        return words * (2 if self.T == "double" else 1) > 128
