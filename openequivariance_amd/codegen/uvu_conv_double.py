"""Double backward of the fused convolution in two passes over the edges.

With cotangents (A, B, V) of the backward's outputs (dX, dY, dW), the four second gradients split by who sums them
(formulas in ``uvu_double.py``; the reference composes them from four backward and three forward calls,
openequivariance/implementations/convolution/ConvolutionBase.py:618-636 and :691-709):

* the gradient of dZ is a sum over the edges of a receiver: the forward's walk (``forward``), with the senders' rows of X
  and A gathered per edge and W, V, Y, B streamed;
* the gradients of X (a sum over the edges of a sender), W and Y (per edge) are proportional to dZ: the backward's walk
  (``backward``), with X and A of the sender held, dZ of the receiver gathered and W, V, Y, B streamed.

Both passes are the loops of ``uvu_det.py`` (pieces of long nodes, groups of output blocks, LDS-staged or register
pipeline) with a cotangent beside each operand; every sum has the order the first-order kernels give it, so the
deterministic operator stays bit-reproducible.
"""
from __future__ import annotations

from .. import tunables
from .uvu_det import UVUDetGenerator
from .uvu_double import DoubleArithmetic
from .uvu_sorted import UVUSortedGenerator

CALL_ARGS = ("const T* __restrict__ X, const T* __restrict__ Y, const T* __restrict__ W, const T* __restrict__ G, \\\n"
             "    const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ V, \\\n"
             "    T* __restrict__ Xg, T* __restrict__ Yg, T* __restrict__ Wg, T* __restrict__ Gg, \\\n"
             "    const IDX* __restrict__ rows, const IDX* __restrict__ cols, u64 nnz, u64 node_count, \\\n"
             "    void* __restrict__ ws, const IDX* __restrict__ tperm")


class _DoublePlan:
    """Both passes' preparations are one: in launches of their own, 4 of the 150 us of forces of 30 000 edges sorted by receiver
    (1001 nodes, 32 channels)."""
    both_prepared = True

    def steps(self):
        return self._one_list(*self.plan()[:2])

    def steps_few(self):
        return self._one_list(*self.plan_few()[:2])

    @staticmethod
    def _one_list(fwd, bwd):
        prep = [s for s in bwd if s["kernel"].startswith(("prep_", "group_"))]
        return prep + fwd + bwd[len(prep):]

    @staticmethod
    def variant():
        """What the source depends on beside the problem."""
        t = tunables.current
        return t.det_lds, t.det_split, t.det_prefetch, t.long_node


class UVUDetDoubleGenerator(_DoublePlan, DoubleArithmetic, UVUDetGenerator):
    """Over an edge list sorted by receiver with its transpose permutation."""
    EDGE_W = (("W", "We_"), ("V", "Ve_"))
    EDGE_Y = (("Y", "y"), ("B", "b"))
    NODE_X = (("X", "x"), ("A", "a"))
    NODE_OUT = "Gg"
    # Rules of the loops, measured on MI355X over whole calls (us; graphs of 1000 - 3000 nodes, 20 000 - 60 000 edges).
    # Receiver pass staged through LDS where the multiplicity fits one chunk (32 channels, 11 paths: 109 registers, 96
    # staged; several chunks, 100 / 128 channels: 415 / 420, 441 / 447)
    FWD_STAGE_WAVES = 8
    F64_STAGE_WORDS = 0
    FWD_STAGE_OPERANDS = 1 << 30
    # ... and one launch up to 48 words of sums in fp64 (38 words: 197, in two 224; 42 words: 566 and 566; 102 words in
    # groups of 32 / 48 / 64: 900 / 879 / 843)
    FWD_SPLIT_WORDS = {"float": 100, "double": 48}
    # Sender pass: an edge brings twice the weights and second-operand words, but a further launch costs X, A, Y, B and
    # the indices again; one launch up to 144 words, as many per launch beyond.  The first-order rule (80 words, 64 / 24
    # per launch) against this: 127 words 128 channels fp32 433 / 418, fp64 654 / 503, 64 channels fp64 566 / 411;
    # 254 words 32 channels fp32 532 / 490 (in one launch 870), 64 channels fp32 566 / 488, fp64 900 / 625 (one: 1121)
    SPLIT_WORDS = 144
    CALL_FWD_ARGS = CALL_BWD_ARGS = CALL_ARGS

    def __init__(self, problem, **kw):
        super().__init__(problem, **kw)
        self.regroup_pairs = True         # (the double backward has one form)

    def split_limit(self) -> int:
        # fp64: with X, A and dX of the sender held beside them, more than 200 words do not fit 512 registers (68 paths,
        # 32 words per in1 row: 76 - 196 bytes of scratch per lane at 144 words, none at 104)
        held = 3 * sum(self.in1[i].D for i in self.used_in1)
        return self.SPLIT_WORDS if self.T == "float" else max(48, min(self.SPLIT_WORDS, 200 - held))

    def sender_launches(self, words: int, limit: int) -> int:
        again = len(self.EDGE_Y) * len(self.used_y)           # words that every launch reads
        return -(-(words - again) // max(16, limit - again))

    def describe(self) -> str:
        return super().describe() + " double backward"

    def _weights(self, E, o) -> None:
        for p in self.paths_into(o.idx):
            E(f"const T w{p.t}_0 = We_{p.t}_0, ww{p.t}_0 = Ve_{p.t}_0;")

    def emit_receiver_block(self, E, o, zname: str) -> None:
        E("{")
        self._weights(E, o)
        self.emit_double_block(E, o, zname, None, declare=False)
        E("}")

    def emit_sender_block(self, E, o, sink) -> None:
        self._weights(E, o)
        self.emit_double_block(E, o, "", sink, declare=False)
        self.emit_settle(E, o.idx)


class UVUSortedDoubleGenerator(_DoublePlan, UVUSortedGenerator):
    """Over an edge list in any order: both groupings are built in the workspace first."""
    SEGMENTED = UVUDetDoubleGenerator

    def __init__(self, problem, **kw):
        super().__init__(problem, grouped_backward=True, recv_backward=False, **kw)


def conv_double_generator(problem, deterministic: bool, idx_ctype: str = "i64"):
    return (UVUDetDoubleGenerator if deterministic else UVUSortedDoubleGenerator)(problem, idx_ctype=idx_ctype)
