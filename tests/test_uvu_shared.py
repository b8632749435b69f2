"""uvu with one weight vector for the batch: dW sums held across rows, one partial row per workgroup.  The generated
source on the host (tests/host_emu) and the operator on the GPU, at the edges of the schedule: several rows per
wavefront, ragged multiplicities, one to three 64-channel chunks per row, more paths than one LDS fold takes, copies of
the second operand, dX through the LDS slot, batches below, at and above what one workgroup walks."""
import numpy as np
import pytest

import common
import openequivariance_amd as oeq
from common import FP32_TOL, FP64_TOL, rel_err
from host_emu import emu
from openequivariance_amd.codegen.uvu_shared import UVUSharedGenerator
from openequivariance_amd.tensor_product import select_generator
from oracle import spec, tp as otp, weights as ow

TWO = ("1x0e+1x1o", [(0, 0, 0, "uvu", True), (1, 1, 0, "uvu", True), (1, 0, 1, "uvu", True)])
CASES = {
    "two_rows_per_wavefront": ("24x0e+24x1o", *TWO, (1, 9)),
    "sixteen_rows": ("3x0e+3x1o", *TWO, (1, 63, 130)),
    "one_chunk": ("64x0e+64x1o", *TWO, (1, 4, 9)),
    "two_ragged_chunks": ("70x0e+5x1o", "1x0e+1x1o", [(0, 0, 0, "uvu", True), (1, 0, 1, "uvu", True), (0, 0, 0, "uvu", True)],
                          (1, 8, 19)),
    "three_chunks": ("130x0e+130x1o", *TWO, (1, 5)),
    "copies_of_the_second_operand": ("12x0e+12x1o", "4x0e+3x1o", [(0, 0, 0, "uvu", True), (1, 1, 0, "uvu", True),
                                                                  (1, 0, 1, "uvu", True)], (7, 33)),
    "long_records": ("20x3o+20x0e", "1x3o+1x0e", [(0, 0, 1, "uvu", True), (0, 1, 0, "uvu", True)], (1, 11)),
}


def _problems(case, dtype=np.float32):
    irreps, in2, ins, _ = CASES[case]
    return (oeq.TPProblem(irreps, in2, irreps, ins, shared_weights=True, internal_weights=False, irrep_dtype=dtype,
                          weight_dtype=dtype), spec.Problem(irreps, in2, irreps, ins, shared_weights=True))


@pytest.mark.parametrize("case", sorted(CASES))
def test_generated_source(case, monkeypatch):
    prob, oprob = _problems(case)
    monkeypatch.setattr(UVUSharedGenerator, "MAX_WORKGROUPS", 2)      # several tiles per workgroup at these sizes
    g = select_generator(prob)
    assert type(g) is UVUSharedGenerator
    fwd, bwd, ws = g.plan()
    for n in CASES[case][3]:
        X, Y, We, G = common.tp_inputs(prob, n, 17)
        W = ow.e3nn_to_oeq(oprob, We)
        out = emu.run_tp(g, fwd, X, Y, W, ws_bytes=ws())
        assert rel_err(out["Z"], otp.forward(oprob, X, Y, We)) < 2e-6
        out = emu.run_tp(g, bwd, X, Y, W, G, ws_bytes=ws())
        dX, dY, dW = otp.backward(oprob, X, Y, We, G)
        for got, ref in ((out["Xg"], dX), (out["Yg"], dY), (ow.oeq_to_e3nn(oprob, out["Wg"]), dW)):
            assert rel_err(got, ref) < 2e-6      # fp32 sums of at most 130 rows x 7 words against fp64


@pytest.mark.parametrize("case", ["sixteen_rows", "two_ragged_chunks"])
def test_generated_source_without_vector_stores(case):
    prob, oprob = _problems(case)
    g = UVUSharedGenerator(prob, vector_stores=False)
    fwd, bwd, ws = g.plan()
    n = CASES[case][3][-1]
    X, Y, We, G = common.tp_inputs(prob, n, 19)
    W = ow.e3nn_to_oeq(oprob, We)
    assert rel_err(emu.run_tp(g, fwd, X, Y, W, ws_bytes=ws())["Z"], otp.forward(oprob, X, Y, We)) < 2e-6
    out = emu.run_tp(g, bwd, X, Y, W, G, ws_bytes=ws())
    for got, ref in zip((out["Xg"], out["Yg"], ow.oeq_to_e3nn(oprob, out["Wg"])), otp.backward(oprob, X, Y, We, G)):
        assert rel_err(got, ref) < 2e-6


# wide second operands beside the sixteen or eight wavefronts of a row: (dtype, in1 = out, in2, taken)
WIDE = {
    "144_words": (np.float64, "1024x0e+1024x1o", "+".join(f"1x{l}e" for l in range(12)), True),
    "169_words": (np.float64, "1024x0e+1024x1o", "+".join(f"1x{l}e" for l in range(13)), False),
    "392_words": (np.float64, "512x0e+512x1o", "+".join(f"8x{l}e" for l in range(7)), False),
    "392_words_fp32": (np.float32, "512x0e+512x1o", "+".join(f"8x{l}e" for l in range(7)), True),
    "dx_slots": (np.float64, "1024x6e", "+".join(f"1x{l}e" for l in range(8)), False),
}


@pytest.mark.parametrize("case", sorted(WIDE))
def test_arrays_fit_lds_together(case):
    dtype, irreps, in2, taken = WIDE[case]
    prob = oeq.TPProblem(irreps, in2, irreps, [(0, 0, 0, "uvu", True), (0, 2, 0, "uvu", True)] if case == "dx_slots" else
                         [(0, 0, 0, "uvu", True), (1, 0, 1, "uvu", True)], shared_weights=True, internal_weights=False,
                         irrep_dtype=dtype, weight_dtype=dtype)
    g = select_generator(prob)
    assert (type(g) is UVUSharedGenerator) == taken
    used = common.lds_bytes(UVUSharedGenerator(prob).render(), np.dtype(dtype).itemsize)["backward"]
    assert used == UVUSharedGenerator(prob).lds_bytes() and (used <= 160 * 1024) == taken
    assert max(common.lds_bytes(g.render(), np.dtype(dtype).itemsize).values()) <= 160 * 1024


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("case", sorted(CASES))
def test_operator(cuda, case, dtype):
    import torch
    prob, oprob = _problems(case, dtype)
    tol = FP32_TOL if dtype == np.float32 else FP64_TOL
    tp = oeq.TensorProduct(prob, torch_op=True)
    assert type(tp.generator) is UVUSharedGenerator
    for n in (0, *CASES[case][3], 5003):
        X, Y, We, G = common.tp_inputs(prob, n, 18, dtype)
        x, y, w = (torch.tensor(t, device=cuda, requires_grad=True) for t in (X, Y, ow.e3nn_to_oeq(oprob, We)))
        z = tp(x, y, w)
        z.backward(torch.tensor(G, device=cuda))
        torch.cuda.synchronize()
        dX, dY, dW = otp.backward(oprob, X, Y, We, G)
        for got, ref in ((z.detach(), otp.forward(oprob, X, Y, We)), (x.grad, dX), (y.grad, dY)):
            assert rel_err(got.cpu().numpy(), ref) <= tol
        assert rel_err(ow.oeq_to_e3nn(oprob, w.grad.cpu().numpy()), dW) <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_misaligned_operands(cuda, dtype):
    """Operands at an odd storage offset take the kernels without 16-byte stores."""
    import torch
    prob, oprob = _problems("two_ragged_chunks", dtype)
    tol = FP32_TOL if dtype == np.float32 else FP64_TOL
    tp = oeq.TensorProduct(prob, torch_op=True)
    X, Y, We, G = common.tp_inputs(prob, 301, 20, dtype)
    odd = lambda a: torch.zeros(a.size + 1, dtype=torch.tensor(a).dtype, device=cuda)[1:].view(a.shape).copy_(torch.tensor(a))
    x, y, w, g = (odd(a) for a in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
    got = [tp.forward(x, y, w), *tp.backward_helper(x, y, w, g)]
    torch.cuda.synchronize()
    assert tp._internal_unaligned is not None
    got = [t.cpu().numpy() for t in got]
    got[3] = ow.oeq_to_e3nn(oprob, got[3])
    for a, b in zip(got, (otp.forward(oprob, X, Y, We), *otp.backward(oprob, X, Y, We, G))):
        assert rel_err(a, b) <= tol
