"""uvw products with per-row weights whose weights pass in batches of 16-byte pieces: chunks of every width that divides
into such, rows of a chunk that would meet in one LDS bank (walked from other columns), several copies of the second operand,
batches of one and of many chunks, both types; rows that do not divide keep the other schedule."""
import numpy as np
import pytest

import common
from common import rel_err
from host_emu import emu
from openequivariance_amd.codegen.uvw_batched import UVWBatchedGenerator
from oracle import tp as otp
from oracle import weights as ow

CASES = {
    "short_chunks": ("10x1o+10x1e+20x0e", "1x0e+1x1o", "10x1o+10x1e+20x0e"),
    "rows_of_32_16_8_4_words": ("34x0e+6x1o", "1x0e+1x1o", "32x0e+48x1o+8x0o+4x2e"),
    "copies": ("10x0e+40x1o", "3x0e+2x1o", "36x0e+10x1o"),
    "l3": ("12x0e+6x1o+10x3o", "1x0e+1x1o+1x2e+1x3o", "12x0e+6x1o+4x2e+10x3o"),
    "rows_in_one_line": ("12x0e+12x2e", "1x0e+1x1o+1x2e", "44x0e+64x2e"),
    "few_to_many": ("4x0e+8x1o+6x1e", "1x0e+1x1o", "66x0e+40x1o+6x1e"),
    "odd_paths_even_row": ("3x0e+5x1o", "1x0e+1x1o", "4x0e+1x1o"),
}
TOL = {np.float32: 4e-6, np.float64: 1e-13}       # a few hundred roundings a value


def generator(case, dtype):
    prob, oprob = common.fully_connected(CASES[case], shared=False, dtype=dtype)
    return UVWBatchedGenerator(prob), prob, oprob


def test_which_rows_stream():
    for case in CASES:
        for dtype in TOL:
            g, prob, _ = generator(case, dtype)
            assert g.stream and g.stream_backward and sum(len(b) for b in g.batches) == sum(len(g.chunks(p.mu)) * len(g.chunks(p.mw)) for p in g.paths)
            assert all(b[0][-1] * g.itemsize % 16 == 0 for b in g.batches) and len(g.batches) > (case != "odd_paths_even_row")
            assert not UVWBatchedGenerator(prob, stream=False).stream
    ragged, lines = (UVWBatchedGenerator(common.fully_connected(irreps, shared=False)[0]) for irreps in
                     (("5x0e+21x1o", "1x0e+1x1o+1x2e", "18x0e+7x1o+3x2e"), ("32x0e+32x1o", "1x0e+1x1o", "32x0e+32x1o")))
    assert not ragged.stream and not ragged.stream_backward and lines.stream and not lines.stream_backward


@pytest.mark.parametrize("mul, lmax, parities, dtype, most", [(44, 1, "eo", np.float32, 256), (10, 3, "", np.float32, 128),
                                                               (17, 2, "eo", np.float64, 256), (36, 3, "", np.float64, 512)])
def test_registers_of_the_backward_are_bounded(mul, lmax, parities, dtype, most):
    """Many paths between few channels: their sums are not all kept until the row ends (two wavefronts per SIMD have 256 registers
    each), and none goes to memory."""
    from openequivariance_amd import runtime as rt
    irreps = "+".join(f"{mul}x{l}{p}" for l in range(lmax + 1) for p in (parities or "eo"[l % 2]))
    g = UVWBatchedGenerator(common.fully_connected((irreps, "+".join(f"1x{l}{'eo'[l % 2]}" for l in range(lmax + 1)), irreps), shared=False,
                                                   dtype=dtype)[0])
    assert g.stream_backward
    k = rt.kernel_metadata(rt.compile_source(g.render(), use_cache=False))["backward"]
    assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_count"] <= most


@pytest.mark.parametrize("mul, out, steps, most", [(12, 60, (4, 2), 192), (10, 40, (4, 2), 168), (42, 42, (8, 4), 256), (60, 12, (8, 4), 256)])
def test_registers_of_chunks_in_one_line(mul, out, steps, most):
    """Rows of eight steps with five words of dZ each (12 channels to 60: 272 registers with all of them in flight)."""
    from openequivariance_amd import runtime as rt
    g = UVWBatchedGenerator(common.fully_connected((f"{mul}x0e+{mul}x1o+{mul}x2e", "1x0e+1x1o+1x2e", f"{out}x0e+{out}x1o+{out}x2e"), shared=False)[0])
    assert g.stream_backward and (g._stream_steps()[0](5), g._stream_steps()[1]) == steps and g._stream_steps()[0](3) == 8
    k = rt.kernel_metadata(rt.compile_source(g.render(), use_cache=False))["backward"]
    assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_count"] <= most


@pytest.mark.parametrize("mul, out, dtype, most", [(8, 36, np.float32, 128), (8, 36, np.float64, 256), (4, 34, np.float64, 256), (6, 50, np.float32, 128),
                                                    (8, 100, np.float64, 320)])
def test_registers_of_the_forward_are_bounded(mul, out, dtype, most):
    """Few channels: a chunk's rows are no loop (8 to 36, fp64: 512 registers and 1972 bytes of scratch where all sums wait for the end)."""
    from openequivariance_amd import runtime as rt
    irreps = tuple("+".join(f"{m}x{l}{p}" for l in range(3) for p in "eo") for m in (mul, out))
    g = UVWBatchedGenerator(common.fully_connected((irreps[0], "1x0e+1x1o+1x2e", irreps[1]), shared=False, dtype=dtype)[0])
    assert g.stream_forward
    k = rt.kernel_metadata(rt.compile_source(g.render(), use_cache=False))["forward"]
    assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_count"] <= most


def test_wide_first_operands_keep_the_walk_over_chunks():
    """A lane of a batch holds its channels' X (and dX) over the whole row."""
    from openequivariance_amd import runtime as rt

    def gen(irreps, dtype):
        return UVWBatchedGenerator(common.fully_connected(irreps, shared=False, dtype=dtype)[0])
    wide, half = ("512x0e+512x1o+512x2e", "1x0e+1x1o", "4x0e+4x1o+4x2e"), ("256x0e+256x1o+256x2e", "1x0e+1x1o+1x2e", "4x0e+4x1o")
    for irreps, dtype, forward, backward in ((wide, np.float32, False, True), (wide, np.float64, False, False), (half, np.float32, True, True),
                                             (half, np.float64, False, True), (("2000x1o", "1x0e+1x1o", "4x0e+4x1o"), np.float64, False, False),
                                             (("100x0e+100x0o+100x1o+100x1e+100x2e+100x2o", "1x0e+1x1o+1x2e", "100x0e+100x1o+100x2e"), np.float64, True, False)):
        g = gen(irreps, dtype)
        assert (g.stream_forward, g.stream_backward, g.stream) == (forward, backward, forward or backward)
    for k in rt.kernel_metadata(rt.compile_source(gen(wide, np.float64).render(), use_cache=False)).values():
        assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_count"] <= 256


def test_long_rows_keep_the_walk_over_chunks():
    """fp32, 25 000 words and more: a wavefront's four chunks in flight do more for few rows than one batch does."""
    gens = [UVWBatchedGenerator(common.fully_connected((f"{m}x0e+{m}x1o+{m}x2e", "1x0e+1x1o+1x2e", f"{m}x0e+{m}x1o+{m}x2e"), shared=False, dtype=dtype)[0])
            for m, dtype in ((46, np.float32), (52, np.float32), (50, np.float64))]
    assert [(g.stream, g.stream_backward) for g in gens] == [(True, True), (True, False), (True, True)]


@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("case", list(CASES))
def test_emulated(case, dtype):
    g, prob, oprob = generator(case, dtype)
    X, Y, We, G = common.tp_inputs(prob, 3, 10, dtype=dtype, w_scale=0.3)
    fwd, bwd, _ = g.plan()
    out = emu.run_tp(g, fwd, X, Y, ow.e3nn_to_oeq(oprob, We))
    assert rel_err(out["Z"], otp.forward(oprob, X, Y, We)) < TOL[dtype]
    out = emu.run_tp(g, bwd, X, Y, ow.e3nn_to_oeq(oprob, We), G)
    dX, dY, dW = otp.backward(oprob, X, Y, We, G)
    assert rel_err(out["Xg"], dX) < TOL[dtype] and rel_err(out["Yg"], dY) < TOL[dtype]
    assert rel_err(ow.oeq_to_e3nn(oprob, out["Wg"]), dW) < TOL[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("case", [*CASES, "diffdock"])
def test_on_the_gpu(cuda, case, dtype, monkeypatch):
    """Against the oracle, also with weights off 16 and off 8 bytes."""
    import torch
    import openequivariance_amd as oeq
    monkeypatch.setitem(CASES, "diffdock", ("10x1o+10x1e+48x0e+48x0o", "1x0e+1x1o+1x2e", "10x1o+10x1e+48x0e+48x0o"))
    g, prob, oprob = generator(case, dtype)
    tp = oeq.TensorProduct(prob, torch_op=True)
    assert tp.generator.stream
    for n in (1, 37, 1025):
        X, Y, We, G = common.tp_inputs(prob, n, n, dtype=dtype, w_scale=0.3)
        x, y, w, dz = (torch.tensor(a, device=cuda) for a in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
        dX, dY, dW = otp.backward(oprob, X, Y, We, G)
        for off in (0, 1, 2):
            v = torch.cat([w.new_zeros(off), w.reshape(-1)])[off:].view(w.shape)
            assert rel_err(tp.forward(x, y, v).cpu().numpy(), otp.forward(oprob, X, Y, We)) < TOL[dtype]
            got = [t.cpu().numpy() for t in tp.backward_helper(x, y, v, dz)]
            for a, b in zip((*got[:2], ow.oeq_to_e3nn(oprob, got[2])), (dX, dY, dW)):
                assert rel_err(a, b) < TOL[dtype]


def test_walk_over_chunks(monkeypatch):
    """Where it takes a path's sums, how far it looks ahead, and the registers of a problem of many paths (all sums kept: 259)."""
    from openequivariance_amd import runtime as rt

    def walk(irreps, in2="1x0e+1x1o+1x2e", dtype=np.float32):
        return UVWBatchedGenerator(common.fully_connected((irreps, in2, irreps), shared=False, dtype=dtype)[0], stream=False)
    seven = "+".join(f"17x{l}{p}" for l in range(3) for p in "eo")
    assert walk("17x0e+17x1o+17x2e")._chunk_walk() == ((4, 8), False)
    assert walk("17x0e+17x1o+17x2e", dtype=np.float64)._chunk_walk() == ((2, 4), False)
    assert walk("65x0e+65x1o")._chunk_walk() == ((4, 8), True) and walk(seven)._chunk_walk() == ((4, 8), True)
    assert walk("64x0e+64x1o")._chunk_walk() == ((2, 4), False) and walk("32x0e+32x1o")._chunk_walk() == ((4, 8), False)
    k = rt.kernel_metadata(rt.compile_source(walk(seven).render(), use_cache=False))["backward"]
    assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_count"] <= 128


@pytest.mark.parametrize("dtype", list(TOL))
@pytest.mark.parametrize("case", ["l3", "copies", "whole"])
def test_walk_over_chunks_emulated(case, dtype, monkeypatch):
    """With sums taken (many paths) and left, looking four and two chunks ahead, more and fewer of them than that."""
    monkeypatch.setitem(CASES, "whole", ("64x0e", "1x0e", "64x0e"))
    _, prob, oprob = generator(case, dtype)
    g = UVWBatchedGenerator(prob, stream=False)
    assert g._chunk_walk()[1] == (case == "l3")
    X, Y, We, G = common.tp_inputs(prob, 3, 10, dtype=dtype, w_scale=0.3)
    out = emu.run_tp(g, g.plan()[1], X, Y, ow.e3nn_to_oeq(oprob, We), G)
    dX, dY, dW = otp.backward(oprob, X, Y, We, G)
    assert rel_err(out["Xg"], dX) < TOL[dtype] and rel_err(out["Yg"], dY) < TOL[dtype]
    assert rel_err(ow.oeq_to_e3nn(oprob, out["Wg"]), dW) < TOL[dtype]


DIFFDOCK = ("10x1o+10x1e+48x0e+48x0o", "1x0e+1x1o+1x2e", "10x1o+10x1e+48x0e+48x0o")


@pytest.mark.parametrize("irreps, rows", [(DIFFDOCK, (1024, 1024)), (("10x0e+10x1o+10x2e", "1x0e+1x1o+1x2e", "10x0e+10x1o+10x2e"), (0, 0)),
                                          (("44x0e+44x1o+44x2e", "1x0e+1x1o+1x2e", "44x0e+44x1o+44x2e"), (512, 0)),
                                          (("34x0e+34x1o", "1x0e+1x1o+1x2e", "70x0e+70x1o"), (1024, None)),
                                          (("30x0e+30x1o", "1x0e+1x1o", "30x0e+30x1o"), (0, 1024)), (("5x0e+31x1o", "1x0e+1x1o", "33x0e+31x1o"), (0, 0))])
def test_forward_of_few_rows(irreps, rows):
    """Rows of 16 to 64 KB that pass in batches, half as many of up to 128 KB, none where the walk spills (None); the set for few of
    them has a forward alone."""
    from openequivariance_amd.tensor_product import few_rows_generator
    for dtype, most in zip(TOL, rows):
        prob = common.fully_connected(irreps, shared=False, dtype=dtype)[0]
        g = UVWBatchedGenerator(prob)
        few, limits = few_rows_generator(prob, g)
        assert (g.rows_chunked == most or most is None and g.rows_chunked) and limits == (most or 0, 0) and (few is None) == (not most)
        if few is not None:
            assert not few.stream and few.plan()[1] == [] and "void backward(" not in few.render() and "void backward(" in g.render()
            assert few.forward_body() == UVWBatchedGenerator(prob, stream=False).forward_body() != g.forward_body()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", list(TOL))
def test_forward_of_few_rows_on_the_gpu(cuda, dtype, monkeypatch):
    """Both sides of the line, through the C++ kernels and the raw entry point; a misaligned operand keeps its own kernels."""
    import torch
    import openequivariance_amd as oeq
    prob, oprob = common.fully_connected(DIFFDOCK, shared=False, dtype=dtype)
    tp = oeq.TensorProduct(prob, torch_op=True)
    assert tp._few_rows_limits == (1024, 0) and tp._few_rows is not None
    calls = []
    monkeypatch.setattr(tp._few_rows, "exec_tensor_product", lambda *a, f=tp._few_rows.exec_tensor_product: calls.append(a[0]) or f(*a))
    for n in (1, 1024, 1025):
        X, Y, We, _ = common.tp_inputs(prob, n, n, dtype=dtype, w_scale=0.3)
        x, y, w = (torch.tensor(a, device=cuda) for a in (X, Y, ow.e3nn_to_oeq(oprob, We)))
        Z = otp.forward(oprob, X, Y, We)
        z = torch.full((n, Z.shape[1]), float("nan"), device=cuda, dtype=x.dtype)
        tp.forward_raw(n, x.data_ptr(), y.data_ptr(), z.data_ptr(), w.data_ptr())
        off = torch.cat([w.new_zeros(1), w.reshape(-1)])[1:].view(w.shape)
        for got in (tp.forward(x, y, w), z, tp.forward(x, y, off)):
            assert rel_err(got.cpu().numpy(), Z) < TOL[dtype]
    assert calls == [1, 1024]
