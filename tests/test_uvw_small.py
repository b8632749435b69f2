"""Dense uvw kernels for batches of few rows: emulated on the CPU and, on the GPU, against the oracle and the kernels for
large batches at the edges of tiles, of a workgroup's share of the batch and of the dispatch."""
import numpy as np
import pytest

import common
from host_emu import emu
from openequivariance_amd.codegen.uvw import UVWGenerator
from openequivariance_amd.codegen.uvw_small import UVWSmallGenerator
from oracle import tp as otp
from oracle import weights as ow

# one, two, three and five 16-channel subtiles, outputs of one to three w tiles, every degree up to 2
MIXED = ("33x0e+7x1o+20x2e", "1x0e+1x1o+1x2e", "18x0e+35x1o+5x2e")
BOTH = ("50x0e+50x1o+50x1e+50x2o+50x2e", "1x0e", "50x0e+50x1o+50x1e+50x2o+50x2e")


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


# a sum of n products in any order errs by at most n units of the last place of the largest partial sum: 33 x 3 terms an
# output element and 37 rows x 5 a weight, six operations each in front of them
TOL = {np.float32: 200 * 6.0e-8, np.float64: 200 * 1.2e-16}


@pytest.mark.parametrize("dtype,n", [(np.float32, 21), (np.float64, 2)])
def test_emulated(dtype, n, monkeypatch):
    monkeypatch.setattr(UVWGenerator, "DW_WORKGROUPS", 7)
    monkeypatch.setattr(UVWSmallGenerator, "DW_WAVES", 4)
    prob, oprob = common.fully_connected(("18x0e+3x1o", "1x0e+1x1o", "17x0e+5x1o"), shared=True, dtype=dtype)
    g = UVWSmallGenerator.create(prob)
    assert len(g.bwd_groups) == 2 and max(g.chunks) > 1
    X, Y, We, G = common.tp_inputs(prob, n, 9, dtype, w_scale=0.3)
    W = ow.e3nn_to_oeq(oprob, We)
    fwd, bwd, ws = g.plan()
    assert ws() <= UVWGenerator(prob).plan()[2]()
    out = emu.run_tp(g, fwd, X, Y, W, ws_bytes=ws())
    assert rel(out["Z"], otp.forward(oprob, X, Y, We)) < TOL[dtype]
    out = emu.run_tp(g, bwd, X, Y, W, G, ws_bytes=ws())
    dX, dY, dW = otp.backward(oprob, X, Y, We, G)
    assert rel(out["Xg"], dX) < TOL[dtype] and rel(out["Yg"], dY) < TOL[dtype]
    assert rel(ow.oeq_to_e3nn(oprob, out["Wg"]), dW) < TOL[dtype]


def natural(mul, lmax):
    return "+".join(f"{mul}x{l}{'eo'[l % 2]}" for l in range(lmax + 1))


# second operands of 16 to 108 words beside wide outputs: the dZ tile and the wavefronts' dY patches share 160 KB of LDS
WIDE = {
    "16_words": (np.float32, (natural(16, 2), natural(1, 3), natural(240, 2)), True),
    "25_words": (np.float32, (natural(16, 4), natural(1, 4), natural(88, 4)), False),
    "25_words_f64": (np.float64, (natural(16, 2), natural(1, 4), natural(124, 2)), False),
    "36_words_f64": (np.float64, (natural(16, 3), natural(1, 5), natural(64, 3)), False),
    "copies_f64": (np.float64, ("16x0e+16x1o", "3x0e+3x1o+3x2e", "120x0e+120x1o+120x2e"), False),
    "copies": (np.float32, (natural(16, 2), natural(12, 2), natural(144, 2)), False),
    "copies_narrow": (np.float32, (natural(16, 2), natural(12, 2), natural(136, 2)), True),
}


@pytest.mark.parametrize("case", sorted(WIDE))
def test_arrays_fit_lds_together(case):
    dtype, irreps, taken = WIDE[case]
    prob, _ = common.fully_connected(irreps, shared=True, dtype=dtype)
    g = UVWSmallGenerator.create(prob)
    assert (g is not None) == taken
    used = common.lds_bytes((g or UVWSmallGenerator(prob)).render(), np.dtype(dtype).itemsize)
    assert (max(used.values()) <= 160 * 1024) == taken
    assert (g or UVWSmallGenerator(prob)).lds_bytes() == max(used["backward"], used["backward_dw"])


def test_source_that_nearly_fills_lds_builds():
    from openequivariance_amd import runtime as rt
    dtype, irreps, _ = WIDE["16_words"]
    g = UVWSmallGenerator.create(common.fully_connected(irreps, shared=True, dtype=dtype)[0])
    assert g.lds_bytes() > 144 * 1024
    assert rt.kernel_metadata(rt.compile_source(g.render()))["backward"][".group_segment_fixed_size"] == g.lds_bytes()


@pytest.mark.parametrize("generator", [UVWGenerator, UVWSmallGenerator])
def test_fp32_forward_loops_are_unrolled_where_the_factor_divides_them(generator):
    """Several paths per block: 1 to 9 batches of four steps."""
    import re
    for batches in range(1, 10):
        irreps = natural(16 * batches - 3, 1)
        g = generator(common.fully_connected((irreps, natural(1, 1), irreps), shared=True, dtype=np.float32)[0])
        body = g.forward_body()
        assert set(re.findall(r"sg < (\d+);", body)) == {str(batches)}
        assert set(re.findall(r"#pragma unroll (\d)\n *for \(int sg", body)) == {"1" if batches % 2 else "2"}


def test_largest_batches():
    """The forward is left to the kernels for large batches where the longest work item stays whole, and earlier where it
    is not halved; the backward where several wavefronts of a large batch would wait for one."""
    def limits(a, b, dtype, in2=natural(1, 2)):
        return UVWSmallGenerator.row_limits(UVWGenerator(common.fully_connected((natural(a, 2), in2, natural(b, 2)), shared=True, dtype=dtype)[0]))
    for dtype, most in ((np.float32, 8192), (np.float64, 2048)):
        assert limits(64, 64, dtype) == limits(50, 50, dtype) == (most, 5120)
        assert limits(50, 50, dtype, "1x0e") == (most, 8192 if dtype == np.float32 else 65536)
        for a, b in ((97, 13), (32, 32), (100, 30)):
            assert limits(a, b, dtype) == (0, 5120)
        assert limits(32, 100, dtype) == limits(68, 68, dtype, natural(1, 1)) == (most, 5120)
        assert limits(16, 100, dtype) == limits(36, 36, dtype) == limits(128, 128, dtype, natural(1, 1)) == (min(most, 4096), 5120)


@pytest.mark.parametrize("irreps,fp32,fp64", [
    (natural(64, 1), 65536, 16384), (BOTH[0], 65536, 65536), (natural(33, 2), 65536, 65536), (natural(80, 2), 8192, 65536),
    (natural(64, 2), 8192, 16384), (natural(64, 3), 5120, 65536)])
def test_largest_batches_of_one_path_per_block(irreps, fp32, fp64):
    for dtype, limit in ((np.float32, fp32), (np.float64, fp64)):
        prob, _ = common.fully_connected((irreps, "1x0e", irreps), shared=True, dtype=dtype)
        assert UVWSmallGenerator.row_limits(UVWGenerator(prob))[1] == limit


def test_fp64_forward_steps():
    """Every channel has a step, none is a whole block beyond the last, and three divides their number only where no step
    past the last channel is left to take."""
    for mu in range(1, 130):
        ir = f"{mu}x0e"
        p = UVWGenerator(common.fully_connected((ir, "1x0e", "20x0e"), shared=True, dtype=np.float64)[0]).paths[0]
        full = 4 * -(-mu // 16)
        need = 4 * (mu // 16) + min(4, mu % 16)
        assert p.SU == (need + 1 if need % 3 == 0 and need < full else need) <= full
        assert p.SU % 3 or p.SU == full
        s = UVWSmallGenerator(common.fully_connected((ir, "1x0e", "20x0e"), shared=True, dtype=np.float64)[0]).paths[0]
        assert s.SU == need


def test_emulated_step_past_the_last_channel():
    prob, oprob = common.fully_connected(("18x0e+33x1o", "1x0e+1x1o", "5x0e+3x1o"), shared=True, dtype=np.float64)
    g = UVWGenerator(prob)
    assert {p.SU for p in g.paths} == {7, 10}
    X, Y, We, _ = common.tp_inputs(prob, 19, 9, np.float64, w_scale=0.3)
    fwd, _, ws = g.plan()
    out = emu.run_tp(g, fwd, X, Y, ow.e3nn_to_oeq(oprob, We), ws_bytes=ws())
    assert rel(out["Z"], otp.forward(oprob, X, Y, We)) < TOL[np.float64]


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["16_words", "copies_f64"])
def test_wide_second_operands_on_the_gpu(cuda, case):
    import torch
    import openequivariance_amd as oeq
    dtype, irreps, taken = WIDE[case]
    prob, oprob = common.fully_connected(irreps, shared=True, dtype=dtype)
    tp = oeq.TensorProduct(prob, torch_op=True)
    X, Y, We, G = common.tp_inputs(prob, 19, 4, dtype, w_scale=0.3)
    x, y, w, g = (torch.tensor(a, device=cuda) for a in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
    got = [tp.forward(x, y, w), *tp.backward_helper(x, y, w, g)]
    assert (tp._few_rows is not None) == taken
    ref = [otp.forward(oprob, X, Y, We), *otp.backward(oprob, X, Y, We, G)]
    ref[3] = ow.e3nn_to_oeq(oprob, ref[3])
    for a, b in zip(got, ref):
        assert rel(a.cpu().numpy(), b) < 4 * TOL[dtype]      # (sums of up to four times the terms of the products above)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("irreps", [MIXED, BOTH, common.DENSE], ids=["mixed", "both", "dense"])
def test_on_the_gpu(cuda, irreps, dtype):
    import torch
    import openequivariance_amd as oeq
    from openequivariance_amd import runtime as rt
    from openequivariance_amd.tensor_product import _make_steps
    prob, oprob = common.fully_connected(irreps, shared=True, dtype=dtype)
    tp = oeq.TensorProduct(prob, torch_op=True)
    limits = UVWSmallGenerator.row_limits(UVWGenerator(prob))
    assert limits[1] == (65536 if irreps is BOTH else 5120)
    # fp32 kernels on split operands leave these fewer rows, and no forward where they leave it none: here both sides are built
    # whole, without them
    kept = tp._few_rows_limits
    assert all(k <= most for k, most in zip(kept, limits)) and (dtype == np.float32 or kept == limits)
    def build(generator):
        return rt.TPImpl(rt.compile_source(generator.render()), *(_make_steps(steps, tp._step_flags) for steps in generator.plan()[:2]))
    few, large = build(UVWSmallGenerator.create(prob)), build(UVWGenerator(prob))
    for n in (1, 16, 37, 2049, 4097, 5120, 5121):
        X, Y, We, G = common.tp_inputs(prob, n, n, dtype, w_scale=0.3)
        x, y, w, g = (torch.tensor(a, device=cuda) for a in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
        assert [tp._pick_rows(n, back) is None for back in (False, True)] == [n > limit for limit in kept]
        def run():
            return [tp.forward(x, y, w), *tp.backward_helper(x, y, w, g)]
        as_built = run()
        tp._few_rows, tp._few_rows_limits, own = few, (n, n), tp._few_rows
        got, again = run(), run()
        if n <= 37:
            ref = [otp.forward(oprob, X, Y, We), *otp.backward(oprob, X, Y, We, G)]
            ref[3] = ow.e3nn_to_oeq(oprob, ref[3])
            tol = TOL[dtype]
        else:
            # the kernels for large batches; a weight gradient is a sum over the batch in another order
            tp._few_rows = large
            ref, tol = [t.cpu().numpy() for t in run()], 4 * TOL[dtype]
        tp._few_rows, tp._few_rows_limits = own, kept
        for a, c, b in zip(got, as_built, ref):
            assert rel(a.cpu().numpy(), b) < tol and rel(c.cpu().numpy(), b) < tol
        assert all(torch.equal(a, b) for a, b in zip(got[1:], again[1:]))
