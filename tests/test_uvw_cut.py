"""fp64 forward of dense uvw products whose l = 1 blocks have five or six w tiles: cut into ranges of tiles, ragged and whole."""
import numpy as np
import pytest

import common
from host_emu import emu
from openequivariance_amd.codegen.uvw import UVWGenerator
from oracle import tp as otp
from oracle import weights as ow

# a sum of up to 96 channels x 3 second operands x 9 products, an operation each: 3e3 units of the last place
TOL = 3e3 * 1.2e-16
CASES = {"five_ragged": ("18x0e+66x1o", "1x0e+1x1o", "5x0e+66x1o", [(0, 3), (3, 5)]),
         "five": ("20x1o", "1x0e", "80x1o", [(0, 3), (3, 5)]), "six": ("96x0e+7x1o", "1x0e+1x1o", "96x1o", [(0, 3), (3, 6)]),
         "four": ("20x1o", "1x0e", "64x1o", [(0, 4)])}


def problem(case):
    prob, oprob = common.fully_connected(CASES[case][:3], shared=True, dtype=np.float64)
    g = UVWGenerator(prob)
    assert sorted((lo, hi) for o, lo, hi in g.fwd_order if o.D == 3) == CASES[case][3]
    return prob, oprob, g


@pytest.mark.parametrize("case", sorted(CASES))
def test_emulated(case):
    prob, oprob, g = problem(case)
    X, Y, We, _ = common.tp_inputs(prob, 19, 9, np.float64, w_scale=0.3)
    fwd, _, ws = g.plan()
    out = emu.run_tp(g, fwd, X, Y, ow.e3nn_to_oeq(oprob, We), ws_bytes=ws())["Z"]
    ref = otp.forward(oprob, X, Y, We)
    assert np.abs(out - ref).max() < TOL * np.abs(ref).max()


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(CASES))
def test_on_the_gpu(cuda, case):
    import torch
    import openequivariance_amd as oeq
    prob, oprob, _ = problem(case)
    tp = oeq.TensorProduct(prob, torch_op=True)
    tp._few_rows_limits = (0, 0)
    for n in (1, 16, 37, 600):
        X, Y, We, _ = common.tp_inputs(prob, n, n, np.float64, w_scale=0.3)
        out = tp.forward(*(torch.tensor(a, device=cuda) for a in (X, Y, ow.e3nn_to_oeq(oprob, We)))).cpu().numpy()
        ref = otp.forward(oprob, X, Y, We)
        assert np.abs(out - ref).max() < TOL * np.abs(ref).max()


def test_forms_by_rows():
    """Five tiles are cut up to so many rows, by the steps of their K loop, where their whole form leaves room for two wavefronts per
    SIMD; six tiles and second operands of l = 2 are cut throughout, and other products have one form."""
    from openequivariance_amd.tensor_product import few_rows_generator, select_generator

    def forms(irreps, dtype=np.float64):
        g = select_generator(common.fully_connected(irreps, shared=True, dtype=dtype)[0])
        small, limits = few_rows_generator(g.problem, g)
        return [(lo, hi) for o, lo, hi in g.fwd_order if o.D == 3], limits[0], small
    whole, rows, small = forms(("80x0e+80x1o", "1x0e+1x1o", "80x0e+80x1o"))
    assert whole == [(0, 5)] and rows == 57000 and small.plan()[0][1]["grid_y"] == 3 and small.plan()[0][0]["kernel"] == "prep_forward"
    assert forms(("100x0e+100x1o", "1x0e+1x1o", "80x0e+80x1o"))[:2] == ([(0, 5)], 28000)
    assert forms(("96x0e+96x1o", "1x0e+1x1o", "96x0e+96x1o"))[:2] == ([(0, 3), (3, 6)], 0)
    assert forms(("66x0e+66x1o", "1x0e+1x1o+1x2e", "66x0e+66x1o"))[:2] == ([(0, 3), (3, 5)], 0)
    assert forms(("64x0e+64x1o", "1x0e+1x1o", "64x0e+64x1o"))[0] == [(0, 4)]


@pytest.mark.parametrize("case", ["five_ragged", "five"])
def test_form_of_few_rows_emulated(case):
    """The forward that the kernels for few rows take over, in the workspace of the others."""
    from openequivariance_amd.tensor_product import few_rows_generator, select_generator
    prob, oprob, _ = problem(case)
    g = select_generator(prob)
    small, limits = few_rows_generator(prob, g)
    assert limits[0] == g.rows_cut > 0
    X, Y, We, _ = common.tp_inputs(prob, 19, 9, np.float64, w_scale=0.3)
    ref = otp.forward(oprob, X, Y, We)
    out = {}
    for name, h in (("few", small), ("many", g)):
        out[name] = emu.run_tp(h, h.plan()[0], X, Y, ow.e3nn_to_oeq(oprob, We), ws_bytes=g.plan()[2]())["Z"]
        assert np.abs(out[name] - ref).max() < TOL * np.abs(ref).max()
    assert np.array_equal(out["few"], out["many"])


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["five_ragged", "five"])
def test_forms_agree_on_the_gpu(cuda, case):
    """Bit for bit, on both sides of the limit: a block's sums are the same in either form."""
    import torch
    import openequivariance_amd as oeq
    prob, oprob, _ = problem(case)
    tp = oeq.TensorProduct(prob, torch_op=True)
    limit = tp._few_rows_limits[0]
    assert limit == tp.generator.rows_cut > 0
    X, Y, We, _ = common.tp_inputs(prob, limit + 1, 3, np.float64, w_scale=0.3)
    x, y, w = (torch.tensor(a, device=cuda) for a in (X, Y, ow.e3nn_to_oeq(oprob, We)))
    many = tp.forward(x, y, w)
    few = tp.forward(x[:limit], y[:limit], w)
    assert torch.equal(few, many[:limit])
    rows = [0, 1, limit - 1, limit]
    ref = otp.forward(oprob, X[rows], Y[rows], We)
    assert np.abs(many[rows].cpu().numpy() - ref).max() < TOL * np.abs(ref).max()
