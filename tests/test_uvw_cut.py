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
