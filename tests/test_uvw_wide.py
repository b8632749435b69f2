"""Dense uvw backward of outputs whose dZ tile fits neither LDS nor (a block of it) the registers: read in the K loop.  Held in
registers all the same, it spilled hundreds of them and dX of the first two GPU problems was wrong."""
import numpy as np
import pytest

import common
import openequivariance_amd as oeq
from host_emu import emu
from openequivariance_amd.codegen.uvw import UVWGenerator
from oracle import tp as otp
from oracle import weights as ow


def _problem(irreps):
    prob, oprob = common.fully_connected(irreps, shared=True, dtype=np.float32)
    g = UVWGenerator(prob)
    assert g.bwd_direct and not g.bwd_lds
    return prob, oprob, g


def _check(got, ref):
    # fp32 sums of at most 512 products: 4e-7
    for a, b in zip(got, ref):
        assert np.linalg.norm(a - b) < 1e-6 * np.linalg.norm(b)


def test_generated_source(monkeypatch):
    monkeypatch.setattr(UVWGenerator, "DW_WORKGROUPS", 2)
    prob, oprob, g = _problem(("18x1o", "1x0e+1x2e", "401x1o+402x3o"))
    X, Y, We, G = common.tp_inputs(prob, 17, 9, np.float32, w_scale=0.3)
    _, bwd, ws = g.plan()
    out = emu.run_tp(g, bwd, X, Y, ow.e3nn_to_oeq(oprob, We), G, ws_bytes=ws())
    _check((out["Xg"], out["Yg"]), otp.backward(oprob, X, Y, We, G))


@pytest.mark.gpu
@pytest.mark.parametrize("irreps", [("320x3o", "1x0e", "320x3o"), ("512x1o", "1x0e", "512x1o"), ("18x1o", "1x0e+1x2e", "401x1o+402x3o")])
def test_gpu(cuda, irreps):
    import torch
    from openequivariance_amd import runtime as rt
    from openequivariance_amd.tensor_product import _make_steps
    prob, oprob, g = _problem(irreps)
    op = oeq.TensorProduct(prob)
    # (whatever kernels the operator itself has for the problem)
    op._few_rows = rt.TPImpl(rt.compile_source(g.render()), *(_make_steps(steps, op._step_flags) for steps in g.plan()[:2]))
    op._few_rows_limits = (1000, 1000)
    X, Y, We, G = common.tp_inputs(prob, 37, 5, np.float32)
    x, y, w, dz = (torch.tensor(t, device=cuda) for t in (X, Y, ow.e3nn_to_oeq(oprob, We), G))
    _check([t.cpu().numpy() for t in op.backward_helper(x, y, w, dz)[:2]], otp.backward(oprob, X, Y, We, G))
