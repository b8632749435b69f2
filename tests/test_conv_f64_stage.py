"""fp64 backward of the convolution with an edge's operands staged through LDS as 4-byte words: records of one to five
values, one to three row groups a wavefront, ragged and several chunks, edges naming no node, both edge orders."""
import numpy as np
import pytest

import common
from host_emu import emu
from openequivariance_amd.codegen.uvu_det import UVUDetGenerator
from openequivariance_amd.codegen.uvu_recv import UVURecvGenerator
from oracle import tp as otp

CASES = {"two_row_groups": common.NEQUIP, "one_chunk": ("40x0e+40x1o", "1x0e+1x1o", "40x0e+40x1o+40x2e"),
         "three_chunks_ragged": ("5x0e+3x1o+130x2e", "1x0e+1x1o+1x2e", "5x0e+3x1o+130x2e")}

# one rounding a product and a sum, at most a hundred terms a value and ten edges a node: 1e3 units of the last place
TOL = 1e3 * 1.2e-16


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def generator(cls, prob, monkeypatch):
    monkeypatch.setattr(UVUDetGenerator, "F64_STAGE_WORDS", 1)
    monkeypatch.setattr(UVURecvGenerator, "RECV_SPLIT_WORDS_REGISTER_LOADS", {"float": 0, "double": 64})
    g = cls(prob)
    assert g.uses_stage if cls is UVURecvGenerator else g.staged_backward
    return g


@pytest.mark.parametrize("cls", [UVUDetGenerator, UVURecvGenerator], ids=["sender", "receiver"])
@pytest.mark.parametrize("case", ["two_row_groups", "three_chunks_ragged"])
def test_emulated(case, cls, monkeypatch):
    prob, oprob = common.channelwise(CASES[case], dtype=np.float64)
    g = generator(cls, prob, monkeypatch)
    nodes, nnz = 5, 17
    rows, cols, _ = common.with_invalid_edges(*common.random_graph(nodes, nnz, 7, self_loops=True), nodes, 8)
    rows, cols, tperm, _ = otp.coord_graph(rows, cols)
    valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 8, dtype=np.float64)
    _, bwd, ws = g.plan()
    out = emu.run_conv(g, bwd, X, Y, W, rows, cols, G=G, tperm=tperm, ws_bytes=ws(nnz, nodes))
    for got, want in zip((out["Xg"], out["Yg"], out["Wg"]),
                         common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)[1:]):
        assert rel(got, want) < TOL


@pytest.mark.gpu
@pytest.mark.parametrize("deterministic", [False, True])
@pytest.mark.parametrize("case", list(CASES))
def test_on_the_gpu(cuda, case, deterministic, monkeypatch):
    """Against the oracle, and the deterministic operator bit for bit twice."""
    import torch
    import openequivariance_amd as oeq
    monkeypatch.setattr(UVUDetGenerator, "F64_STAGE_WORDS", 1)
    prob, oprob = common.channelwise(CASES[case], dtype=np.float64)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=deterministic)
    if not deterministic:
        conv.autotune = False
    for nodes, nnz in ((3, 1), (40, 700), (7, 0)):
        rows, cols, tperm, _ = otp.coord_graph(*common.random_graph(nodes, nnz, 5, self_loops=True))
        X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 6, dtype=np.float64)
        args = [torch.tensor(a, device=cuda) for a in (X, Y, W, G, rows, cols, tperm)][:None if deterministic else -1]
        got = conv.backward_helper(*args)
        for a, b in zip(got, otp.conv_backward(oprob, X, Y, W, G, rows, cols)):
            assert a.shape == b.shape and (b.size == 0 or not b.any() and not a.any() or rel(a.cpu().numpy(), b) < TOL)
        if deterministic:
            assert all(torch.equal(a, b) for a, b in zip(got, conv.backward_helper(*args)))
