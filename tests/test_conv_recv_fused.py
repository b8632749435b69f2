"""fp64 pass 1 of the receiver-order backward with its groups of output blocks in one launch: one and two row groups a
wavefront, ragged and several chunks, edges naming no node, both edge orders, hubs; groups of very different length keep a
launch each."""
import numpy as np
import pytest

import common
from host_emu import emu
from openequivariance_amd.codegen.uvu_recv import UVURecvGenerator
from openequivariance_amd.codegen.uvu_sorted import UVUSortedGenerator
from oracle import tp as otp

SH3 = "1x0e+1x1o+1x2e+1x3o"
CASES = {"two_row_groups": ("32x0e+32x1o+32x2e", SH3, "32x0e+32x1o+32x2e+32x3o"),
         "three_chunks_ragged": ("35x0e+3x1o+130x2e", SH3, "35x0e+3x1o+130x2e+35x3o")}

# one rounding a product and a sum, at most a hundred terms a value and ten edges a node: 1e3 units of the last place
TOL = 1e3 * 1.2e-16


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("order", ["sorted", "unsorted"])
@pytest.mark.parametrize("case", list(CASES))
def test_emulated(case, order):
    prob, oprob = common.channelwise(CASES[case], dtype=np.float64)
    det = order == "sorted"
    g = UVURecvGenerator(prob) if det else UVUSortedGenerator(prob, grouped_backward=True, recv_backward=True)
    b = g if det else g.bwd
    assert b.fused and b.HR >= 2
    nodes, nnz = 5, 19
    rows, cols, _ = common.with_invalid_edges(*common.random_graph(nodes, nnz, 7, self_loops=True), nodes, 8)
    tperm = np.arange(nnz)
    if det:
        rows, cols, tperm, _ = otp.coord_graph(rows, cols)
    valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 8, dtype=np.float64)
    _, bwd, ws = g.plan()
    steps = [s for s in bwd if s["kernel"] == "backward"]
    assert len(steps) == 1 and steps[0]["grid_y"] == b.NCH * b.HR and not any("backward_g" in s["kernel"] for s in bwd)
    out = emu.run_conv(g, bwd, X, Y, W, rows, cols, G=G, tperm=tperm, ws_bytes=ws(nnz, nodes))
    for got, want in zip((out["Xg"], out["Yg"], out["Wg"]),
                         common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)[1:]):
        assert rel(got, want) < TOL


@pytest.mark.parametrize("irreps, words", [(("64x0e+64x2e", "1x1o+1x3o+1x5o", "64x1o+64x3o"), [10, 27]),
                                           (("64x0e+64x2e", "1x1o+1x3o", "64x1o+64x3o"), [10, 20])])
def test_groups_of_different_length_keep_a_launch_each(irreps, words):
    g = UVURecvGenerator(common.channelwise(irreps, dtype=np.float64)[0], recv_split=29)
    assert g.staged_f64 and [sum(g.out[i].D for i in grp) for grp in g.recv_groups] == words
    assert g.fused == (2 * words[0] >= words[1])
    assert [s["kernel"] for s in g.plan()[1] if s["kernel"] in ("backward", "backward_g1")] == \
        ["backward", "backward_g1"][:1 if g.fused else 2]


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_on_the_gpu(cuda, case):
    """Against the oracle, and bit for bit twice; no edges, one edge, a hub, edges naming no node."""
    import torch
    import openequivariance_amd as oeq
    prob, oprob = common.channelwise(CASES[case], dtype=np.float64)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=True)
    assert conv.generator.fused
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for nodes, nnz in ((3, 1), (40, 700), (7, 0)):
        if nnz == 700:
            rows, cols = common.hub_graph(nodes, nnz, 45, hub_in=3, hub_out=5, in_edges=300, out_edges=200)
            rows, cols, _ = common.with_invalid_edges(rows, cols, nodes, 16)
        else:
            rows, cols = common.random_graph(nodes, nnz, 5, self_loops=True)
        rows, cols, tperm, _ = otp.coord_graph(rows, cols)
        valid = (rows >= 0) & (rows < nodes) & (cols >= 0) & (cols < nodes)
        X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 6, dtype=np.float64)
        runs = []
        for _ in range(2):
            x, y, w = (t(a).requires_grad_() for a in (X, Y, W))
            z = conv(x, y, w, t(rows), t(cols), t(tperm))
            runs.append(torch.autograd.grad(z, (x, y, w), t(G)))
        assert all(torch.equal(a, b) for a, b in zip(*runs))
        if not nnz:
            assert not runs[0][0].any()
            continue
        for got, want in zip(runs[0], common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, valid)[1:]):
            if np.abs(want).max():
                assert rel(got.cpu().numpy(), want) < TOL


TWO = ("64x0e+64x1o", SH3, "64x0e+64x1o+64x2e+64x3o")             # groups of 16 and 24 words


def test_two_groups_go_together_on_few_nodes():
    """Together, the shorter of two groups loses a wavefront per SIMD: a launch each, but on graphs that do not fill the chip."""
    for irreps, chunks in ((TWO, 1), (tuple(s.replace("64x", "128x") if s != SH3 else s for s in TWO), 2)):
        g = UVURecvGenerator(common.channelwise(irreps, dtype=np.float64)[0]).add_few_nodes()
        assert not g.fused and g.fused_few and g.NCH == chunks and "void backward_together(" in g.render()
        steps = {s["kernel"]: s for s in g.plan_few()[1] if s["kernel"] in ("backward", "backward_g1", "backward_together")}
        assert list(steps) == ["backward_together", "backward", "backward_g1"] and steps["backward_together"]["grid_y"] == 2 * chunks
        assert [s.get("few_nodes", s.get("many_nodes")) for s in steps.values()] == [(512 // chunks, 0, 0)] + [(512 // chunks, 0)] * 2
        assert not any("few_nodes" in s or s["kernel"] == "backward_together" for s in g.plan()[1])
    three = UVURecvGenerator(common.channelwise(CASES["two_row_groups"], dtype=np.float64)[0]).add_few_nodes()
    assert three.fused and not three.fused_few and "backward_together" not in three.render()


@pytest.mark.parametrize("together", [False, True])
def test_two_groups_emulated(together):
    prob, oprob = common.channelwise(TWO, dtype=np.float64)
    g = UVURecvGenerator(prob)
    g.fused = together                            # (what backward_together runs)
    nodes, nnz = 5, 19
    rows, cols, tperm, _ = otp.coord_graph(*common.random_graph(nodes, nnz, 7, self_loops=True))
    X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 8, dtype=np.float64)
    _, bwd, ws = g.plan()
    out = emu.run_conv(g, bwd, X, Y, W, rows, cols, G=G, tperm=tperm, ws_bytes=ws(nnz, nodes))
    want = common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, np.ones(nnz, bool))[1:]
    for got, ref in zip((out["Xg"], out["Yg"], out["Wg"]), want):
        assert rel(got, ref) < TOL


@pytest.mark.gpu
def test_two_groups_on_the_gpu(cuda):
    """Both sides of the line in nodes, few and many edges."""
    import torch
    import openequivariance_amd as oeq
    prob, oprob = common.channelwise(TWO, dtype=np.float64)
    conv = oeq.TensorProductConv(prob, torch_op=True, deterministic=True)
    assert conv.generator.fused_few
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for nodes, nnz in ((1, 3), (512, 100), (512, 4000), (513, 100), (513, 4000)):
        rows, cols, tperm, _ = otp.coord_graph(*common.random_graph(nodes, nnz, 5, self_loops=True))
        X, Y, W, G = common.conv_inputs(prob, nodes, nnz, 6, dtype=np.float64)
        x, y, w = (t(a).requires_grad_() for a in (X, Y, W))
        got = torch.autograd.grad(conv(x, y, w, t(rows), t(cols), t(tperm)), (x, y, w), t(G))
        for a, ref in zip(got, common.conv_reference_on_valid_edges(otp, oprob, X, Y, W, G, rows, cols, np.ones(nnz, bool))[1:]):
            assert rel(a.cpu().numpy(), ref) < TOL
